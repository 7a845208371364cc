// pfm_forces.hip -- force and energy passes on gfx950.
//
// Every pass is a gather over full neighbour lists: T lanes share one atom
// row, each lane walks every T-th entry, the row's force is summed across the
// T lanes with DPP/shuffle reductions and written by the row's first lane.
// No atomics; per-atom sums are FP64 in both precisions.  Template parameter
// R is the pair arithmetic (double, or float for the mixed path: dr formed in
// FP64 and rounded once), E adds the per-row energy of the reference's
// *_energy routines.
//
//   rjl     density pass + embedding-force pass   (RosatoGuillopeLegrand.f90:23-94)
//   lj      pair gather over nl(1) and nl(2)      (LennardJones.f90:23-69)
//   lj1g    pair gather over the full list with the reference's half-list
//           weights                                (LennardJones_1g.f90:28-117)
//   tb      bond-order pass + force pass          (TersoffBrenner.f90:26-150)
//   ljc/morsec  normals, graphene pass, normal-derivative pass, metal pass
//           (graphenenorm.f90:38-56, LennardJonesCosine.f90, MorseCosine.f90)
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "pfm_internal.h"

struct RowArgs {
  int nrows, stride;
  const int* rows;
  const int* nnum;
  const int* nbr;
  const double4* pos;  // FP64 positions
  const uint4* qpos;   // fixed-point positions (mixed path)
  float3 hq;           // L / 2^32 per axis
  float hiso;          // L / 2^32 when the box is a cube, else 0 (one replica; else RepDev::hiso)
  double3 hb, L, iL;
  const int* rep;      // replica of every internal atom (null: one replica, geometry above)
  const RepDev* rdev;
  double4* frc;
  int accumulate;  // 0: this pass writes the first contribution of the step
  double* e_row;
};

// geometry of the replica that holds atom i
template <class R> __device__ __forceinline__ Geo<R> geo_of(const RowArgs& a, int i);
template <> __device__ __forceinline__ Geo<double> geo_of<double>(const RowArgs& a, int i) {
  if (a.rep) {
    const RepDev& R = a.rdev[a.rep[i]];
    return Geo<double>{a.pos, R.L, R.iL};
  }
  return Geo<double>{a.pos, a.L, a.iL};
}
template <> __device__ __forceinline__ Geo<float> geo_of<float>(const RowArgs& a, int i) {
  if (a.rep) {
    const float3 hq = a.rdev[a.rep[i]].hq;
    return Geo<float>{a.qpos, hq.x, hq.y, hq.z};
  }
  return Geo<float>{a.qpos, a.hq.x, a.hq.y, a.hq.z};
}

// store v in the w slot of atom i's position record (pos4 or qpos)
template <class R> __device__ __forceinline__ void store_w(const RowArgs& a, int i, double v);
template <> __device__ __forceinline__ void store_w<double>(const RowArgs& a, int i, double v) {
  const_cast<double4*>(a.pos)[i].w = v;
}
template <> __device__ __forceinline__ void store_w<float>(const RowArgs& a, int i, double v) {
  const_cast<uint4*>(a.qpos)[i].w = __float_as_uint((float)v);
}

#define ROW_PROLOGUE(T) ROW_PROLOGUE_AT(T, xcd_block(nb_real))
#define ROW_PROLOGUE_AT(T, LB) ROW_PROLOGUE_RET(T, LB, )
#define ROW_PROLOGUE_RET(T, LB, RET)                      \
  int lb = (LB);                                          \
  if (lb < 0) return RET;                                 \
  int gt = lb * blockDim.x + threadIdx.x;                 \
  int row = gt / (T), t = threadIdx.x & ((T)-1);          \
  if (row >= a.nrows) return RET;                         \
  int i = a.rows[row];                                    \
  const Geo<R> G = geo_of<R>(a, i);                       \
  const typename Geo<R>::P pi = G.at(i);                  \
  int n = a.nnum[row];                                    \
  const int* nbrow = a.nbr + (size_t)row * a.stride;

// Walk a row's entries four at a time: lane t of the row's T lanes takes
// entries 4t..4t+3 of every block of 4T, with one 16-byte index load (rows
// start on 16 bytes and are padded past their end), then the four
// position-record gathers, then the arithmetic f(j, record, valid).  A block
// waits on two memory latencies.  Entries past the end of the row gather the
// row atom's own record and reach f with valid = false (f masks their
// contribution without branching).
// The FP64 passes take one entry per iteration (every T-th entry), which costs
// fewer registers, and load the next entry's record and the index after it
// before the arithmetic of the current one: on small systems, whose few
// wavefronts cannot hide the two dependent loads, the lj / lj1g / rjl passes
// of a 14,000-atom batch went from 11.5 to 9.9 us a launch; large ones are
// unchanged within 3%.
// The FP32 walk calls flush() after every block of four entries: passes that
// sum a block's contributions in FP32 registers (RowAcc<float>) move them to
// the row's FP64 sums there, one conversion and FP64 add per block and
// component instead of one per entry.
struct NoFlush {
  __device__ __forceinline__ void operator()() const {}
};
template <int T, class R, class F, class B = NoFlush>
__device__ __forceinline__ void walk_row(const Geo<R>& G, const int* __restrict__ nbrow, int n, int t, int self, F f,
                                         B flush = B{}) {
  if constexpr (sizeof(R) == 8) {
    int j = t < n ? nbrow[t] : self, jn = t + T < n ? nbrow[t + T] : self;
    typename Geo<R>::P q = G.at(j);
    for (int p = t; p < n; p += T) {
      const typename Geo<R>::P qn = G.at(jn);
      const int jf = p + 2 * T < n ? nbrow[p + 2 * T] : self;
      f(j, q, true);
      q = qn;
      j = jn;
      jn = jf;
    }
    return;
  }
  for (int p0 = 4 * t; p0 < n; p0 += 4 * T) {
    const int4 v = *reinterpret_cast<const int4*>(nbrow + p0);
    const int jj[4] = {v.x, p0 + 1 < n ? v.y : self, p0 + 2 < n ? v.z : self, p0 + 3 < n ? v.w : self};
    typename Geo<R>::P q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) q[u] = G.at(jj[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) f(jj[u], q[u], p0 + u < n);
    flush();
  }
}

// Per-lane sums of a row pass, a vector (fx, fy, fz) and a scalar e:
// force(c, dr) subtracts c dr, add(v) / sub(v) add / subtract the vector v,
// energy(x) adds x to e.  FP64: every term goes straight into the FP64 sums.
// FP32 terms: a block of four entries is summed in FP32 and flush() adds the
// block to the FP64 sums.  The two sides of a pair then round in different
// blocks, so a system's forces sum to zero within about 1e-8 of sum |F_i|
// instead of within FP64 rounding.
template <class R> struct RowAcc;
template <> struct RowAcc<double> {
  double fx = 0, fy = 0, fz = 0, e = 0;
  __device__ __forceinline__ void force(double c, double dx, double dy, double dz) {
    fx -= c * dx; fy -= c * dy; fz -= c * dz;
  }
  __device__ __forceinline__ void add(double x, double y, double z) { fx += x; fy += y; fz += z; }
  __device__ __forceinline__ void sub(double x, double y, double z) { fx -= x; fy -= y; fz -= z; }
  __device__ __forceinline__ void energy(double v) { e += v; }
  __device__ __forceinline__ void flush() {}
};
template <> struct RowAcc<float> {
  double fx = 0, fy = 0, fz = 0, e = 0;
  float bx = 0, by = 0, bz = 0, be = 0;
  __device__ __forceinline__ void force(float c, float dx, float dy, float dz) {
    bx = __builtin_fmaf(-c, dx, bx); by = __builtin_fmaf(-c, dy, by); bz = __builtin_fmaf(-c, dz, bz);
  }
  __device__ __forceinline__ void add(float x, float y, float z) { bx += x; by += y; bz += z; }
  __device__ __forceinline__ void sub(float x, float y, float z) { bx -= x; by -= y; bz -= z; }
  __device__ __forceinline__ void energy(float v) { be += v; }
  __device__ __forceinline__ void flush() {
    fx += (double)bx; fy += (double)by; fz += (double)bz; e += (double)be;
    bx = by = bz = be = 0.0f;
  }
};

// walk_row with one per-atom side value of each neighbour (aux[j]) gathered
// together with its position record: f(j, record, aux value, valid)
template <int T, class R, class A, class F, class B = NoFlush>
__device__ __forceinline__ void walk_row_aux(const Geo<R>& G, const int* __restrict__ nbrow, int n, int t, int self,
                                             const A* __restrict__ aux, F f, B flush = B{}) {
  if constexpr (sizeof(R) == 8) {
    int j = t < n ? nbrow[t] : self, jn = t + T < n ? nbrow[t + T] : self;
    typename Geo<R>::P q = G.at(j);
    A x = aux[j];
    for (int p = t; p < n; p += T) {
      const typename Geo<R>::P qn = G.at(jn);
      const A xn = aux[jn];
      const int jf = p + 2 * T < n ? nbrow[p + 2 * T] : self;
      f(j, q, x, true);
      q = qn;
      x = xn;
      j = jn;
      jn = jf;
    }
    return;
  }
  for (int p0 = 4 * t; p0 < n; p0 += 4 * T) {
    const int4 v = *reinterpret_cast<const int4*>(nbrow + p0);
    const int jj[4] = {v.x, p0 + 1 < n ? v.y : self, p0 + 2 < n ? v.z : self, p0 + 3 < n ? v.w : self};
    typename Geo<R>::P q[4];
    A x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      q[u] = G.at(jj[u]);
      x[u] = aux[jj[u]];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) f(jj[u], q[u], x[u], p0 + u < n);
    flush();
  }
}

// walk_row over entries that carry a two-bit tag in bits 30-31 (lj1g's
// weights): f(record, tag, valid)
#define ENTRY_ATOM 0x3fffffff
template <int T, class R, class F, class B = NoFlush>
__device__ __forceinline__ void walk_row_tag(const Geo<R>& G, const int* __restrict__ nbrow, int n, int t, int self,
                                             F f, B flush = B{}) {
  if constexpr (sizeof(R) == 8) {
    unsigned e = t < n ? nbrow[t] : self, en = t + T < n ? nbrow[t + T] : self;
    typename Geo<R>::P q = G.at((int)(e & ENTRY_ATOM));
    for (int p = t; p < n; p += T) {
      const typename Geo<R>::P qn = G.at((int)(en & ENTRY_ATOM));
      const unsigned ef = p + 2 * T < n ? nbrow[p + 2 * T] : self;
      f(q, e >> 30, true);
      q = qn;
      e = en;
      en = ef;
    }
    return;
  }
  for (int p0 = 4 * t; p0 < n; p0 += 4 * T) {
    const int4 v = *reinterpret_cast<const int4*>(nbrow + p0);
    const unsigned ee[4] = {(unsigned)v.x, p0 + 1 < n ? (unsigned)v.y : (unsigned)self,
                            p0 + 2 < n ? (unsigned)v.z : (unsigned)self, p0 + 3 < n ? (unsigned)v.w : (unsigned)self};
    typename Geo<R>::P q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) q[u] = G.at((int)(ee[u] & ENTRY_ATOM));
#pragma unroll
    for (int u = 0; u < 4; ++u) f(q[u], ee[u] >> 30, p0 + u < n);
    flush();
  }
}

// r < R2; in FP64 the NaN distance of two atoms on one point counts as
// inside, so it reaches the forces and the out-of-cell check stops the run
template <class R> __device__ __forceinline__ bool inside(R r, R R2);
template <> __device__ __forceinline__ bool inside<double>(double r, double R2) { return !(r >= R2); }
template <> __device__ __forceinline__ bool inside<float>(float r, float R2) { return r < R2; }

__device__ __forceinline__ void write_force(const RowArgs& a, int i, double fx, double fy, double fz) {
  double4 f = a.accumulate ? a.frc[i] : make_double4(0, 0, 0, 0);
  f.x += fx; f.y += fy; f.z += fz;
  a.frc[i] = f;
}

// the force a row's first lane wrote (i < 0: this lane wrote none)
struct RowForce {
  int i = -1;
  double x = 0, y = 0, z = 0;
};

// ------------------------------------------------------------------- RGL

// Mixed-path dr of the RGL passes and its square.  Any box: the fixed-point
// differences scaled per axis (Geo<float>::d2).  ISO (the row's replica is a
// cube, h = L / 2^32 on every axis): the unscaled differences and
// h^2 (ux^2 + uy^2 + uz^2), two multiplies fewer; dr = h (ux, uy, uz), so
// a pass that sums c dr sums c u and multiplies the row's sum by h.  The
// choice is the replica's own, so with the same lanes per row (pfm_set_tuning;
// row_lanes starts a handle by its atoms) a replica takes the same arithmetic
// in a batch as alone.
__device__ __forceinline__ float hiso_of(const RowArgs& a, int i) { return a.rep ? a.rdev[a.rep[i]].hiso : a.hiso; }
template <bool ISO>
__device__ __forceinline__ float rjl_d2(const Geo<float>& G, const uint4& a, const uint4& b, float h2, float& dx,
                                        float& dy, float& dz) {
  if constexpr (ISO) {
    dx = (float)(int)(b.x - a.x);
    dy = (float)(int)(b.y - a.y);
    dz = (float)(int)(b.z - a.z);
    return __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)) * h2;
  } else {
    return G.d2(a, b, dx, dy, dz);
  }
}

// -pi/(2 (R2 - R1)) of a potential's parameters: in FP64 from one division
template <class R, class P>
__device__ __forceinline__ R cutoff_kdf(const P& p) {
  if constexpr (sizeof(R) == 8) return -p.hw;
  return -0.5 * PFM_PI * p.invw;
}

struct RjlP {
  double A0, xi, p, q, r0, R1, R2, invw, hw;  // hw: pi/(2 (R2 - R1)), FP64 passes
};

// largest workgroup of the row passes: FP32 pair arithmetic fits 128 VGPRs
// (16 waves per CU), FP64 needs up to 256
template <class R> struct PairBlock { static constexpr int max = sizeof(R) == 4 ? 1024 : 256; };
#define PAIR_BLOCK (PairBlock<R>::max)

// density pass: rho_i = sum_{r <= R2} exp(-2q(r/r0-1)) fc(r); stores
// Eb_i = sqrt(rho_i) and 1/Eb_i in the w slot of atom i's position record
template <int T, class R>
__device__ __forceinline__ void rjl_density_rows(const RowArgs& a, const RjlP& P, double* __restrict__ eb, int blk) {
  ROW_PROLOGUE_AT(T, blk)
  double rho = 0.0;
  if constexpr (sizeof(R) == 4) {
    // exp(-2q(r/r0 - 1)) = 2^(r kr + k0); cutoff argument in revolutions as in cutoff_bl<float>
    const float R2 = P.R2, ca = 0.5 * P.invw, cb = -0.5 * P.R1 * P.invw;
    const float kr = PM<float>::kexp(-2.0 * P.q / P.r0), k0 = PM<float>::kexp(2.0 * P.q);
    const float hiso = hiso_of(a, i);
    auto body = [&](auto iso) {
      constexpr bool ISO = decltype(iso)::value;
      const float h2 = hiso * hiso;
      RowAcc<float> acc;
      walk_row<T, float>(G, nbrow, n, t, i, [&](int, const uint4& q, bool valid) {
        float dx, dy, dz;
        const float r = __builtin_amdgcn_sqrtf(rjl_d2<ISO>(G, pi, q, h2, dx, dy, dz));
        const float c = __builtin_amdgcn_cosf(__builtin_amdgcn_fmed3f(__builtin_fmaf(r, ca, cb), 0.0f, 0.5f));
        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(r, kr, k0)) * __builtin_fmaf(0.5f, c, 0.5f);
        acc.energy(valid && r <= R2 ? e : 0.0f);
      }, [&] { acc.flush(); });
      return acc.e;
    };
    rho = hiso > 0.0f ? body(std::true_type{}) : body(std::false_type{});
  } else {
    // FP64: exp(-2q(r/r0 - 1)) with its argument as (r - r0) (-2q/r0), whose
    // rounding vanishes where the term is largest; two atoms on one point
    // count as at a vanishing distance
    const double R1 = P.R1, R2 = P.R2, hw = P.hw, r0 = P.r0, kr = -2.0 * P.q / P.r0;
    walk_row<T, R>(G, nbrow, n, t, i, [&](int, const typename Geo<R>::P& q, bool) {
      double dx, dy, dz, r, ir;
      f64::sqrt_rsqrt(fmax(G.d2(pi, q, dx, dy, dz), 1e-300), r, ir);
      const double e = f64::exp((r - r0) * kr) * CutoffHalf(r, R1, R2, hw).f();
      rho += r <= R2 ? e : 0.0;
    });
  }
  rho = group_sum<T>(rho);
  if (t == 0) {
    double s = sqrt(rho);
    eb[i] = s;
    store_w<R>(a, i, 1.0 / s);
  }
}

template <int T, class R>
__global__ void __launch_bounds__(PAIR_BLOCK) k_rjl_density(RowArgs a, RjlP P, double* __restrict__ eb, int nb_real) {
  rjl_density_rows<T, R>(a, P, eb, xcd_block(nb_real));
}

// embedding-force pass (RosatoGuillopeLegrand.f90:80-93):
// F_i -= sum_j [2 A0 (p/r0 fc - df r) e_p - xi (q/r0 fc - df r/2)(1/Eb_i + 1/Eb_j) e_q]/r dr
// with 1/Eb read from the w slot of the gathered position records
template <int T, class R, bool E>
__device__ __forceinline__ void rjl_force_rows(const RowArgs& a, const RjlP& P, const double* __restrict__ eb,
                                               int blk) {
  ROW_PROLOGUE_AT(T, blk)
  double fx = 0, fy = 0, fz = 0, er = 0;
  if constexpr (sizeof(R) == 4) {
    // The two brackets with fc = (1 + cos)/2 and df r = kdf sin folded into
    // their constants: 2 A0 (p/r0 fc - df r) = Ac (1 + cos) + As sin and
    // xi (q/r0 fc - df r/2) = Bc (1 + cos) + Bs sin; the exponentials as
    // 2^(r k + k0).
    const double kdf = -0.5 * PFM_PI * P.invw;
    const float R2 = P.R2, ca = 0.5 * P.invw, cb = -0.5 * P.R1 * P.invw;
    const float Ac = P.A0 * P.p / P.r0, As = -2.0 * P.A0 * kdf;
    const float Bc = 0.5 * P.xi * P.q / P.r0, Bs = -0.5 * P.xi * kdf;
    const float kpr = PM<float>::kexp(-P.p / P.r0), kp0 = PM<float>::kexp(P.p);
    const float kqr = PM<float>::kexp(-2.0 * P.q / P.r0), kq0 = PM<float>::kexp(2.0 * P.q);
    const float ie = Geo<float>::w(pi);
    const float hiso = hiso_of(a, i);
    auto body = [&](auto iso) {
      constexpr bool ISO = decltype(iso)::value;
      const float h2 = hiso * hiso;
      RowAcc<float> acc;
      walk_row<T, float>(G, nbrow, n, t, i, [&](int, const uint4& q, bool valid) {
        float dx, dy, dz, r, ir;
        dist_and_inverse<float>(rjl_d2<ISO>(G, pi, q, h2, dx, dy, dz), r, ir);
        const float x = __builtin_amdgcn_fmed3f(__builtin_fmaf(r, ca, cb), 0.0f, 0.5f);
        const float sn = __builtin_amdgcn_sinf(x), cs = __builtin_amdgcn_cosf(x);
        const float ep = __builtin_amdgcn_exp2f(__builtin_fmaf(r, kpr, kp0));
        const float eq = __builtin_amdgcn_exp2f(__builtin_fmaf(r, kqr, kq0));
        const float A = __builtin_fmaf(As, sn, __builtin_fmaf(Ac, cs, Ac));
        const float B = __builtin_fmaf(Bs, sn, __builtin_fmaf(Bc, cs, Bc));
        const bool in = valid && r <= R2;
        float c = __builtin_fmaf(A, ep, -(B * (ie + Geo<float>::w(q)) * eq)) * ir;
        c = in ? c : 0.0f;
        acc.force(c, dx, dy, dz);
        if (E) {
          const float e = ep * __builtin_fmaf(0.5f, cs, 0.5f);
          acc.energy(in ? e : 0.0f);
        }
      }, [&] { acc.flush(); });
      // with ISO the sums are of c u: dr = h u
      const double hs = ISO ? (double)hiso : 1.0;
      fx = acc.fx * hs; fy = acc.fy * hs; fz = acc.fz * hs; er = acc.e;
    };
    if (hiso > 0.0f) body(std::true_type{});
    else body(std::false_type{});
  } else {
    // FP64: df r = -2 hw times the cutoff's half_sine
    const double R1 = P.R1, R2 = P.R2, hw = P.hw;
    const double r0 = P.r0, kp = -P.p / P.r0, kq = -2.0 * P.q / P.r0;
    const double Ac = 2.0 * P.A0 * P.p / P.r0, As = 4.0 * P.A0 * hw;
    const double Bc = P.xi * P.q / P.r0, Bs = P.xi * hw;
    const double ie = Geo<R>::w(pi);
    walk_row<T, R>(G, nbrow, n, t, i, [&](int, const typename Geo<R>::P& q, bool) {
      double dx, dy, dz, r, ir;
      dist_and_inverse<double, E>(G.d2(pi, q, dx, dy, dz), r, ir);
      const CutoffHalf cut(r, R1, R2, hw);
      const double fc = cut.f(), hs = cut.half_sine();
      const double ep = f64::exp((r - r0) * kp), eq = f64::exp((r - r0) * kq);
      const double A = fma(As, hs, Ac * fc), B = fma(Bs, hs, Bc * fc);
      double c = fma(A, ep, -(B * (ie + Geo<R>::w(q)) * eq)) * ir;
      const bool in = !(r > R2);
      c = in ? c : 0.0;
      fx = fma(-c, dx, fx); fy = fma(-c, dy, fy); fz = fma(-c, dz, fz);
      if (E) er += in ? ep * fc : 0.0;
    });
  }
  fx = group_sum<T>(fx); fy = group_sum<T>(fy); fz = group_sum<T>(fz);
  if (E) er = group_sum<T>(er);
  if (t == 0) {
    write_force(a, i, fx, fy, fz);
    if (E) a.e_row[row] = P.A0 * er - P.xi * eb[i];
  }
}

template <int T, class R, bool E>
__global__ void __launch_bounds__(PAIR_BLOCK) k_rjl_force(RowArgs a, RjlP P, const double* __restrict__ eb,
                                                          int nb_real) {
  rjl_force_rows<T, R, E>(a, P, eb, xcd_block(nb_real));
}

// -------------------------------------------------------------------- LJ

struct LjP {
  double eps4, sig, R1, R2, invw, hw;
};

// a row's lj entries into acc
template <int T, class R, bool E>
__device__ __forceinline__ void lj_walk(const LjP& P, const Geo<R>& G, const typename Geo<R>::P& pi,
                                        const int* __restrict__ nbrow, int n, int t, int i, RowAcc<R>& acc) {
  const R R1 = P.R1, R2 = P.R2, invw = P.invw, sig = P.sig, e4 = P.eps4, kdf = cutoff_kdf<R>(P);
  walk_row<T, R>(G, nbrow, n, t, i, [&](int, const typename Geo<R>::P& q, bool valid) {
    R dx, dy, dz;
    R r, ir;
    dist_and_inverse<R, E>(G.d2(pi, q, dx, dy, dz), r, ir);
    R fc, dfr;
    cutoff_bl<R>(r, R1, R2, invw, kdf, fc, dfr);
    R s = sig * ir, s2 = s * s, V = s2 * s2 * s2;
    R c = e4 * (V * (R(12) * V - R(6)) * fc * ir - V * (V - R(1)) * dfr) * ir;
    const bool in = valid && inside<R>(r, R2);
    c = in ? c : R(0);
    acc.force(c, dx, dy, dz);
    if (E) {
      const R v = e4 * V * (V - R(1)) * fc;
      acc.energy(in ? v : R(0));
    }
  }, [&] { acc.flush(); });
}

// (E with a.e_row null: the converse rows nl(2), which carry no energy)
template <int T, class R, bool E>
__device__ __forceinline__ RowForce lj_rows(const RowArgs& a, const LjP& P, int blk) {
  ROW_PROLOGUE_RET(T, blk, RowForce{})
  RowAcc<R> acc;
  lj_walk<T, R, E>(P, G, pi, nbrow, n, t, i, acc);
  const double fx = group_sum<T>(acc.fx), fy = group_sum<T>(acc.fy), fz = group_sum<T>(acc.fz);
  const double e = E ? group_sum<T>(acc.e) : 0.0;
  if (t == 0) {
    write_force(a, i, fx, fy, fz);
    if (E && a.e_row) a.e_row[row] = e;
  }
  return t == 0 ? RowForce{i, fx, fy, fz} : RowForce{};
}

template <int T, class R, bool E>
__global__ void __launch_bounds__(PAIR_BLOCK) k_lj(RowArgs a, LjP P, int nb_real) {
  lj_rows<T, R, E>(a, P, xcd_block(nb_real));
}

// lj1g: the reference sums entries p <= lessnnum(i) of each row once and
// applies Newton's third law (LennardJones_1g.f90:63-99).  Entry k of row i is
// in that half iff loc(k) < cut(i); the full-list gather weights pair (i,k)
// by [loc(k) < cut(i)] + [loc(i) < cut(k)], which reproduces the reference
// for any group order (for ascending groups the weight is always 1).
struct Lj1gP {
  double c6, c12, c6t6, c12t12, R1, R2, invw;
};

// The weights come from the entries' tags (k_lj1g_tag): bit 30 the pair is in
// i's half list, bit 31 in j's.  A row's entries into acc.
template <int T, class R, bool E>
__device__ __forceinline__ void lj1g_walk(const Lj1gP& P, const Geo<R>& G, const typename Geo<R>::P& pi,
                                          const int* __restrict__ nbrow, int n, int t, int i, RowAcc<R>& acc) {
  const R R1 = P.R1, R2 = P.R2, invw = P.invw, c6 = P.c6, c12 = P.c12, c6t6 = P.c6t6, c12t12 = P.c12t12;
  walk_row_tag<T, R>(G, nbrow, n, t, i, [&](const typename Geo<R>::P& q, unsigned tag, bool valid) {
    int wh = valid && (tag & 1u) ? 1 : 0;
    int w = wh + (valid && (tag & 2u) ? 1 : 0);
    R dx, dy, dz;
    R r, invr2;
    R tr;
    // r and 1/r from one reciprocal square root
    R ir;
    const R d2 = G.d2(pi, q, dx, dy, dz);
    dist_and_inverse<R, E>(d2, r, ir);
    invr2 = ir * ir;
    if constexpr (sizeof(R) == 4) {
      tr = __builtin_amdgcn_fmed3f(r, R1, R2);  // the clamp to [R1, R2]
    } else {
      const double c2 = fma(fma(-d2, invr2, 1.0), invr2, invr2);  // its third power follows: to within half an ulp
      invr2 = !E || d2 > 0.0 ? c2 : invr2;
      tr = fmin(fmax(r, R1), R2);
    }
    // f_dfr_cut (cut_off_poly.f90:30-43), dfr without the 1/(R2-R1) factor
    R x = (tr - R1) * invw, x2 = x * x;
    R f = R(1) + x2 * x * (R(-10) + R(15) * x - R(6) * x2);
    R dfr = tr * x2 * (R(-30) + R(60) * x - R(30) * x2);
    R U = invr2 * invr2 * invr2;
    R Fs = U * invr2 * ((c12t12 * U - c6t6) * f - (c12 * U - c6) * dfr);
    R cw = w ? Fs * R(w) : R(0);  // past the row's end r = 0 and Fs is not finite
    acc.force(cw, dx, dy, dz);
    if (E) {
      // cut_off_poly f_cut (cut_off_poly.f90:6-17)
      R fe = (r > R1 && r < R2) ? f : (r <= R1 ? R(1) : R(0));
      const R v = U * (c12 * U - c6) * fe;
      acc.energy(wh ? v : R(0));
    }
  }, [&] { acc.flush(); });
}

template <int T, class R, bool E>
__device__ __forceinline__ RowForce lj1g_rows(const RowArgs& a, const Lj1gP& P, int blk) {
  ROW_PROLOGUE_RET(T, blk, RowForce{})
  RowAcc<R> acc;
  lj1g_walk<T, R, E>(P, G, pi, nbrow, n, t, i, acc);
  const double fx = group_sum<T>(acc.fx), fy = group_sum<T>(acc.fy), fz = group_sum<T>(acc.fz);
  const double e = E ? group_sum<T>(acc.e) : 0.0;
  if (t == 0) {
    write_force(a, i, fx, fy, fz);
    if (E) a.e_row[row] = e;
  }
  return t == 0 ? RowForce{i, fx, fy, fz} : RowForce{};
}

// lj1g rows and the lj rows of the same atoms (a species' own pairs, then its
// pairs with the other species) in one pass: the row atom's loads, the
// reduction and the force write are shared, and a binary gas's forces need
// one launch instead of two
struct LjRows {
  int stride;
  const int* nnum;
  const int* nbr;
  double* e_row;  // null: the converse rows nl(2)
  LjP p;
};
template <int T, class R, bool E>
__device__ __forceinline__ RowForce lj_both_rows(const RowArgs& a, const Lj1gP& P, const LjRows& b, int blk) {
  ROW_PROLOGUE_RET(T, blk, RowForce{})
  const int n2 = b.nnum[row];
  RowAcc<R> acc;
  lj1g_walk<T, R, E>(P, G, pi, nbrow, n, t, i, acc);
  const double e1 = acc.e;
  acc.e = 0;
  lj_walk<T, R, E>(b.p, G, pi, b.nbr + (size_t)row * b.stride, n2, t, i, acc);
  const double fx = group_sum<T>(acc.fx), fy = group_sum<T>(acc.fy), fz = group_sum<T>(acc.fz);
  const double es = E ? group_sum<T>(e1) : 0.0, el = E ? group_sum<T>(acc.e) : 0.0;
  if (t == 0) {
    write_force(a, i, fx, fy, fz);
    if (E) {
      a.e_row[row] = es;
      if (b.e_row) b.e_row[row] = el;
    }
  }
  return t == 0 ? RowForce{i, fx, fy, fz} : RowForce{};
}

template <int T, class R, bool E>
__global__ void __launch_bounds__(PAIR_BLOCK) k_lj1g(RowArgs a, Lj1gP P, int nb_real) {
  lj1g_rows<T, R, E>(a, P, xcd_block(nb_real));
}

// -------------------------------------------------------------------- TB

struct TbP {
  double D, S, beta, r0, delt, a0, c02, d02, R1, R2, invw, hw;
};

// Tersoff-Brenner rows are short (three bonds in graphene): TB_T lanes share
// a row and lane t owns bonds p = t, t + TB_T, ..; the angular sums of a bond
// over the row's other bonds read their geometry from the owning lane
// (shuffles inside the row's lane group), one chunk of TB_T bonds at a time.
// A row's time is its chain of dependent loads and functions.  Registers for
// one bond a lane instead of arrays for four, loads ahead of the arithmetic
// and the branch-free functions took the force pass of 24,960 atoms from 10.6
// to 7.9 us in FP64 (205 -> 139 VGPRs) and 8.1 to 6.4 mixed.  Eight and
// sixteen lanes a row (two and four for each bond's sums) shortened small
// systems (1,664 atoms, FP64: 13.4 -> 10.4 and 8.6 us) but cost more work on
// large ones, where these rows share a launch (30.0 -> 32.6 and 36.3 us).
#define TB_T 4

// one bond: dr, r, cutoff and its derivative / r
template <class R>
struct TbBond {
  R x = 0, y = 0, z = 0, r = 1, fc = 0, dfc = 0;
  __device__ __forceinline__ void set(const Geo<R> G, const typename Geo<R>::P pa, const typename Geo<R>::P pb,
                                      const TbP& P) {
    const R d2 = G.d2(pa, pb, x, y, z);
    if constexpr (sizeof(R) == 4) {
      r = PM<R>::sqrt_(d2);
      cos_cutoff<R>(r, R(P.R1), R(P.R2), R(P.invw), fc, dfc);
    } else {
      // no branch, and the polynomials instead of the library's sine and cosine
      R ir;
      dist_and_inverse<R>(d2, r, ir);
      cutoff_bl<R>(r, P.R1, P.R2, P.invw, cutoff_kdf<R>(P), fc, dfc);
      // two atoms on one point are at distance 0, inside the cutoff: the bond
      // has an energy, and a force that is not a number stops the run
      r = d2 > R(0) ? r : d2;
      // the selects of cos_cutoff: below R1 nothing of 1/(R2 - R1), which is
      // infinite in a cutoff without a switching zone
      const bool below = r < P.R1, in = r < P.R2;
      fc = below ? R(1) : in ? fc : R(0);
      dfc = !below && in ? dfc * ir : R(0);
    }
  }
  // the bond of lane s of the row's group
  __device__ __forceinline__ TbBond from(int s) const {
    TbBond o;
    o.x = __shfl(x, s, TB_T); o.y = __shfl(y, s, TB_T); o.z = __shfl(z, s, TB_T);
    o.r = __shfl(r, s, TB_T); o.fc = __shfl(fc, s, TB_T); o.dfc = __shfl(dfc, s, TB_T);
    return o;
  }
};

// f(bond q) for every bond q != p of the row, on the lane that owns bond p
// (own: this lane's bond of the chunk at p0).  Rows of one chunk take one turn
// fewer than they have bonds, each lane its next bond cyclically.
template <class R, class F>
__device__ __forceinline__ void tb_other_bonds(const Geo<R>& G, const typename Geo<R>::P& pi,
                                               const int* __restrict__ nbrow, int n, int t, const TbP& P, int p0,
                                               const TbBond<R>& own, F f) {
  if (n <= TB_T) {
    for (int s = 1; s < n; ++s) {
      const TbBond<R> c = own.from(t + s < n ? t + s : t + s - n);
      if (t < n) f(c);
    }
    return;
  }
  for (int q0 = 0; q0 < n; q0 += TB_T) {
    TbBond<R> c = own;
    if (q0 != p0 && q0 + t < n) c.set(G, pi, G.at(nbrow[q0 + t]), P);
    for (int s = 0; s < TB_T && q0 + s < n; ++s) {
      const TbBond<R> d = c.from(s);
      if (p0 + t < n && q0 + s != p0 + t) f(d);
    }
  }
}

// bond order B(p,i) (TersoffBrenner.f90:81-91) and, per entry, the factors
// of the force pass: Bp = B**(1/delt+1) and
// BT = delt/2 * Bp * fc * D/(S-1) * S * exp(-sqrt(2S) beta (r-r0)/S)
template <class R>
__device__ __forceinline__ void tb_bond_rows(const RowArgs& a, const TbP& P, double* __restrict__ B,
                                             double* __restrict__ Bp, double* __restrict__ BT, int blk) {
  constexpr int T = TB_T;
  ROW_PROLOGUE_AT(T, blk)
  const R R2 = P.R2, a0 = P.a0, c02 = P.c02, d02 = P.d02;
  const R ex = R(1.0 / P.delt + 1.0), md = R(-P.delt);
  const R tailc = R(P.D / (P.S - 1.0) * P.S), tailk = R(-sqrt(2.0 * P.S) * P.beta / P.S), r0 = P.r0;
  for (int p0 = 0; p0 < n; p0 += T) {
    const int p = p0 + t;
    TbBond<R> o;
    if (p < n) o.set(G, pi, G.at(nbrow[p]), P);
    R b = 0;
    tb_other_bonds<R>(G, pi, nbrow, n, t, P, p0, o, [&](const TbBond<R>& c) {
      if (o.r < R2 && c.r < R2) {
        R cs = R(1) + (o.x * c.x + o.y * c.y + o.z * c.z) * PM<R>::rcp(o.r * c.r);
        b += c.fc * (R(1) + c02 / d02 - c02 * PM<R>::rcp(d02 + cs * cs));
      }
    });
    if (p >= n) continue;
    R bb = o.r < R2 ? PM<R>::pow_(R(1) + a0 * b, md) : R(0);
    size_t e = (size_t)row * a.stride + p;
    R bp = bb > R(0) ? PM<R>::pow_(bb, ex) : R(0);
    B[e] = (double)bb;
    Bp[e] = (double)bp;
    BT[e] = (double)(R(0.5 * P.delt) * bp * o.fc * tailc * PM<R>::exp_(tailk * (o.r - r0)));
  }
}

template <class R>
__global__ void __launch_bounds__(256) k_tb_bond(RowArgs a, TbP P, double* __restrict__ B, double* __restrict__ Bp,
                                                 double* __restrict__ BT, int nb_real) {
  tb_bond_rows<R>(a, P, B, Bp, BT, xcd_block(nb_real));
}

// The normal-derivative terms of ljc/morsec for a graphene row (the rows of
// the tb list are the rows of the nearest-neighbour list nl(3)): row i adds,
// for each of its three nearest neighbours j, the vector that j's graphene
// pass stored for i's place in j's nearest-neighbour row (cos_nn_coef).
struct NdArgs {
  const int* nnum;    // nl(3) row lengths
  const int* nbr;     // nl(3) entries
  const int* rev;     // place of the row atom in the neighbour's nl(3) row
  const int* row_of;  // internal atom -> row of the graphene group
  const double4* gC;
  int stride;
};

// force pass (TersoffBrenner.f90:193-242): for each bond (i,j): dB_ij/dr_i
// over i's row, dB_ji/dr_i and i as third body of j's bonds over j's row;
// with ND also the row's normal-derivative terms (lane q < 3 takes the q-th
// nearest neighbour).
template <class R, bool E, bool ND>
__device__ __forceinline__ void tb_force_rows(const RowArgs& a, const TbP& P, const int* __restrict__ row_of,
                                              const int* __restrict__ rev, const double* __restrict__ B,
                                              const double* __restrict__ Bp, const double* __restrict__ BT,
                                              const NdArgs& nd, int blk) {
  constexpr int T = TB_T;
  ROW_PROLOGUE_AT(T, blk)
  const R R2 = P.R2, a0 = P.a0, c02 = P.c02, d02 = P.d02;
  const R D_S1 = R(P.D / (P.S - 1.0)), S = P.S, r0 = P.r0;
  const R s2S = R(sqrt(2.0 * P.S) * P.beta), s2oS = R(sqrt(2.0 / P.S) * P.beta), hdel = R(-P.delt * 0.5);
  double fx = 0, fy = 0, fz = 0, e = 0;
  for (int p0 = 0; p0 < n; p0 += T) {
    const int p = p0 + t;
    const size_t ep = (size_t)row * a.stride + (p < n ? p : 0);
    const int j = nbrow[p < n ? p : 0], l = rev[ep], jr = row_of[j];
    const R bpp = (R)Bp[ep], Bi = (R)B[ep];
    const typename Geo<R>::P pj = G.at(j);
    const bool sym = jr >= 0 && l >= 0;  // asymmetric list: reported by k_rev
    const size_t jbase = (size_t)(sym ? jr : 0) * a.stride;
    const int nj = sym && p < n ? a.nnum[jr] : 0;
    const R Bl = (R)B[jbase + (sym ? l : 0)], Bpl = (R)Bp[jbase + (sym ? l : 0)];
    TbBond<R> o;
    if (p < n) o.set(G, pi, pj, P);
    const R irp2 = PM<R>::rcp(o.r * o.r);
    // dB(p,i)/dr_i over i's other bonds q
    R bx = 0, by = 0, bz = 0;
    tb_other_bonds<R>(G, pi, nbrow, n, t, P, p0, o, [&](const TbBond<R>& c) {
      R rr = PM<R>::rcp(o.r * c.r);
      R cosi = (o.x * c.x + o.y * c.y + o.z * c.z) * rr;
      R tt = d02 + (R(1) + cosi) * (R(1) + cosi);
      R c1 = c.fc * R(2) * a0 * c02 * (R(1) + cosi) * PM<R>::rcp(tt * tt);
      R c2 = c.dfc * a0 * (R(1) + c02 / d02 - c02 * PM<R>::rcp(tt));
      R irq2 = PM<R>::rcp(c.r * c.r);
      bx += c1 * ((o.x + c.x) * rr - cosi * (o.x * irp2 + c.x * irq2)) + c2 * c.x;
      by += c1 * ((o.y + c.y) * rr - cosi * (o.y * irp2 + c.y * irq2)) + c2 * c.y;
      bz += c1 * ((o.z + c.z) * rr - cosi * (o.z * irp2 + c.z * irq2)) + c2 * c.z;
    });
    if (p >= n || !sym) continue;
    R gx = bx * bpp, gy = by * bpp, gz = bz * bpp;
    // over j's row; (xl, yl, zl) from j to i
    const R xl = -o.x, yl = -o.y, zl = -o.z;
    R tx = 0, ty = 0, tz = 0;
    // j's entries but its l-th (i itself)
    auto entry = [&](int q) { return jbase + (q + 1 < nj ? (q < l ? q : q + 1) : 0); };
    typename Geo<R>::P pk = G.at(a.nbr[entry(0)]);
    int kn = a.nbr[entry(1)];
    for (int q = 0; q + 1 < nj; ++q) {
      const R bt = (R)BT[entry(q)];
      TbBond<R> c;
      c.set(G, pj, pk, P);
      pk = G.at(kn);
      kn = a.nbr[entry(q + 2)];
      R rr = PM<R>::rcp(o.r * c.r);
      R cosi = (xl * c.x + yl * c.y + zl * c.z) * rr;
      R tt = d02 + (R(1) + cosi) * (R(1) + cosi);
      R gq = R(2) * a0 * c02 * (R(1) + cosi) * PM<R>::rcp(tt * tt);
      R vx = -c.x * rr + cosi * xl * irp2, vy = -c.y * rr + cosi * yl * irp2, vz = -c.z * rr + cosi * zl * irp2;
      R c1 = Bpl * c.fc * gq;
      gx += c1 * vx; gy += c1 * vy; gz += c1 * vz;
      // i as third body of bond (j,k)
      R g2 = o.dfc * a0 * (R(1) + c02 / d02 - c02 * PM<R>::rcp(tt));
      R g1 = o.fc * gq;
      tx += bt * (g1 * vx + o.x * g2);
      ty += bt * (g1 * vy + o.y * g2);
      tz += bt * (g1 * vz + o.z * g2);
    }
    gx *= hdel; gy *= hdel; gz *= hdel;
    fx += (double)tx; fy += (double)ty; fz += (double)tz;
    if (o.r < R2) {
      R fc = o.fc;
      R dff = o.dfc * PM<R>::rcp(fc);
      R av = -s2S * (o.r - r0);
      R ea = PM<R>::exp_(av), eas = PM<R>::exp_(av * PM<R>::rcp(S));
      R pre = fc * D_S1;
      R Bm = Bi + Bl;
      R k1 = (dff - s2S * PM<R>::rcp(o.r)) * ea;
      R k2 = (dff - s2oS * PM<R>::rcp(o.r)) * Bm * R(0.5);
      R se = S * eas;
      fx += (double)(pre * (o.x * k1 - (gx + o.x * k2) * se));
      fy += (double)(pre * (o.y * k1 - (gy + o.y * k2) * se));
      fz += (double)(pre * (o.z * k1 - (gz + o.z * k2) * se));
      if (E) e += 0.5 * (double)(pre * (ea - Bm * R(0.5) * se));
    }
  }
  if (ND && t < 3 && nd.nnum[row] == 3) {
    const int j = nd.nbr[(size_t)row * nd.stride + t];
    const int l = nd.rev[(size_t)row * 3 + t];
    if (l >= 0 && l <= 2 && nd.row_of[j] >= 0) {  // reported by k_rev / k_nn_from_tb otherwise
      const double4 c = nd.gC[(size_t)j * 3 + l];
      fx -= c.x; fy -= c.y; fz -= c.z;
    }
  }
  fx = group_sum<T>(fx); fy = group_sum<T>(fy); fz = group_sum<T>(fz);
  if (E) e = group_sum<T>(e);
  if (t == 0) {
    write_force(a, i, fx, fy, fz);
    if (E) a.e_row[row] = e;
  }
}

template <class R, bool E>
__global__ void __launch_bounds__(256) k_tb_force(RowArgs a, TbP P, const int* __restrict__ row_of,
                                                  const int* __restrict__ rev, const double* __restrict__ B,
                                                  const double* __restrict__ Bp, const double* __restrict__ BT,
                                                  int nb_real) {
  tb_force_rows<R, E, false>(a, P, row_of, rev, B, Bp, BT, NdArgs{}, xcd_block(nb_real));
}

// ------------------------------------------------------------ ljc / morsec

struct CosP {
  double pref, sig, a, r0, delt, R1, R2, invw, nn_coef;
  int morse;
  int whole;  // delt when it is 1, 2, 3 or 4, else 0
  double hw;
};

// x**delt, x >= 0.  FP64: whole exponents up to 4 by products, the third and
// fourth power from the square in two parts (0.50 ulp); the general power is
// about a third of an entry's instructions (the graphene pass of 24,960 rows
// takes 17.3 us and the metal rows 19.2, some 3.5 and 6 more with it; with the
// library's functions 30.1 and 38.2).  The mixed path's power is two
// transcendental instructions for any exponent.
template <class R>
__device__ __forceinline__ R cos_power(const CosP& P, R x) {
  if constexpr (sizeof(R) == 8) {
    if (P.whole) {  // uniform
      const R x2 = x * x, l = fma(x, x, -x2);
      return P.whole == 1 ? x : P.whole == 2 ? x2 : P.whole == 3 ? fma(x2, x, l * x) : fma(x2, x2, (l + l) * x2);
    }
  }
  return PM<R>::pow_(x, R(P.delt));
}

template <class R>
__device__ __forceinline__ void cos_pair(const CosP& P, R r, R ir, R nd, R nnorm_r, R& A, R& Bc, R& S_coef,
                                         R& epair) {
  const R R1 = P.R1, R2 = P.R2, invw = P.invw, delt = P.delt, kdf = cutoff_kdf<R>(P);
  R fc, dfr;
  cutoff_bl<R>(r, R1, R2, invw, kdf, fc, dfr);
  R dfc = dfr * ir;
  R V2;
  if (P.morse) V2 = PM<R>::exp_(-R(P.a) * (r - R(P.r0)));
  else { R s = R(P.sig) * ir, s2 = s * s; V2 = s2 * s2 * s2; }
  R V1 = V2 * V2;
  R c = nd < R(0) ? -nd : nd;
  R V3 = cos_power<R>(P, c * nnorm_r);
  R ind = PM<R>::rcp(nd);
  if (P.morse) {
    A = (R(2) * (R(P.a) * V1 - (R(P.a) + delt * ir) * V2 * V3) * ir * fc - (V1 - R(2) * V2 * V3) * dfc);
    Bc = R(2) * delt * V2 * V3 * ind * fc;
    epair = V1 - R(2) * V2 * V3;
  } else {
    A = ((R(12) * V1 - (R(6) + delt) * V2 * V3) * ir * ir * fc - (V1 - V2 * V3) * dfc);
    Bc = delt * V2 * V3 * ind * fc;
    epair = V1 - V2 * V3;
  }
  epair *= fc;
  S_coef = V2 * V3 * fc * ind;
}

// Coefficients of the normal-derivative term (*_forces_for_graphene second
// loop, MorseCosine.f90:81-107), per graphene atom j.  For the l-th of j's
// three nearest neighbours i, the reference's sum over j's metal neighbours p
// of  c V2 V3 fc /(den (n_j.dr_jp)) (dr_jp . W) n_j  is linear in dr_jp, so
// it equals  c/den (S_j . W) n_j  with S_j = sum_p V2 V3 fc/(n_j.dr_jp) dr_jp.
// Lanes l = t, t+T, .. of row j store that vector for i = its l-th nearest
// neighbour, in FP64.  The FP64 path takes dr from the FP64 positions; the
// mixed path from the fixed-point records it already reads (the exact wrapped
// difference, in FP64: within two quantisation steps, 2.7e-8 A at L = 115 A).
template <int T, class R>
__device__ __forceinline__ void cos_nn_coef(const RowArgs& a, const CosP& P, const int* __restrict__ nn, int row,
                                            int i, int t, double sx, double sy, double sz, const double4& g,
                                            double4* __restrict__ gC) {
  if (t >= 3) return;
  double d[3][3];
  if constexpr (sizeof(R) == 8) {
    const Geo<double> G = geo_of<double>(a, i);
    const double4 pj = G.at(i);
    for (int k = 0; k < 3; ++k) G.d2(pj, G.at(nn[(size_t)row * 3 + k]), d[k][0], d[k][1], d[k][2]);
  } else {
    const double3 L = a.rep ? a.rdev[a.rep[i]].L : a.L;
    const double hx = L.x / 4294967296.0, hy = L.y / 4294967296.0, hz = L.z / 4294967296.0;
    const uint4 pj = a.qpos[i];
    for (int k = 0; k < 3; ++k) {
      const uint4 q = a.qpos[nn[(size_t)row * 3 + k]];
      d[k][0] = (double)(int)(q.x - pj.x) * hx;
      d[k][1] = (double)(int)(q.y - pj.y) * hy;
      d[k][2] = (double)(int)(q.z - pj.z) * hz;
    }
  }
  for (int l1 = t; l1 < 3; l1 += T) {
    int l2 = (l1 + 1) % 3, l3 = (l1 + 2) % 3;
    double d12[3], d31[3], d23[3];
    for (int k = 0; k < 3; ++k) {
      d12[k] = d[l2][k] - d[l1][k];
      d31[k] = d[l1][k] - d[l3][k];
      d23[k] = d[l3][k] - d[l2][k];
    }
    double s1212 = d12[0] * d12[0] + d12[1] * d12[1] + d12[2] * d12[2];
    double s3131 = d31[0] * d31[0] + d31[1] * d31[1] + d31[2] * d31[2];
    double s1231 = d12[0] * d31[0] + d12[1] * d31[1] + d12[2] * d31[2];
    double s2331 = d23[0] * d31[0] + d23[1] * d31[1] + d23[2] * d31[2];
    double s2312 = d23[0] * d12[0] + d23[1] * d12[1] + d23[2] * d12[2];
    double den = s1212 * s3131 - s1231 * s1231;
    double w = sx * (d12[0] * s2331 - d31[0] * s2312) + sy * (d12[1] * s2331 - d31[1] * s2312) +
               sz * (d12[2] * s2331 - d31[2] * s2312);
    double c = P.nn_coef * w / den;
    gC[(size_t)i * 3 + l1] = make_double4(c * g.x, c * g.y, c * g.z, 0);
  }
}

// graphene side, pair and normal terms (*_forces_for_graphene first loop).
// The row's own normal (graphenenorm.f90:38-56) is formed here from its three
// nearest neighbours (rows of nl(3) are the rows of nl(1)) and stored for the
// metal pass (gnorm, and gnf in FP32 for the mixed path); with nearest
// neighbours, the row's normal-derivative coefficients go to gC.
template <int T, class R, bool E>
__device__ __forceinline__ void cos_graphene_rows(const RowArgs& a, const CosP& P, const int* __restrict__ nn,
                                                  int simplified, double4* __restrict__ gnorm,
                                                  float4* __restrict__ gnf, double4* __restrict__ gC, int blk) {
  ROW_PROLOGUE_AT(T, blk)
  double4 g;
  if (simplified) {
    g = make_double4(0, 0, 1, 1);
  } else {
    R d[3][3];
    for (int k = 0; k < 3; ++k) G.d2(pi, G.at(nn[(size_t)row * 3 + k]), d[k][0], d[k][1], d[k][2]);
    R ax = d[1][0] - d[0][0], ay = d[1][1] - d[0][1], az = d[1][2] - d[0][2];
    R bx = d[0][0] - d[2][0], by = d[0][1] - d[2][1], bz = d[0][2] - d[2][2];
    R gx = ay * bz - az * by, gy = az * bx - ax * bz, gz = ax * by - ay * bx;
    if (gz < R(0)) { gx = -gx; gy = -gy; gz = -gz; }
    R inv = R(1) / PM<R>::sqrt_(gx * gx + gy * gy + gz * gz);
    g = make_double4(gx * inv, gy * inv, gz * inv, 0);
    // 1/|n| of the rounded components, for the FP64 metal pass
    if (sizeof(R) == 8) g.w = 1.0 / sqrt(g.x * g.x + g.y * g.y + g.z * g.z);
  }
  const R nx = g.x, ny = g.y, nz = g.z, R2 = P.R2, pref = P.pref;
  RowAcc<R> acc, sacc;  // force and energy; S
  walk_row<T, R>(G, nbrow, n, t, i, [&](int, const typename Geo<R>::P& q, bool valid) {
    R dx, dy, dz;
    R r, ir;
    dist_and_inverse<R>(G.d2(pi, q, dx, dy, dz), r, ir);
    R nd = nx * dx + ny * dy + nz * dz;
    R A, Bc, Sc, ep;
    cos_pair<R>(P, r, ir, nd, ir, A, Bc, Sc, ep);
    const bool in = valid && inside<R>(r, R2);
    A = in ? A * pref : R(0);
    Bc = in ? Bc * pref : R(0);
    Sc = in ? Sc : R(0);
    acc.sub(A * dx + Bc * nx, A * dy + Bc * ny, A * dz + Bc * nz);
    sacc.add(Sc * dx, Sc * dy, Sc * dz);
    if (E) {
      const R v = ep * pref;
      acc.energy(in ? v : R(0));
    }
  }, [&] { acc.flush(); sacc.flush(); });
  const double fx = group_sum<T>(acc.fx), fy = group_sum<T>(acc.fy), fz = group_sum<T>(acc.fz);
  const double e = E ? group_sum<T>(acc.e) : 0.0;
  if (!simplified) {
    const double sx = group_sum<T>(sacc.fx), sy = group_sum<T>(sacc.fy), sz = group_sum<T>(sacc.fz);
    cos_nn_coef<T, R>(a, P, nn, row, i, t, sx, sy, sz, g, gC);
  }
  if (t == 0) {
    write_force(a, i, fx, fy, fz);
    gnorm[i] = g;
    if (sizeof(R) == 4) gnf[i] = make_float4((float)g.x, (float)g.y, (float)g.z, 0.f);
    if (E) a.e_row[row] = e;
  }
}

template <int T, class R, bool E>
__global__ void __launch_bounds__(PAIR_BLOCK) k_cos_graphene(RowArgs a, CosP P, const int* __restrict__ nn,
                                                             int simplified, double4* __restrict__ gnorm,
                                                             float4* __restrict__ gnf, double4* __restrict__ gC,
                                                             int nb_real) {
  cos_graphene_rows<T, R, E>(a, P, nn, simplified, gnorm, gnf, gC, xcd_block(nb_real));
}

// normal-derivative rows (*_forces_for_graphene second loop): row i adds, for
// each of its three nearest neighbours j, the vector that j's graphene pass
// stored for i's place l in j's nearest-neighbour row (cos_nn_coef)
__device__ __forceinline__ void cos_nn_rows(const RowArgs& a, const int* __restrict__ row_of,
                                            const int* __restrict__ rev, const double4* __restrict__ gC, int block) {
  int lb = block;
  int row = lb * blockDim.x + threadIdx.x;
  if (row >= a.nrows) return;
  const int i = a.rows[row];
  const int n = a.nnum[row];
  const int* nbrow = a.nbr + (size_t)row * a.stride;
  int jj[3], ll[3];
  for (int q = 0; q < 3; ++q) {
    jj[q] = n == 3 ? nbrow[q] : 0;
    ll[q] = n == 3 ? rev[(size_t)row * 3 + q] : -1;
  }
  int jr[3];
  double4 c[3];
  for (int q = 0; q < 3; ++q) {
    jr[q] = row_of[jj[q]];
    const bool ok = ll[q] >= 0 && ll[q] <= 2;  // reported by k_rev / k_nn_from_tb otherwise
    c[q] = ok ? gC[(size_t)jj[q] * 3 + ll[q]] : make_double4(0, 0, 0, 0);
    if (!ok) jr[q] = -1;
  }
  double fx = 0, fy = 0, fz = 0;
  for (int q = 0; q < 3; ++q) {
    if (jr[q] < 0) continue;
    fx -= c[q].x; fy -= c[q].y; fz -= c[q].z;
  }
  write_force(a, i, fx, fy, fz);
}

__global__ void __launch_bounds__(256) k_cos_nn(RowArgs a, const int* __restrict__ row_of, const int* __restrict__ rev,
                                                const double4* __restrict__ gC, int nb_real) {
  int lb = xcd_block(nb_real);
  if (lb < 0) return;
  cos_nn_rows(a, row_of, rev, gC, lb);
}

// metal side (*_forces_for_other_atoms): rows of nl(2), neighbours are
// graphene atoms whose normal enters V3 (morsec divides by |n|); the mixed
// path gathers the FP32 copy of the normals (the same values it rounds to).
// Only the rows with entries run, from the work list k_mark_rows builds with
// the list (most metal atoms lie out of reach of the sheet); the pass always
// adds to forces an earlier pass has written, so the other rows keep theirs.
// Work items take hardware block order, which spreads the short list over
// all XCDs.
template <int T, class R>
__device__ __forceinline__ void cos_metal_rows(const RowArgs& a, const CosP& P, const double4* __restrict__ gnorm,
                                               const float4* __restrict__ gnf, const int* __restrict__ mrows,
                                               int block) {
  const int w = (block * blockDim.x + threadIdx.x) / T, t = threadIdx.x & (T - 1);
  if (w >= mrows[a.nrows]) return;
  const int row = mrows[w];
  const int i = a.rows[row];
  const Geo<R> G = geo_of<R>(a, i);
  const typename Geo<R>::P pi = G.at(i);
  const int n = a.nnum[row];
  const int* nbrow = a.nbr + (size_t)row * a.stride;
  const R R2 = P.R2, pref = P.pref;
  RowAcc<R> acc;
  auto f = [&](int, const typename Geo<R>::P& q, const auto& g, bool valid) {
    R dx, dy, dz;
    R r, ir;
    dist_and_inverse<R>(G.d2(pi, q, dx, dy, dz), r, ir);
    const R gx = g.x, gy = g.y, gz = g.z;
    R nd = gx * dx + gy * dy + gz * dz;
    R inr;  // 1/(|n| r)
    if constexpr (sizeof(R) == 8) inr = P.morse ? ir * g.w : ir;
    else inr = P.morse ? PM<R>::rcp(PM<R>::sqrt_(gx * gx + gy * gy + gz * gz) * r) : ir;
    R A, Bc, Sc, ep;
    cos_pair<R>(P, r, ir, nd, inr, A, Bc, Sc, ep);
    const bool in = valid && inside<R>(r, R2);
    A = in ? A * pref : R(0);
    Bc = in ? Bc * pref : R(0);
    acc.sub(A * dx + Bc * gx, A * dy + Bc * gy, A * dz + Bc * gz);
  };
  auto flush = [&] { acc.flush(); };
  if constexpr (sizeof(R) == 4) walk_row_aux<T, R>(G, nbrow, n, t, i, gnf, f, flush);
  else walk_row_aux<T, R>(G, nbrow, n, t, i, gnorm, f, flush);
  const double fx = group_sum<T>(acc.fx), fy = group_sum<T>(acc.fy), fz = group_sum<T>(acc.fz);
  if (t == 0) write_force(a, i, fx, fy, fz);
}

template <int T, class R>
__global__ void __launch_bounds__(PAIR_BLOCK) k_cos_metal(RowArgs a, CosP P, const double4* __restrict__ gnorm,
                                                          const float4* __restrict__ gnf,
                                                          const int* __restrict__ mrows, int nb_real) {
  if ((int)blockIdx.x >= nb_real) return;
  cos_metal_rows<T, R>(a, P, gnorm, gnf, mrows, blockIdx.x);
}

// the normal-derivative rows (graphene atoms) and the metal rows in one
// launch, for groups without common atoms (every force is written once):
// blocks [0, nb_nn) take the graphene rows, the rest the metal work list
template <int T, class R>
__global__ void __launch_bounds__(256) k_cos_nn_metal(RowArgs an, RowArgs am, CosP P, const int* __restrict__ row_of,
                                                      const int* __restrict__ rev, const double4* __restrict__ gC,
                                                      const double4* __restrict__ gnorm, const float4* __restrict__ gnf,
                                                      const int* __restrict__ mrows, int nb_nn, int nb_real) {
  const int lb = blockIdx.x;
  if (lb >= nb_real) return;
  if (lb < nb_nn) cos_nn_rows(an, row_of, rev, gC, lb);
  else cos_metal_rows<T, R>(am, P, gnorm, gnf, mrows, lb - nb_nn);
}

// ------------------------------------------------ passes sharing a launch
//
// lj, lj1g and rjl passes whose rows write disjoint atoms (the species of a
// gas, the replicas of a batch that hold other materials) run as sub-ranges
// of one launch: a binary gas's lj1g A and B rows and a batch's rjl
// densities together, then the lj rows of both directions and the rjl
// forces.  Block b belongs to the last sub-range starting at or before it;
// each sub-range is XCD-remapped on its own.

#define MULTI_MAXP 6
enum MultiKind { MK_LJ1G = 0, MK_LJ = 1, MK_RJL_DENSITY = 2, MK_RJL_FORCE = 3, MK_LJ_BOTH = 4 };
struct MultiPass {
  int kind, start, np, nb;  // first block of the sub-range, its padded and real block counts
  RowArgs a;
  union {
    RjlP rjl;
    LjP lj;
    Lj1gP lj1g;
  } p;
  double* eb;
  LjRows lj;  // MK_LJ_BOTH
};
struct MultiArgs {
  int n;
  MultiPass s[MULTI_MAXP];
  KeArgs ke;
};

// KeArgs: the block's kinetic-energy partials from the forces its rows wrote
// (a mixed gas of 4,000 atoms: the launch 7.1 us for 5.7, in place of a
// k_kick2_ke of 3.1 us that reads the forces again)
__device__ __forceinline__ void ke_parts(const KeArgs& K, const RowForce& f) {
  __shared__ double sh[2 * RED_THREADS];
  double ke = 0.0;
  uint32_t m = 0u;
  if (f.i >= 0) {
    m = K.mask[f.i];
    double4 v = K.vel[f.i];
    kick2_atom(v, make_double4(f.x, f.y, f.z, 0.0), kick_factor(v.w), m, K.P, false);
    ke = v.w * (v.x * v.x + v.y * v.y + v.z * v.z) / 2 * PFM_MASS_COEF;
  }
#pragma unroll 1
  for (int q = 0; q < K.Q.nq; ++q) {
    const CSum s = block_csum(CSum{(m & K.Q.bit[q]) ? ke : 0.0, 0.0}, sh);
    if (threadIdx.x == 0) put_part(K.part, q, K.nb, blockIdx.x, s);
  }
  if (K.C0 && blockIdx.x == 0)
    for (int j = threadIdx.x; j < K.cw; j += RED_THREADS) K.C0[j] = K.C[j];
}

template <int T, class R, bool E>
__global__ void __launch_bounds__(256) k_multi(MultiArgs A) {
  const int b = blockIdx.x;
  int k = 0;
  while (k + 1 < A.n && b >= A.s[k + 1].start) ++k;
  const MultiPass& S = A.s[k];
  const int lb = xcd_local(b - S.start, S.np, S.nb);
  RowForce f;
  if (lb >= 0) {
    switch (S.kind) {
      case MK_LJ1G: f = lj1g_rows<T, R, E>(S.a, S.p.lj1g, lb); break;
      case MK_LJ: f = lj_rows<T, R, E>(S.a, S.p.lj, lb); break;
      case MK_LJ_BOTH: f = lj_both_rows<T, R, E>(S.a, S.p.lj1g, S.lj, lb); break;
      case MK_RJL_DENSITY: rjl_density_rows<T, R>(S.a, S.p.rjl, S.eb, lb); break;
      default: rjl_force_rows<T, R, E>(S.a, S.p.rjl, S.eb, lb); break;
    }
  }
  if (A.ke.nb) ke_parts(A.ke, f);
}

// ------------------------------------------------- graphene on a metal
//
// With rjl on the metal, tb on the graphene and ljc/morsec between them (no
// common atom), the passes of the two sides share launches: the graphene
// passes are short rows (three bonds, or about forty metal entries) whose
// blocks wait on chains of dependent loads, and on their own they fill a
// fraction of the GPU.  Three launches replace six:
//   first:  tb bond orders (graphene rows) | rjl densities (metal rows)
//   second: ljc/morsec graphene pass       | rjl forces
//   third:  tb forces + normal-derivative  | ljc/morsec metal rows
// The graphene range comes first in each grid, so its long blocks start
// early; each range is XCD-remapped on its own (the metal work list keeps
// hardware order).  Every atom's force is summed by one row per launch.

template <int T, class R>
__global__ void __launch_bounds__(256) k_gm_first(RowArgs ac, TbP Pt, double* __restrict__ B, double* __restrict__ Bp,
                                                  double* __restrict__ BT, int npc, int nbc, RowArgs am, RjlP Pr,
                                                  double* __restrict__ eb, int npm, int nbm) {
  const int b = blockIdx.x;
  if (b < npc) {
    const int lb = xcd_local(b, npc, nbc);
    if (lb >= 0) tb_bond_rows<R>(ac, Pt, B, Bp, BT, lb);
  } else {
    const int lb = xcd_local(b - npc, npm, nbm);
    if (lb >= 0) rjl_density_rows<T, R>(am, Pr, eb, lb);
  }
}

template <int T, class R, bool E>
__global__ void __launch_bounds__(256) k_gm_second(RowArgs ag, CosP Pc, const int* __restrict__ nn, int simplified,
                                                   double4* __restrict__ gnorm, float4* __restrict__ gnf,
                                                   double4* __restrict__ gC, int npc, int nbc, RowArgs am, RjlP Pr,
                                                   const double* __restrict__ eb, int npm, int nbm) {
  const int b = blockIdx.x;
  if (b < npc) {
    const int lb = xcd_local(b, npc, nbc);
    if (lb >= 0) cos_graphene_rows<(T < 4 ? T : 4), R, E>(ag, Pc, nn, simplified, gnorm, gnf, gC, lb);
  } else {
    const int lb = xcd_local(b - npc, npm, nbm);
    if (lb >= 0) rjl_force_rows<T, R, E>(am, Pr, eb, lb);
  }
}

template <int T, class R, bool E, bool ND>
__global__ void __launch_bounds__(256) k_gm_third(RowArgs at, TbP Pt, const int* __restrict__ row_of,
                                                  const int* __restrict__ rev, const double* __restrict__ B,
                                                  const double* __restrict__ Bp, const double* __restrict__ BT,
                                                  NdArgs nd, int npc, int nbc, RowArgs amet, CosP Pc,
                                                  const double4* __restrict__ gnorm, const float4* __restrict__ gnf,
                                                  const int* __restrict__ mrows, int nbm) {
  const int b = blockIdx.x;
  if (b < npc) {
    const int lb = xcd_local(b, npc, nbc);
    if (lb >= 0) tb_force_rows<R, E, ND>(at, Pt, row_of, rev, B, Bp, BT, nd, lb);
  } else if (b - npc < nbm) {
    cos_metal_rows<T, R>(amet, Pc, gnorm, gnf, mrows, b - npc);
  }
}

// ----------------------------------------------------------------- dispatch

static RowArgs row_args(pfm_ctx* h, Inter& it, int k, int accumulate) {
  ListDev& L = it.nl[k];
  RowArgs a;
  a.nrows = L.nrows;
  a.stride = L.stride;
  a.rows = h->grp.rows[L.g1];
  a.nnum = L.nnum;
  a.nbr = L.nbr;
  a.pos = h->pos4;
  a.qpos = h->qpos;
  a.hq = make_float3((float)(h->box[0] / 4294967296.0), (float)(h->box[1] / 4294967296.0),
                     (float)(h->box[2] / 4294967296.0));
  a.hb = make_double3(h->hbox[0], h->hbox[1], h->hbox[2]);
  a.L = make_double3(h->box[0], h->box[1], h->box[2]);
  a.iL = make_double3(1.0 / h->box[0], 1.0 / h->box[1], 1.0 / h->box[2]);
  a.rep = h->rep;
  a.rdev = h->rdev;
  a.hiso = (a.hq.x == a.hq.y && a.hq.y == a.hq.z) ? a.hq.x : 0.0f;
  a.frc = h->frc4;
  a.accumulate = accumulate;
  a.e_row = it.e_row;
  return a;
}

static int row_blocks(int nrows, int T, int block) { return (int)(((long)nrows * T + block - 1) / block); }

// lanes per row of an interaction's separately launched row passes (the
// co-scheduled launches take the handle's count for all their passes)
static int pass_lanes(const pfm_ctx* h, const Inter& it) { return it.lanes ? it.lanes : h->lanes; }

#define DISPATCH_T(T_, ...)                       \
  switch (T_) {                                   \
    case 1: { constexpr int T = 1; __VA_ARGS__; } break;   \
    case 2: { constexpr int T = 2; __VA_ARGS__; } break;   \
    case 4: { constexpr int T = 4; __VA_ARGS__; } break;   \
    case 16: { constexpr int T = 16; __VA_ARGS__; } break; \
    case 32: { constexpr int T = 32; __VA_ARGS__; } break; \
    default: { constexpr int T = 8; __VA_ARGS__; } break;  \
  }

// the lane counts of the co-scheduled launches
#define DISPATCH_T3(T_, ...)                                 \
  switch (T_) {                                            \
    case 4: { constexpr int T = 4; __VA_ARGS__; } break;   \
    case 16: { constexpr int T = 16; __VA_ARGS__; } break; \
    default: { constexpr int T = 8; __VA_ARGS__; } break;  \
  }

// pi/(2 (R2 - R1)) of a cosine cutoff (hw of the parameters)
static double half_width(double R1, double R2) { return 0.5 * PFM_PI / (R2 - R1); }
static TbP tb_params(const Inter& it) {
  return TbP{it.p[0], it.p[1], it.p[2], it.p[3], it.p[4], it.p[5], it.p[6] * it.p[6], it.p[7] * it.p[7],
             it.p[8], it.p[9], 1.0 / (it.p[9] - it.p[8]), half_width(it.p[8], it.p[9])};
}
static RjlP rjl_params(const Inter& it) {
  return RjlP{it.p[0], it.p[1], it.p[2], it.p[3], it.p[4], it.p[5], it.p[6], 1.0 / (it.p[6] - it.p[5]),
              half_width(it.p[5], it.p[6])};
}
static CosP cos_params(const Inter& it) {
  const bool morse = it.kind == PFM_MORSEC;
  const double delt = morse ? it.p[3] : it.p[2];
  const int whole = delt == 1.0 || delt == 2.0 || delt == 3.0 || delt == 4.0 ? (int)delt : 0;
  if (morse)
    return CosP{it.p[0], 0.0, it.p[2], it.p[1], delt, it.p[4], it.p[5], 1.0 / (it.p[5] - it.p[4]),
                2.0 * it.p[0] * delt, 1, whole, half_width(it.p[4], it.p[5])};
  return CosP{4.0 * it.p[0], it.p[1], 0.0, 0.0, delt, it.p[3], it.p[4], 1.0 / (it.p[4] - it.p[3]),
              4.0 * it.p[0] * delt, 0, whole, half_width(it.p[3], it.p[4])};
}

static LjP lj_params(const Inter& it) {
  return LjP{4.0 * it.p[0], it.p[1], it.p[2], it.p[3], 1.0 / (it.p[3] - it.p[2]), half_width(it.p[2], it.p[3])};
}
static Lj1gP lj1g_params(const Inter& it) {
  double eps = it.p[0], sig = it.p[1], s6 = sig * sig * sig * sig * sig * sig;
  return Lj1gP{4.0 * eps * s6, 4.0 * eps * s6 * s6, 6.0 * 4.0 * eps * s6, 12.0 * 4.0 * eps * s6 * s6,
               it.p[2], it.p[3], 1.0 / (it.p[3] - it.p[2])};
}

// Phases of lj / lj1g / rjl passes (an lj1g takes the lj list of its own rows
// into its pass): each pass goes into the earliest phase
// after its prerequisite (an rjl force after its density) holding no pass
// that writes any of its atoms (forces, or the density's per-atom value).
// Worth it when fewer launches result; other interactions keep separate
// launches (plan not taken).
static void plan_multi(pfm_ctx* h) {
  auto& M = h->mp;
  M.planned = true;
  M.ok = false;
  M.phases.clear();
  struct P {
    pfm_ctx::MultiPlan::Pass pass;
    int group, after;
  };
  std::vector<P> passes;
  // an lj list whose rows are an lj1g's rows goes into that lj1g's pass
  std::vector<std::pair<int, int>> taken;
  auto partner = [&](int g) -> std::pair<int, int> {
    for (size_t jj = 0; jj < h->inter.size(); ++jj)
      for (int k = 0; k < 2; ++k) {
        const std::pair<int, int> c{(int)jj, k};
        if (h->inter[jj].kind == PFM_LJ && h->inter[jj].nl[k].g1 == g &&
            std::find(taken.begin(), taken.end(), c) == taken.end())
          return c;
      }
    return {-1, 0};
  };
  size_t launches = 0;  // of the passes one by one
  for (size_t ii = 0; ii < h->inter.size(); ++ii) {
    const Inter& it = h->inter[ii];
    if (it.kind == PFM_LJ1G) {
      const auto c = partner(it.nl[0].g1);
      if (c.first >= 0) taken.push_back(c);
      passes.push_back({{(int)ii, c.first >= 0 ? MK_LJ_BOTH : MK_LJ1G, 0, false, c.first, c.second}, it.nl[0].g1, -1});
      launches += c.first >= 0 ? 2 : 1;
    }
  }
  for (size_t ii = 0; ii < h->inter.size(); ++ii) {
    const Inter& it = h->inter[ii];
    const int I = (int)ii;
    if (it.kind == PFM_LJ) {
      for (int k = 0; k < 2; ++k)
        if (std::find(taken.begin(), taken.end(), std::make_pair(I, k)) == taken.end()) {
          passes.push_back({{I, MK_LJ, k, false, -1, 0}, it.nl[k].g1, -1});
          ++launches;
        }
    } else if (it.kind == PFM_RJL) {
      passes.push_back({{I, MK_RJL_DENSITY, 0, false, -1, 0}, it.nl[0].g1, -1});
      passes.push_back({{I, MK_RJL_FORCE, 0, false, -1, 0}, it.nl[0].g1, (int)passes.size() - 1});
      launches += 2;
    } else if (it.kind != PFM_LJ1G) {
      return;
    }
  }
  if (passes.size() > MULTI_MAXP) return;
  // groups sharing an atom
  auto overlap = [&](int g1, int g2) {
    if (g1 == g2) return true;
    std::vector<char> in(h->N, 0);
    for (int x : h->grp.idx[g1]) in[x] = 1;
    for (int x : h->grp.idx[g2])
      if (in[x]) return true;
    return false;
  };
  std::vector<int> phase_of(passes.size(), 0);
  int nphase = 0;
  for (size_t a = 0; a < passes.size(); ++a) {
    int ph = passes[a].after >= 0 ? phase_of[passes[a].after] + 1 : 0;
    for (;; ++ph) {
      bool clash = false;
      for (size_t b = 0; b < a && !clash; ++b) {
        if (phase_of[b] != ph) continue;
        // a density and a force pass of one atom set write different things,
        // but the force pass of another interaction would read the
        // density's per-atom value while it is written: keep them apart too
        clash = overlap(passes[a].group, passes[b].group);
      }
      if (!clash) break;
    }
    phase_of[a] = ph;
    nphase = std::max(nphase, ph + 1);
  }
  if (nphase >= (int)launches) return;
  M.phases.assign(nphase, {});
  for (size_t a = 0; a < passes.size(); ++a) M.phases[phase_of[a]].push_back(passes[a].pass);
  // first writers in launch order (phases in turn; the passes of a phase
  // hold disjoint atoms): a force pass is first when none of its group's
  // atoms is written earlier; a force pass with some atoms written earlier
  // and some not leaves the plan without first writes
  std::vector<char> written(h->N, 0);
  M.first_ok = true;
  for (auto& ph : M.phases) {
    for (auto& ps : ph) {
      ps.first = false;
      if (ps.kind == MK_RJL_DENSITY) continue;
      const Inter& it = h->inter[ps.inter];
      const auto& members = h->grp.idx[it.nl[ps.list].g1];
      size_t before = 0;
      for (int x : members) before += written[x] ? 1 : 0;
      if (before == 0) ps.first = true;
      else if (before != members.size()) M.first_ok = false;
    }
    for (auto& ps : ph)
      if (ps.first)
        for (int x : h->grp.idx[h->inter[ps.inter].nl[ps.list].g1]) written[x] = 1;
  }
  M.ok = true;
}

// The shared launches write every atom's force first when the plan has first
// writers only (plan_multi), no group changes, and the first writers' rows
// cover every atom now: their groups are disjoint, so the row counts add up
// to N exactly then.
bool multi_first_writes(pfm_ctx* h) {
  if (!h->mp.planned) plan_multi(h);
  const int T = h->lanes;
  if (!h->fuse || !h->mp.ok || !h->mp.first_ok || !h->changes.empty() || (T != 4 && T != 8 && T != 16)) return false;
  long rows = 0;
  for (const auto& ph : h->mp.phases)
    for (const auto& ps : ph)
      if (ps.first) rows += h->inter[ps.inter].nl[ps.list].nrows;
  return rows == h->N;
}

// Blocks of the shared launch when it alone completes every atom's force and
// can form an nvt step's kinetic energies as well (KeArgs), else 0: one phase
// of lj / lj1g passes, each the only writer of its atoms.  Up to 1,024 blocks,
// whose partials every block of the next kick_drift adds up: with 8 lanes
// 32,768 atoms, where that costs what the launch saves (us a step with and
// without, FP64: 8,192 atoms 16.3 and 17.4, 16,000 18.8 and 20.0, 32,000 25.3
// and 25.1; mixed 15.0 and 16.2, 16.8 and 18.0, 21.6 and 21.9).  And what
// red_part holds.
int multi_ke_blocks(pfm_ctx* h) {
  if (h->gm.ok || !multi_first_writes(h) || h->mp.phases.size() != 1 || h->nhc.size() > RED_MAXQ) return 0;
  int nb = 0;
  for (const auto& ps : h->mp.phases[0]) {
    if (!ps.first || (ps.kind != MK_LJ1G && ps.kind != MK_LJ && ps.kind != MK_LJ_BOTH)) return 0;
    const int nrows = h->inter[ps.inter].nl[ps.list].nrows;
    if (nrows) nb += pad8(row_blocks(nrows, h->lanes, 256));
  }
  const size_t room = (size_t)(PFM_MAXI + 1 + RED_MAXQ) * h->red_blocks;
  return nb <= 1024 && h->nhc.size() * nb <= room ? nb : 0;
}

// the phases of h->mp, one launch each.  Every pass adds to forces the kick
// cleared, or with `first` (multi_first_writes) the first writer of each atom
// writes its force.  Returns 1 when the lane count has no variant here.
template <class R>
static int multi_forces(pfm_ctx* h, bool energy, bool first) {
  const int T = h->lanes;
  if (T != 4 && T != 8 && T != 16) return 1;
  const int BS = 256;
  for (const auto& ph : h->mp.phases) {
    MultiArgs A;
    memset(&A, 0, sizeof A);
    int start = 0;
    for (const auto& ps : ph) {
      Inter& it = h->inter[ps.inter];
      MultiPass& S = A.s[A.n];
      S.kind = ps.kind;
      S.a = row_args(h, it, ps.list, first && ps.first ? 0 : 1);
      if (S.a.nrows == 0) continue;
      if (ps.kind == MK_LJ && ps.list == 1) S.a.e_row = nullptr;  // nl(2) rows carry no energy
      if (ps.kind == MK_LJ1G || ps.kind == MK_LJ_BOTH) S.p.lj1g = lj1g_params(it);
      else if (ps.kind == MK_LJ) S.p.lj = lj_params(it);
      else S.p.rjl = rjl_params(it);
      S.eb = h->eb;
      if (ps.kind == MK_LJ_BOTH) {
        Inter& jt = h->inter[ps.inter2];
        const ListDev& L2 = jt.nl[ps.list2];
        S.lj = LjRows{L2.stride, L2.nnum, L2.nbr, ps.list2 == 0 ? jt.e_row : nullptr, lj_params(jt)};
      }
      S.nb = row_blocks(S.a.nrows, T, BS);
      S.np = pad8(S.nb);
      S.start = start;
      start += S.np;
      ++A.n;
    }
    if (A.n == 0) continue;
    if (h->mp_ke.nb) {
      if (h->mp_ke.nb != start) return PFM_E_INVALID;  // the launch multi_ke_blocks counted
      A.ke = h->mp_ke;
    }
    DISPATCH_T3(T, {
      if (energy) PFM_LAUNCH(h, "multi", (k_multi<T, R, true>), start, BS, A);
      else PFM_LAUNCH(h, "multi", (k_multi<T, R, false>), start, BS, A);
    });
  }
  return PFM_OK;
}

// The three co-scheduled launches of graphene on a metal (h->gm); every
// pass adds to forces the step's kick cleared, or with `first`
// (gm_first_writes) the second launch writes them.  Returns 1 when the lane
// count has no fused variant (the caller launches the passes one by one).
template <class R>
static int gm_forces(pfm_ctx* h, bool energy, bool first) {
  const int T = h->lanes;
  if (T != 4 && T != 8 && T != 16) return 1;
  Inter& ir = h->inter[h->gm.rjl];
  Inter& it = h->inter[h->gm.tb];
  Inter& ic = h->inter[h->gm.cos];
  if (ir.nl[0].nrows == 0 || it.nl[0].nrows == 0 || ic.nl[0].nrows == 0) return 1;
  const int BS = 256;
  // with `first` the second launch's passes (graphene rows, rjl forces) write
  // their rows' forces and the third launch adds to them
  const int acc2 = first ? 0 : 1;
  RowArgs am = row_args(h, ir, 0, acc2), at = row_args(h, it, 0, 1), ag = row_args(h, ic, 0, acc2);
  RowArgs amet = row_args(h, ic, 1, 1);
  const RjlP Pr = rjl_params(ir);
  const TbP Pt = tb_params(it);
  const CosP Pc = cos_params(ic);
  const bool morse = ic.kind == PFM_MORSEC;
  const int simp = (int)ic.p[morse ? 6 : 5] ? 1 : 0;
  ListDev& NN = ic.nl[2];
  const bool nd = !simp && NN.nrows > 0;
  double* BT = it.Bp + (size_t)it.nl[0].nrows * it.nl[0].stride;
  const int* row_of_tb = h->grp.row_of[it.nl[0].g1];
  NdArgs ndA{NN.nnum, NN.nbr, NN.rev, h->grp.row_of[NN.g1], ic.gC, NN.stride};
  // blocks of each range
  const int nbt = row_blocks(at.nrows, TB_T, BS), npt = pad8(nbt);
  const int nbm = row_blocks(am.nrows, T, BS), npm = pad8(nbm);
  const int Tg = T < 4 ? T : 4;
  const int nbg = row_blocks(ag.nrows, Tg, BS), npg = pad8(nbg);
  const int nbmet = row_blocks(amet.nrows, T, BS);
  DISPATCH_T3(T, {
    PFM_LAUNCH(h, "gm_first", (k_gm_first<T, R>), npt + npm, BS, at, Pt, it.B, it.Bp, BT, npt, nbt, am, Pr, h->eb,
               npm, nbm);
    if (energy)
      PFM_LAUNCH(h, "gm_second", (k_gm_second<T, R, true>), npg + npm, BS, ag, Pc, NN.nbr, simp, ic.gnorm, ic.gnf,
                 ic.gC, npg, nbg, am, Pr, h->eb, npm, nbm);
    else
      PFM_LAUNCH(h, "gm_second", (k_gm_second<T, R, false>), npg + npm, BS, ag, Pc, NN.nbr, simp, ic.gnorm, ic.gnf,
                 ic.gC, npg, nbg, am, Pr, h->eb, npm, nbm);
    const int g3 = npt + nbmet;
    if (energy && nd)
      PFM_LAUNCH(h, "gm_third", (k_gm_third<T, R, true, true>), g3, BS, at, Pt, row_of_tb, it.nl[0].rev, it.B, it.Bp,
                 BT, ndA, npt, nbt, amet, Pc, ic.gnorm, ic.gnf, ic.mrows, nbmet);
    else if (energy)
      PFM_LAUNCH(h, "gm_third", (k_gm_third<T, R, true, false>), g3, BS, at, Pt, row_of_tb, it.nl[0].rev, it.B, it.Bp,
                 BT, ndA, npt, nbt, amet, Pc, ic.gnorm, ic.gnf, ic.mrows, nbmet);
    else if (nd)
      PFM_LAUNCH(h, "gm_third", (k_gm_third<T, R, false, true>), g3, BS, at, Pt, row_of_tb, it.nl[0].rev, it.B, it.Bp,
                 BT, ndA, npt, nbt, amet, Pc, ic.gnorm, ic.gnf, ic.mrows, nbmet);
    else
      PFM_LAUNCH(h, "gm_third", (k_gm_third<T, R, false, false>), g3, BS, at, Pt, row_of_tb, it.nl[0].rev, it.B,
                 it.Bp, BT, ndA, npt, nbt, amet, Pc, ic.gnorm, ic.gnf, ic.mrows, nbmet);
  });
  return PFM_OK;
}

// The rjl rows and the graphene rows of the second launch write every atom's
// force first when they share no atom (h->gm.first_ok), no group changes are
// pending and their rows add up to N; the first launch writes no force and
// the third only adds.  The conditions under which gm_forces returns 1 are
// excluded here.
bool gm_first_writes(pfm_ctx* h) {
  const int T = h->lanes;
  if (!h->fuse || !h->gm.ok || !h->gm.first_ok || !h->changes.empty() || (T != 4 && T != 8 && T != 16)) return false;
  const Inter& ir = h->inter[h->gm.rjl];
  const Inter& it = h->inter[h->gm.tb];
  const Inter& ic = h->inter[h->gm.cos];
  if (ir.nl[0].nrows == 0 || it.nl[0].nrows == 0 || ic.nl[0].nrows == 0) return false;
  return (long)ir.nl[0].nrows + ic.nl[0].nrows == h->N;
}

template <class R>
static int forces_T(pfm_ctx* h, bool energy, bool first_writes) {
  bool written = !first_writes;  // has any pass written this step's forces yet
  if (h->fuse && h->gm.ok && (written || gm_first_writes(h))) {
    const int rc = gm_forces<R>(h, energy, !written);
    if (rc != 1) return rc;
  }
  if (!h->mp.planned) plan_multi(h);
  if (h->fuse && h->mp.ok && (written || multi_first_writes(h))) {
    const int rc = multi_forces<R>(h, energy, !written);
    if (rc != 1) return rc;
  }
  const int BS = std::min(h->block, PairBlock<R>::max);  // row passes (T lanes per row)
  const int BS1 = 256;           // one-lane-per-row passes (tb, cos_nn)
  for (size_t ii = 0; ii < h->inter.size(); ++ii) {
    Inter& it = h->inter[ii];
    switch (it.kind) {
      case PFM_RJL: {
        RowArgs a = row_args(h, it, 0, written ? 1 : 0);
        if (a.nrows == 0) break;
        const RjlP P = rjl_params(it);
        int T = pass_lanes(h, it);
        DISPATCH_T(T, {
          int nb = row_blocks(a.nrows, T, BS);
          PFM_LAUNCH(h, "rjl_density", (k_rjl_density<T, R>), pad8(nb), BS, a, P, h->eb, nb);
          if (energy) PFM_LAUNCH(h, "rjl_force", (k_rjl_force<T, R, true>), pad8(nb), BS, a, P, h->eb, nb);
          else PFM_LAUNCH(h, "rjl_force", (k_rjl_force<T, R, false>), pad8(nb), BS, a, P, h->eb, nb);
        });
        written = true;
        break;
      }
      case PFM_LJ: {
        const LjP P = lj_params(it);
        for (int k = 0; k < 2; ++k) {
          RowArgs a = row_args(h, it, k, written ? 1 : 0);
          if (a.nrows == 0) continue;
          bool E = energy && k == 0;
          int T = pass_lanes(h, it);
          DISPATCH_T(T, {
            int nb = row_blocks(a.nrows, T, BS);
            if (E) PFM_LAUNCH(h, "lj", (k_lj<T, R, true>), pad8(nb), BS, a, P, nb);
            else PFM_LAUNCH(h, "lj", (k_lj<T, R, false>), pad8(nb), BS, a, P, nb);
          });
          written = true;
        }
        break;
      }
      case PFM_LJ1G: {
        RowArgs a = row_args(h, it, 0, written ? 1 : 0);
        if (a.nrows == 0) break;
        const Lj1gP P = lj1g_params(it);
        int T = pass_lanes(h, it);
        DISPATCH_T(T, {
          int nb = row_blocks(a.nrows, T, BS);
          if (energy) PFM_LAUNCH(h, "lj1g", (k_lj1g<T, R, true>), pad8(nb), BS, a, P, nb);
          else PFM_LAUNCH(h, "lj1g", (k_lj1g<T, R, false>), pad8(nb), BS, a, P, nb);
        });
        written = true;
        break;
      }
      case PFM_TB: {
        RowArgs a = row_args(h, it, 0, written ? 1 : 0);
        if (a.nrows == 0) break;
        const TbP P = tb_params(it);
        int nb = row_blocks(a.nrows, TB_T, BS1);
        double* BT = it.Bp + (size_t)it.nl[0].nrows * it.nl[0].stride;
        PFM_LAUNCH(h, "tb_bond", (k_tb_bond<R>), pad8(nb), BS1, a, P, it.B, it.Bp, BT, nb);
        const int* row_of = h->grp.row_of[it.nl[0].g1];
        if (energy) PFM_LAUNCH(h, "tb_force", (k_tb_force<R, true>), pad8(nb), BS1, a, P, row_of, it.nl[0].rev, it.B, it.Bp, BT, nb);
        else PFM_LAUNCH(h, "tb_force", (k_tb_force<R, false>), pad8(nb), BS1, a, P, row_of, it.nl[0].rev, it.B, it.Bp, BT, nb);
        written = true;
        break;
      }
      case PFM_REBOSC: {
        int rc = launch_rebo(h, it, energy, written ? 1 : 0);
        if (rc) return rc;
        written = true;
        break;
      }
      case PFM_SUR: {
        int rc = launch_sur_forces(h, it, written ? 1 : 0);
        if (rc) {
          h->err = "error: surrogate parameters not set";
          return rc;
        }
        written = true;
        break;
      }
      case PFM_LJC:
      case PFM_MORSEC: {
        bool morse = it.kind == PFM_MORSEC;
        bool simplified = (int)it.p[morse ? 6 : 5];
        const CosP P = cos_params(it);
        ListDev& NN = it.nl[2];
        RowArgs a = row_args(h, it, 0, written ? 1 : 0);
        int T = pass_lanes(h, it);
        int simp = simplified ? 1 : 0;
        if (a.nrows > 0) {
          // graphene rows hold about 40 metal entries: at most four lanes each
          const int Tg = T > 4 ? 4 : T;
          DISPATCH_T(Tg, {
            int nb = row_blocks(a.nrows, T, BS);
            if (energy) PFM_LAUNCH(h, "cos_graphene", (k_cos_graphene<T, R, true>), pad8(nb), BS, a, P, NN.nbr, simp, it.gnorm, it.gnf, it.gC, nb);
            else PFM_LAUNCH(h, "cos_graphene", (k_cos_graphene<T, R, false>), pad8(nb), BS, a, P, NN.nbr, simp, it.gnorm, it.gnf, it.gC, nb);
          });
          written = true;
        }
        RowArgs c = row_args(h, it, 1, written ? 1 : 0);
        if (c.nrows > 0 && !c.accumulate) {
          // the metal pass skips rows without entries, so it never writes first
          h->err = "error: the ljc/morsec metal pass would write the first forces of its step";
          return PFM_E_INVALID;
        }
        const bool nn = !simplified && NN.nrows > 0;
        if (nn && c.nrows > 0 && it.rows_disjoint && BS == BS1) {
          RowArgs b = row_args(h, it, 2, written ? 1 : 0);
          int nbn = row_blocks(b.nrows, 1, BS1);
          DISPATCH_T(T, {
            int nb = nbn + row_blocks(c.nrows, T, BS1);
            PFM_LAUNCH(h, "cos_nn_metal", (k_cos_nn_metal<T, R>), pad8(nb), BS1, b, c, P, h->grp.row_of[NN.g1],
                       NN.rev, it.gC, it.gnorm, it.gnf, it.mrows, nbn, nb);
          });
          written = true;
          break;
        }
        if (nn) {
          RowArgs b = row_args(h, it, 2, written ? 1 : 0);
          int nb = row_blocks(b.nrows, 1, BS1);
          PFM_LAUNCH(h, "cos_nn", k_cos_nn, pad8(nb), BS1, b, h->grp.row_of[NN.g1], NN.rev, it.gC, nb);
          written = true;
        }
        c.accumulate = written ? 1 : 0;
        if (c.nrows > 0) {
          DISPATCH_T(T, {
            int nb = row_blocks(c.nrows, T, BS);
            PFM_LAUNCH(h, "cos_metal", (k_cos_metal<T, R>), pad8(nb), BS, c, P, it.gnorm, it.gnf, it.mrows, nb);
          });
          written = true;
        }
        break;
      }
    }
  }
  return PFM_OK;
}

int launch_forces(pfm_ctx* h, bool energy, bool first_writes) {
  if (h->precision == PFM_MIXED) return forces_T<float>(h, energy, first_writes);
  return forces_T<double>(h, energy, first_writes);
}
