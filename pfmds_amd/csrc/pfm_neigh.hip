// pfm_neigh.hip -- cell binning, Morton re-sort of the atoms and neighbour-list
// construction on gfx950.
//
// Replaces find_neighbours (md_neighbours.f90:56-100, brute force over all
// N1*N2 pairs), converce_neighbour_list (md_neighbours.f90:128-160, a serial
// transpose) and find_gr_nearest_neighbors (graphenenorm.f90:8-36).  The
// membership test is the reference's own: j != i, j in group 2, and
// dr2 < r_cut**2 with find_distance's arithmetic (min_image_dist2), so the
// lists are identical to the reference's as sets.  Lists are rebuilt on the
// reference's schedule (mod(md_step, update_period) == 0); between rebuilds
// nothing is refreshed because the force passes recompute dr from positions.
#include "pfm_internal.h"

// ------------------------------------------------------------------ binning

__device__ __forceinline__ int cell_coord(double x, double inv_len, int nc) {
  int c = (int)floor(x * inv_len);
  return c < 0 ? 0 : (c >= nc ? nc - 1 : c);
}

__global__ void k_fill_int(int n, int* __restrict__ x, int v) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = v;
}

// ctr[key] += 1 for every valid lane of the wavefront, with one atomic per run
// of equal keys in consecutive lanes (atoms arrive nearly in cell order, so
// runs are long); returns the lane's previous count (its slot).  Invalid
// lanes (past the end of the array) are the top lanes of the last wavefront.
__device__ __forceinline__ int run_atomic_inc(int* ctr, int key, bool valid) {
  const int lane = threadIdx.x & 63;
  const int prev = __shfl_up(key, 1);
  const bool head = valid && (lane == 0 || prev != key);
  const unsigned long long heads = __ballot(head);
  const int nvalid = __popcll(__ballot(valid));
  const unsigned long long upto = (2ull << lane) - 1ull;  // lanes 0..lane
  const int start = valid ? 63 - __clzll(heads & upto) : lane;
  const unsigned long long above = heads & ~upto;
  const int next = above ? __ffsll(above) - 1 : 64;
  int base = 0;
  if (head) base = atomicAdd(&ctr[key], (next < nvalid ? next : nvalid) - lane);
  base = __shfl(base, start);
  return base + (lane - start);
}

__global__ void k_cell_keys(int N, const double4* __restrict__ pos, const int* __restrict__ rep,
                            const RepDev* __restrict__ rdev, const int* __restrict__ cell_rank,
                            int* __restrict__ atom_rank, int* __restrict__ cell_count) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < N;
  int r = -1;
  if (valid) {
    const RepDev& R = rdev[rep ? rep[i] : 0];
    double4 p = pos[i];
    int cx = cell_coord(p.x, R.inv_clen.x, R.nc[0]);
    int cy = cell_coord(p.y, R.inv_clen.y, R.nc[1]);
    int cz = cell_coord(p.z, R.inv_clen.z, R.nc[2]);
    r = cell_rank[R.cell_base + (cz * R.nc[1] + cy) * R.nc[0] + cx];
    atom_rank[i] = r;
  }
  run_atomic_inc(cell_count, r, valid);
}

// exclusive scan of n ints by one workgroup of 1024 threads (small n: the
// cell counts, and the block sums of scan_excl below)
__device__ __forceinline__ void scan_excl_wg(int n, const int* __restrict__ in, int* __restrict__ out,
                                             int* __restrict__ total) {
  __shared__ int s[1024];
  int t = threadIdx.x;
  int chunk = (n + 1023) / 1024;
  int b = t * chunk, e = min(n, b + chunk);
  int sum = 0;
  for (int k = b; k < e; ++k) sum += in[k];
  s[t] = sum;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    int v = t >= o ? s[t - o] : 0;
    __syncthreads();
    s[t] += v;
    __syncthreads();
  }
  int run = s[t] - sum;
  for (int k = b; k < e; ++k) {
    int v = in[k];
    out[k] = run;
    run += v;
  }
  if (t == 1023 && total) *total = s[1023];
}

__global__ void __launch_bounds__(1024) k_scan_excl(int n, const int* __restrict__ in, int* __restrict__ out,
                                                    int* __restrict__ total) {
  scan_excl_wg(n, in, out, total);
}

#define SCAN_B 1024  // items per workgroup of the multi-block scan (256 threads x 4)

__device__ __forceinline__ int wg_inclusive_scan(int v, int* sh) {
  int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    int w = t >= o ? sh[t - o] : 0;
    __syncthreads();
    sh[t] += w;
    __syncthreads();
  }
  int r = sh[t];
  __syncthreads();
  return r;
}

__global__ void __launch_bounds__(256) k_scan_blocksum(int n, const int* __restrict__ in, int* __restrict__ bsum) {
  __shared__ int sh[256];
  int base = blockIdx.x * SCAN_B + threadIdx.x * 4, v = 0;
  for (int k = 0; k < 4; ++k)
    if (base + k < n) v += in[base + k];
  int inc = wg_inclusive_scan(v, sh);
  if (threadIdx.x == 255) bsum[blockIdx.x] = inc;
}

__global__ void __launch_bounds__(256) k_scan_apply(int n, const int* __restrict__ in, const int* __restrict__ boff,
                                                    int* __restrict__ out) {
  __shared__ int sh[256];
  int base = blockIdx.x * SCAN_B + threadIdx.x * 4;
  int x[4], v = 0;
  for (int k = 0; k < 4; ++k) {
    x[k] = base + k < n ? in[base + k] : 0;
    v += x[k];
  }
  int run = wg_inclusive_scan(v, sh) - v + boff[blockIdx.x];
  for (int k = 0; k < 4; ++k) {
    if (base + k < n) out[base + k] = run;
    run += x[k];
  }
}

// exclusive scan of n ints; tmp holds ceil(n/1024) block sums and their scan
void scan_excl(pfm_ctx* h, int n, const int* in, int* out, int* tmp) {
  int nb = (n + SCAN_B - 1) / SCAN_B;
  if (n <= 16 * 1024) {
    // one workgroup, up to 16 items a thread: one launch instead of three
    PFM_LAUNCH(h, "scan", k_scan_excl, 1, 1024, n, in, out, (int*)nullptr);
    return;
  }
  PFM_LAUNCH(h, "scan", k_scan_blocksum, nb, 256, n, in, tmp);
  PFM_LAUNCH(h, "scan", k_scan_excl, 1, 1024, nb, tmp, tmp + nb, (int*)nullptr);
  PFM_LAUNCH(h, "scan", k_scan_apply, nb, 256, n, in, tmp + nb, out);
}

__global__ void k_scatter(int N, const int* __restrict__ atom_rank, const int* __restrict__ cell_start,
                          int* __restrict__ cell_fill, int* __restrict__ perm) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < N;
  const int r = valid ? atom_rank[i] : -1;
  const int slot = run_atomic_inc(cell_fill, r, valid);
  if (valid) perm[cell_start[r] + slot] = i;
}

// k_cell_keys, the scan of the counts and k_scatter in one workgroup, the
// counts in LDS: up to BIN_N atoms, whose ranks stay in registers, and BIN_C
// cells.  Three launches of 2.6 to 3.2 us each took longer than one workgroup
// takes for it all (6,312 atoms 7.2 us, 4,000 5.4, 500 3.6; 9.2, 8.4 and 8 in three).
#define BIN_N 8192
#define BIN_C 4096
__global__ void __launch_bounds__(1024) k_bin_small(int N, int ncell, const double4* __restrict__ pos,
                                                    const int* __restrict__ rep, const RepDev* __restrict__ rdev,
                                                    const int* __restrict__ cell_rank, int* __restrict__ cell_start,
                                                    int* __restrict__ cell_tmp, int* __restrict__ perm) {
  __shared__ int cnt[BIN_C];
  __shared__ int wsum[16];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  for (int c = t; c < ncell; c += 1024) cnt[c] = 0;
  // each phase for all of a thread's atoms at once (those past the end repeat
  // the last one): loads of one wait beside those of the others
  constexpr int U = BIN_N / 1024;
  int rank[U], slot[U];
  double4 p[U];
#pragma unroll
  for (int u = 0; u < U && u * 1024 < N; ++u) p[u] = pos[min(u * 1024 + t, N - 1)];
  auto cell_of = [](const double4& x, const RepDev& R) {
    const int cx = cell_coord(x.x, R.inv_clen.x, R.nc[0]);
    const int cy = cell_coord(x.y, R.inv_clen.y, R.nc[1]);
    const int cz = cell_coord(x.z, R.inv_clen.z, R.nc[2]);
    return R.cell_base + (cz * R.nc[1] + cy) * R.nc[0] + cx;
  };
  if (rep) {
#pragma unroll
    for (int u = 0; u < U && u * 1024 < N; ++u) rank[u] = rep[min(u * 1024 + t, N - 1)];
#pragma unroll
    for (int u = 0; u < U && u * 1024 < N; ++u) rank[u] = cell_of(p[u], rdev[rank[u]]);
  } else {
#pragma unroll
    for (int u = 0; u < U && u * 1024 < N; ++u) rank[u] = cell_of(p[u], rdev[0]);
  }
#pragma unroll
  for (int u = 0; u < U && u * 1024 < N; ++u) rank[u] = cell_rank[rank[u]];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u * 1024 >= N) break;
    const bool valid = u * 1024 + t < N;
    slot[u] = run_atomic_inc(cnt, valid ? rank[u] : -1, valid);
  }
  __syncthreads();
  // exclusive scan: BIN_C / 1024 consecutive cells a thread
  int x[BIN_C / 1024], sum = 0;
#pragma unroll
  for (int k = 0; k < BIN_C / 1024; ++k) {
    const int c = t * (BIN_C / 1024) + k;
    x[k] = c < ncell ? cnt[c] : 0;
    sum += x[k];
  }
  int inc = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(inc, o);
    if (lane >= o) inc += v;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  int run = inc - sum;
  for (int k = 0; k < w; ++k) run += wsum[k];
#pragma unroll
  for (int k = 0; k < BIN_C / 1024; ++k) {
    const int c = t * (BIN_C / 1024) + k;
    if (c < ncell) {
      cell_start[c] = run;
      cell_tmp[c] = x[k];
      cnt[c] = run;
    }
    run += x[k];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (u * 1024 + t < N) perm[cnt[rank[u]] + slot[u]] = u * 1024 + t;
}

// the per-atom arrays in their current order (0) and in cell order (1)
struct PermArgs {
  const double4 *p0, *v0, *f0;
  const uint32_t* m0;
  const int *o0, *r0;
  double4 *p1, *v1, *f1;
  uint32_t* m1;
  int *o1, *r1;
  uint4* q1;  // fixed-point copy of the new positions (mixed path), or null
  const RepDev* rdev;
};

// order the atoms of each cell by original index, so the layout (and every
// sum over it) does not depend on the order of the scatter's atomics: one
// 64-lane workgroup per cell, each lane ranks its entries against the cell.
// PERM: every atom's data moves to its new place (the re-sort); otherwise
// the order goes to perm_out (binning without moving the atoms).  Also the
// cell's count for the searches, the union of its group bits (cell_grp,
// which lets a list search skip tiles that hold no candidate), and the
// binning's counters cleared for the next binning.
template <bool PERM>
__global__ void __launch_bounds__(64) k_cell_sort(int ncell, const int* __restrict__ cell_start,
                                                  int* __restrict__ cell_tmp, int* __restrict__ cell_fill,
                                                  int* __restrict__ cell_count, const int* __restrict__ perm_in,
                                                  int* __restrict__ perm_out, const int* __restrict__ orig,
                                                  const uint32_t* __restrict__ mask, uint32_t* __restrict__ cell_grp,
                                                  PermArgs P) {
  __shared__ int key[512];
  int c = blockIdx.x;
  if (c >= ncell) return;
  int s = cell_start[c], n = cell_tmp[c];
  bool lds = n <= 512;
  uint32_t g = 0u;
  if (lds)
    for (int k = threadIdx.x; k < n; k += 64) key[k] = orig[perm_in[s + k]];
  __syncthreads();
  for (int k = threadIdx.x; k < n; k += 64) {
    int v = perm_in[s + k];
    g |= mask[v];
    int rank = 0;
    if (lds) {
      const int kk = key[k];
#pragma unroll 8
      for (int m = 0; m < n; ++m) rank += key[m] < kk ? 1 : 0;
    } else {
      const int kk = orig[v];
      for (int m = 0; m < n; ++m) rank += orig[perm_in[s + m]] < kk ? 1 : 0;
    }
    if constexpr (PERM) {
      const int d = s + rank;
      const double4 p = P.p0[v];
      P.p1[d] = p;
      int r = 0;
      if (P.r0) { r = P.r0[v]; P.r1[d] = r; }
      if (P.q1) P.q1[d] = quantize(p, P.rdev[r].qs, 0u);
      P.v1[d] = P.v0[v];
      P.f1[d] = P.f0[v];
      P.m1[d] = P.m0[v];
      P.o1[d] = P.o0[v];
    } else {
      perm_out[s + rank] = v;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) g |= (uint32_t)__shfl_xor((int)g, o);
  if (threadIdx.x == 0) {
    cell_grp[c] = g;
    cell_count[c] = n;
    cell_tmp[c] = 0;
    cell_fill[c] = 0;
  }
}

// Bin atoms into cells and re-order every per-atom array in Morton cell
// order.  The binning counters (cell_tmp, cell_fill) are zero on entry: the
// allocation clears them and k_cell_sort clears them again for the next call.
int launch_sort_and_bin(pfm_ctx* h, int step, bool permute) {
  (void)step;
  int N = h->N, nb = (N + 255) / 256;
  if (N <= BIN_N && h->ncell <= BIN_C) {
    PFM_LAUNCH(h, "cell_keys", k_bin_small, 1, 1024, N, h->ncell, h->pos4, h->rep, h->rdev, h->cell_rank,
               h->cell_start, h->cell_tmp, h->scan_tmp + N);
  } else {
    PFM_LAUNCH(h, "cell_keys", k_cell_keys, nb, 256, N, h->pos4, h->rep, h->rdev, h->cell_rank, h->atom_rank,
               h->cell_tmp);
    scan_excl(h, h->ncell, h->cell_tmp, h->cell_start, h->scan_tmp);
    PFM_LAUNCH(h, "scatter", k_scatter, nb, 256, N, h->atom_rank, h->cell_start, h->cell_fill, h->scan_tmp + N);
  }
  PermArgs P{h->pos4, h->vel4, h->frc4, h->mask, h->orig, h->rep, h->pos4b, h->vel4b, h->frc4b, h->maskb,
             h->origb, h->repb, h->qpos, h->rdev};
  if (!permute) {
    // lists that are not due keep their internal indices: the search reads
    // the atoms of every cell through the cell-ordered index
    PFM_LAUNCH(h, "cell_sort", k_cell_sort<false>, h->ncell, 64, h->ncell, h->cell_start, h->cell_tmp,
               h->cell_fill, h->cell_count, h->scan_tmp + N, h->perm, h->orig, h->mask, h->cell_grp, P);
    h->bin = h->perm;
    return PFM_OK;
  }
  PFM_LAUNCH(h, "cell_sort", k_cell_sort<true>, h->ncell, 64, h->ncell, h->cell_start, h->cell_tmp, h->cell_fill,
             h->cell_count, h->scan_tmp + N, h->perm, h->orig, h->mask, h->cell_grp, P);
  std::swap(h->pos4, h->pos4b);
  std::swap(h->vel4, h->vel4b);
  std::swap(h->frc4, h->frc4b);
  std::swap(h->mask, h->maskb);
  std::swap(h->orig, h->origb);
  std::swap(h->rep, h->repb);
  h->bin = nullptr;  // atoms are in cell order
  launch_group_rows(h);
  return PFM_OK;
}

// --------------------------------------------------------------- group rows
//
// The rows of up to GR_MAX groups in three launches (one on few atoms,
// k_grp_rows_small) whatever their number:
// per 256-atom block and group the member count (wave ballots), one
// workgroup per group scanning its block counts, then every member's row
// from its block's offset, its wave's offset and its rank in the wave.  Rows
// come out in internal order, as a stable compaction gives them.

#define GR_MAX 8
struct GroupRowsArgs {
  int ng, nb;
  uint32_t bit[GR_MAX];
  int* rows[GR_MAX];
  int* row_of[GR_MAX];
};

__global__ void __launch_bounds__(256) k_grp_count(int N, const uint32_t* __restrict__ mask, GroupRowsArgs G,
                                                   int* __restrict__ cnt) {
  __shared__ int wc[GR_MAX][4];
  const int i = blockIdx.x * 256 + threadIdx.x, w = threadIdx.x >> 6;
  const uint32_t m = i < N ? mask[i] : 0u;
  for (int q = 0; q < G.ng; ++q) {
    const unsigned long long b = __ballot((m & G.bit[q]) != 0);
    if ((threadIdx.x & 63) == 0) wc[q][w] = __popcll(b);
  }
  __syncthreads();
  if (threadIdx.x < G.ng) {
    const int q = threadIdx.x;
    cnt[q * G.nb + blockIdx.x] = wc[q][0] + wc[q][1] + wc[q][2] + wc[q][3];
  }
}

__global__ void __launch_bounds__(1024) k_grp_scan(int nb, int* __restrict__ cnt, int* __restrict__ off) {
  const int q = blockIdx.x;
  scan_excl_wg(nb, cnt + (size_t)q * nb, off + (size_t)q * nb, nullptr);
}

__global__ void __launch_bounds__(256) k_grp_write(int N, const uint32_t* __restrict__ mask, GroupRowsArgs G,
                                                   const int* __restrict__ off) {
  __shared__ int wc[GR_MAX][4];
  const int i = blockIdx.x * 256 + threadIdx.x, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t m = i < N ? mask[i] : 0u;
  unsigned long long bal[GR_MAX];
  for (int q = 0; q < G.ng; ++q) {
    bal[q] = __ballot((m & G.bit[q]) != 0);
    if (lane == 0) wc[q][w] = __popcll(bal[q]);
  }
  __syncthreads();
  if (i >= N) return;
  const unsigned long long below = (1ull << lane) - 1ull;
  for (int q = 0; q < G.ng; ++q) {
    if (m & G.bit[q]) {
      int r = off[q * G.nb + blockIdx.x] + __popcll(bal[q] & below);
      for (int v = 0; v < w; ++v) r += wc[q][v];
      G.rows[q][r] = i;
      G.row_of[q][i] = r;
    } else {
      G.row_of[q][i] = -1;
    }
  }
}

// k_grp_count, k_grp_scan and k_grp_write in one launch: every block counts
// the members in the masks before it for itself, which up to GR_SMALL blocks
// costs less than two launches (6,312 atoms 4.8 us against 3.4 + 3.2 + 4.3)
#define GR_SMALL 32
__global__ void __launch_bounds__(256) k_grp_rows_small(int N, const uint32_t* __restrict__ mask, GroupRowsArgs G) {
  __shared__ int wc[GR_MAX][4], before[GR_MAX][4];
  const int i = blockIdx.x * 256 + threadIdx.x, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t m = i < N ? mask[i] : 0u;
  int cnt[GR_MAX];
#pragma unroll
  for (int q = 0; q < GR_MAX; ++q) cnt[q] = 0;
  for (int b0 = 0; b0 < (int)blockIdx.x; b0 += 8) {
    uint32_t mb[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint32_t x = mask[min(b0 + u, (int)blockIdx.x - 1) * 256 + threadIdx.x];
      mb[u] = b0 + u < (int)blockIdx.x ? x : 0u;
    }
#pragma unroll
    for (int q = 0; q < GR_MAX; ++q) {
      if (q >= G.ng) break;
#pragma unroll
      for (int u = 0; u < 8; ++u) cnt[q] += __popcll(__ballot((mb[u] & G.bit[q]) != 0));
    }
  }
  unsigned long long bal[GR_MAX];
#pragma unroll
  for (int q = 0; q < GR_MAX; ++q) {
    if (q >= G.ng) break;
    bal[q] = __ballot((m & G.bit[q]) != 0);
    if (lane == 0) {
      wc[q][w] = __popcll(bal[q]);
      before[q][w] = cnt[q];
    }
  }
  __syncthreads();
  if (i >= N) return;
  const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
  for (int q = 0; q < GR_MAX; ++q) {
    if (q >= G.ng) break;
    int r = -1;
    if (m & G.bit[q]) {
      r = __popcll(bal[q] & below);
      for (int v = 0; v < 4; ++v) r += before[q][v] + (v < w ? wc[q][v] : 0);
      G.rows[q][r] = i;
    }
    G.row_of[q][i] = r;
  }
}

__global__ void k_identity_rows(int N, int* __restrict__ rows, int* __restrict__ row_of) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < N) { rows[i] = i; row_of[i] = i; }
}

// rows of every group that some list or role uses: members in internal order
void launch_group_rows(pfm_ctx* h) {
  int N = h->N, nb = (N + 255) / 256;
  GroupRowsArgs G{};
  G.nb = nb;
  auto flush = [&]() {
    if (!G.ng) return;
    if (nb <= GR_SMALL) {
      PFM_LAUNCH(h, "group_rows", k_grp_rows_small, nb, 256, N, h->mask, G);
      G.ng = 0;
      return;
    }
    int* cnt = h->scan_tmp;
    int* off = h->scan_tmp + (size_t)GR_MAX * nb;
    PFM_LAUNCH(h, "group_rows", k_grp_count, nb, 256, N, h->mask, G, cnt);
    PFM_LAUNCH(h, "group_rows", k_grp_scan, G.ng, 1024, nb, cnt, off);
    PFM_LAUNCH(h, "group_rows", k_grp_write, nb, 256, N, h->mask, G, off);
    G.ng = 0;
  };
  for (int g = 1; g <= PFM_MAXG; ++g) {
    if (!h->grp.used[g] || h->grp.size[g] == 0) continue;
    // members (a growing group's spare bit), not only the active atoms
    uint32_t bit = 1u << ((h->grp.shadow[g] ? h->grp.shadow[g] : g) - 1);
    if (h->grp.size[g] == N) {
      // every atom is a member: row r is internal atom r whatever the order
      if (!h->grp.ident[g]) PFM_LAUNCH(h, "group_rows", k_identity_rows, nb, 256, N, h->grp.rows[g], h->grp.row_of[g]);
      h->grp.ident[g] = true;
      continue;
    }
    G.bit[G.ng] = bit;
    G.rows[G.ng] = h->grp.rows[g];
    G.row_of[G.ng] = h->grp.row_of[g];
    if (++G.ng == GR_MAX) flush();
  }
  flush();
}

// ------------------------------------------------------------ list building

struct SearchArgs {
  int nrows;
  const int* rows;
  uint32_t g1bit;  // active row atoms; the rows of a growing group hold inactive members with no entries
  uint32_t g1mem;  // members of group 1 (a growing group's spare bit): the atoms that have rows
  uint32_t g2bit;
  const double4* pos;
  const uint32_t* mask;
  const int* orig;
  const RepDev* rdev;   // replica geometry
  const int* rep;       // replica of every internal atom (null: one replica)
  const int* cell_rep;  // replica of every cell (null: one replica)
  const int* cells;     // the cells to search (null: all of them)
  const int* bin;       // atoms of the cells in cell order (null: atoms are stored in cell order)
  double rc2, rc2_lo, rc2_hi;
  const int* cell_rank;
  const int* cell_start;
  const int* cell_count;
  const uint32_t* cell_grp;  // union of the group bits of each cell's atoms
  int nmax, stride;
  int* nnum;
  int* nbr;
  DevErr* err;
  int step, err_code;
  int exact;  // require exactly nmax entries (graphene nearest neighbours)
  // a second list with the same rows, cutoff and rebuild steps searched in
  // the same pass (PAIR): g2bit is then the union
  // of the two candidate groups, g2bit1 / g2bit2 the groups of the two lists
  uint32_t g2bit1, g2bit2;
  int nmax2, stride2;
  int* nnum2;
  int* nbr2;
  // a second pair in the same pass (QUAD):
  // rows of another group (side b, disjoint from group 1), whose two lists
  // take the candidates of g2bit1 (b1) and of g2bit2 (b2); g1mem is then
  // the union of the two row groups' member bits
  uint32_t g1bit_b, g1mem_b;
  const int* row_of_b;
  int nmax_b1, stride_b1, nmax_b2, stride_b2;
  int *nnum_b1, *nbr_b1, *nnum_b2, *nbr_b2;
};

// slot of the row atom inside each neighbour's own row (Tersoff-Brenner's
// `do l=1,nl%nnum(j); if(nl%nlist(l,j)==i) exit` and graphene's l1 search);
// REV_T lanes a row, an entry each (bound by the chain of dependent loads of
// one entry: 3.9 us at 1,664 rows, 6.3 with one lane taking them in turn)
#define REV_T 4
__global__ void __launch_bounds__(256) k_rev(int nrows, const int* __restrict__ rows, const int* __restrict__ row_of,
                                             const int* __restrict__ nnum, const int* __restrict__ nbr, int stride,
                                             int* __restrict__ rev, DevErr* err, const int* __restrict__ orig,
                                             int step) {
  const int gt = blockIdx.x * 256 + threadIdx.x, r = gt / REV_T;
  if (r >= nrows) return;
  const int i = rows[r], n = nnum[r];
  for (int p = gt & (REV_T - 1); p < n; p += REV_T) {
    const int jr = row_of[nbr[(size_t)r * stride + p]];
    int l = -1;
    if (jr >= 0) {
      const int nj = nnum[jr];
      const int* row = nbr + (size_t)jr * stride;
#pragma unroll 4
      for (int q = nj - 1; q >= 0; --q) l = row[q] == i ? q : l;  // the first match, without leaving early
    }
    rev[(size_t)r * stride + p] = l;
    if (l < 0) raise_err(err, PFM_E_GRAPHENE_NN, orig[i] + 1, -1, step);
  }
}

// lj1g: every row atom's group-local index, and that of the first listed
// neighbour whose atom index is larger than the row atom's (the reference's
// lessnnum boundary, in list order = ascending group order); T lanes per row,
// the minimum over the row's entries
template <int T>
__global__ void __launch_bounds__(256) k_lj1g_cut(int nrows, const int* __restrict__ rows,
                                                  const int* __restrict__ nnum, const int* __restrict__ nbr, int stride,
                                                  const int* __restrict__ orig, const int* __restrict__ loc,
                                                  int2* __restrict__ lc) {
  int gt = blockIdx.x * blockDim.x + threadIdx.x;
  int r = gt / T, t = threadIdx.x & (T - 1);
  if (r >= nrows) return;
  int i = rows[r], oi = orig[i], n = nnum[r], c = 0x7fffffff;
#pragma unroll 4
  for (int p = t; p < n; p += T) {
    const int oj = orig[nbr[(size_t)r * stride + p]];
    const int l = loc[oj];
    c = oj > oi && l < c ? l : c;
  }
#pragma unroll
  for (int o = T / 2; o > 0; o >>= 1) {
    int v = __shfl_xor(c, o, T);
    c = v < c ? v : c;
  }
  if (t == 0) lc[i] = make_int2(loc[oi], c);
}

// ljc/morsec metal rows (nl(2)) that have entries, appended in any order
// (each row's force is summed on its own, so the order of the work list does
// not change any result); the count goes after the rows.  One atomic per
// 1024-thread workgroup: wave ballots, then the wave counts' prefix in LDS.
// ONE: a single workgroup takes all the rows in turn and writes the count,
// which needs no clearing launch before it.
template <bool ONE>
__global__ void __launch_bounds__(1024) k_mark_rows(int nrows, const int* __restrict__ nnum, int* __restrict__ mrows) {
  __shared__ int wc[17];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int base = 0;
  for (int r0 = ONE ? 0 : blockIdx.x * 1024; r0 < nrows; r0 += ONE ? 1024 : nrows) {
    const int r = r0 + threadIdx.x;
    const bool keep = r < nrows && nnum[r] > 0;
    const unsigned long long bal = __ballot(keep);
    if (lane == 0) wc[w] = __popcll(bal);
    __syncthreads();
    if (threadIdx.x == 0) {
      int tot = 0;
      for (int q = 0; q < 16; ++q) { const int c = wc[q]; wc[q] = tot; tot += c; }
      wc[16] = ONE ? tot : (tot ? atomicAdd(&mrows[nrows], tot) : 0);
    }
    __syncthreads();
    const int at = ONE ? base : wc[16];
    if (keep) mrows[at + wc[w] + __popcll(bal & ((1ull << lane) - 1ull))] = r;
    if (ONE) base += wc[16];
    __syncthreads();
  }
  if (ONE && threadIdx.x == 0) mrows[nrows] = base;
}

// lj1g: each entry's weight in the gather, [loc(j) < cut(i)] (the pair is in
// i's half list) and [loc(i) < cut(j)] (in j's), packed into bits 30 and 31
// of the entry once per rebuild, so the force pass gathers positions only
__global__ void __launch_bounds__(256) k_lj1g_tag(int nrows, const int* __restrict__ rows,
                                                  const int* __restrict__ nnum, int* __restrict__ nbr, int stride,
                                                  const int2* __restrict__ lc) {
  int gt = blockIdx.x * blockDim.x + threadIdx.x;
  int r = gt / 8, t = threadIdx.x & 7;
  if (r >= nrows) return;
  const int2 mi = lc[rows[r]];
  const int n = nnum[r];
  for (int p = t; p < n; p += 8) {
    const int j = nbr[(size_t)r * stride + p];
    const int2 mj = lc[j];
    const unsigned tag = (mj.x < mi.y ? 1u : 0u) | (mi.x < mj.y ? 2u : 0u);
    nbr[(size_t)r * stride + p] = (int)((unsigned)j | (tag << 30));
  }
}

// graphene nearest neighbours from the tb list: entries with |dr| < r_cut_nn,
// exactly three per atom (find_gr_nearest_neighbors, graphenenorm.f90:8-36)
__global__ void k_nn_from_tb(int nrows, const int* __restrict__ rows, const int* __restrict__ tnnum,
                             const int* __restrict__ tnbr, int tstride, const double4* __restrict__ pos,
                             const int* __restrict__ rep, const RepDev* __restrict__ rdev, double rnn,
                             int* __restrict__ nnum, int* __restrict__ nbr, DevErr* err, const int* __restrict__ orig,
                             int step) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  int i = rows[r], n = tnnum[r], k = 0;
  const double3 hb = rdev[rep ? rep[i] : 0].hb;
  double4 pi = pos[i];
  for (int p = 0; p < n; ++p) {
    int j = tnbr[(size_t)r * tstride + p];
    double dx, dy, dz;
    double d = sqrt(min_image_dist2(pi, pos[j], hb, dx, dy, dz));
    if (d < rnn) {
      if (k < 3) nbr[(size_t)r * 3 + k] = j;
      ++k;
    }
  }
  nnum[r] = k < 3 ? k : 3;
  if (k != 3) raise_err(err, PFM_E_GRAPHENE_NN, orig[i] + 1, k, step);
}

// Cell-tile list search: one workgroup per cell.  The atoms of the 27
// surrounding cells are staged in LDS as FP32 coordinates unwrapped into the
// frame of the centre cell's origin, with the atom index in w.  Atoms outside
// group 2, and the padding after the last atom, are staged far away, so they
// never pass the distance test.  With CMP (group 2 under half of the atoms:
// another species' list) only the group-2 atoms are staged, compacted in tile
// order by ballots and a prefix over the workgroup's four waves, so the rows
// walk only real candidates.  Every group-1 atom of the centre cell is a row
// scanned by T lanes; all rows of a wavefront walk the tile in the same order,
// so their LDS reads are broadcasts.  Each lane takes 32 of its candidates
// (every T-th slot) into a register bitmask, two instructions per candidate
// after the distance; the row's lanes then take their output offsets from a
// prefix sum over the T lanes and write their hits.  The FP32 distance decides
// unless it lies within a relative 3e-5 of r_cut**2, where the reference's
// FP64 find_distance test (min_image_dist2) on the global positions decides.
// Tiles larger than the LDS buffer are staged in several passes.
// PAIR and QUAD: two or four lists in one pass, see SearchArgs.
//
// Directions under three cells wide hold each of their cells once in the tile
// (two or one instead of three) and cannot be unwrapped once per cell: there
// the coordinates are staged as they are and every pair takes its nearest
// image (TileImage), nine more instructions a candidate.  A row-by-row search
// of such grids, whose candidates wait on two dependent loads each, took 45 us
// for a 256-atom Cu replica's list.
// Handles with such a grid take the IMG kernel, which holds both scans and
// chooses by cell (launches of their own for the narrow cells waited on 28 us
// of dependent steps each: a 12-replica batch's step 37.2 -> 33.6 us without).
struct TileImage {
  float3 L, iL;  // box and its inverse in the directions under three cells wide, 0 in the others
  // a value equal on all lanes, in a scalar register
  static __device__ __forceinline__ float uni(bool on, double x) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(on ? (float)x : 0.f)));
  }
  __device__ __forceinline__ TileImage(const RepDev& R)
      : L(make_float3(uni(R.nc[0] < 3, R.L.x), uni(R.nc[1] < 3, R.L.y), uni(R.nc[2] < 3, R.L.z))),
        iL(make_float3(uni(R.nc[0] < 3, R.iL.x), uni(R.nc[1] < 3, R.iL.y), uni(R.nc[2] < 3, R.iL.z))) {}
  // the nearest image of a difference; the clamp keeps far-away padding far
  static __device__ __forceinline__ float near(float d, float L, float iL) {
    return fmaf(-L, rintf(__builtin_amdgcn_fmed3f(d * iL, -2.0f, 2.0f)), d);
  }
  template <bool IMG>
  __device__ __forceinline__ void diff(const float4& v, float px, float py, float pz, float& dx, float& dy,
                                       float& dz) const {
    dx = v.x - px; dy = v.y - py; dz = v.z - pz;
    if constexpr (IMG) {
      dx = near(dx, L.x, iL.x); dy = near(dy, L.y, iL.y); dz = near(dz, L.z, iL.z);
    }
  }
};

// tile cell k (0..26) of a grid cell cc: its coordinates, and whether it is
// one of the tile's own (a direction two cells wide holds offsets 0 and 1,
// one cell wide offset 0)
template <bool IMG>
__device__ __forceinline__ bool tile_cell(const RepDev& R, const int* cc, int k, int* q) {
  const int o[3] = {k % 3 - 1, (k / 3) % 3 - 1, k / 9 - 1};
  bool own = true;
  for (int d = 0; d < 3; ++d) {
    const int nd = R.nc[d];
    if (IMG) own = own && (nd >= 3 || o[d] == 0 || (nd == 2 && o[d] > 0));
    q[d] = cc[d] + o[d];
    q[d] = q[d] < 0 ? q[d] + nd : (q[d] >= nd ? q[d] - nd : q[d]);
  }
  return own;
}

// coordinate x of an atom of the tile cell at offset o, relative to the centre
// cell's origin: the image next to the centre cell (directions of three cells
// or more)
template <bool IMG>
__device__ __forceinline__ double unwrap(double x, int o, double L, int nd) {
  if (!IMG || nd >= 3) {
    if (o < 0 && x > 0.0) x -= L;
    else if (o > 0 && x < 0.0) x += L;
  }
  return x;
}

// the row of atom i (if it has one) when its tile holds no candidate: what
// the search writes for a row with no entries
__device__ __forceinline__ void empty_row(const SearchArgs& a, const int* __restrict__ row_of, int i) {
  const int row = row_of[i];
  if (row < 0) return;
  a.nnum[row] = 0;
  if (a.nnum2) a.nnum2[row] = 0;
  if ((a.mask[i] & a.g1bit) && a.exact && a.nmax != 0) raise_err(a.err, PFM_E_GRAPHENE_NN, a.orig[i] + 1, 0, a.step);
}

#define TILE_MAX 1536      // staged candidates per pass (24 KB of LDS), a multiple of 32 * T
#define TILE_FAR 1.0e30f   // staged coordinate of the padding

struct TileCells {
  int start[27], cnt[27], off[28];
};

#define ENTRY_IDX 0x3fffffff  // staged index without the pair search's group bits

// what staging keeps in w: the atom's index, with PAIR also its membership of
// list 1's candidate group in bit 30 and of list 2's in bit 31
template <bool PAIR>
__device__ __forceinline__ float staged_w(const SearchArgs& a, int j, uint32_t mj) {
  uint32_t w = (uint32_t)j;
  if constexpr (PAIR) w |= ((mj & a.g2bit1) ? 0x40000000u : 0u) | ((mj & a.g2bit2) ? 0x80000000u : 0u);
  return __uint_as_float(w);
}

// The rows of one list (PAIR: two) that a row atom's lanes fill: destinations
// and counts.  QUAD: atoms of side b take side b's lists.
template <int T, bool PAIR, bool QUAD>
struct RowOut {
  bool active;
  int i, row, count, count2;
  int *out, *out2, *nnum1, *nnum2;
  int nmax1, nmax2;
  __device__ __forceinline__ RowOut(const SearchArgs& a, const int* __restrict__ row_of, int atom, bool inrow) {
    i = atom;
    const uint32_t mi = a.mask[i];
    const bool sb = QUAD && (mi & a.g1mem_b) != 0;
    row = inrow ? (sb ? a.row_of_b[i] : row_of[i]) : -1;
    active = row >= 0 && (mi & (sb ? a.g1bit_b : a.g1bit));
    count = count2 = 0;
    const size_t r = active ? row : 0;
    nnum1 = sb ? a.nnum_b1 : a.nnum;
    nmax1 = sb ? a.nmax_b1 : a.nmax;
    out = (sb ? a.nbr_b1 : a.nbr) + r * (sb ? a.stride_b1 : a.stride);
    nnum2 = out2 = nullptr;
    nmax2 = 0;
    if constexpr (PAIR) {
      nnum2 = sb ? a.nnum_b2 : a.nnum2;
      nmax2 = sb ? a.nmax_b2 : a.nmax2;
      out2 = (sb ? a.nbr_b2 : a.nbr2) + r * (sb ? a.stride_b2 : a.stride2);
    }
  }
  // the row's hits of one round into one list: offsets from a prefix sum over
  // the row's lanes, entries without the group bits
  static __device__ __forceinline__ void put(unsigned hit, const float4* sv, int t, int* o, int nmax, int& cnt) {
    const int nh = __popc(hit);
    int pre = nh;
#pragma unroll
    for (int d = 1; d < T; d <<= 1) {
      int w = __shfl_up(pre, d, T);
      if (t >= d) pre += w;
    }
    const int tot = __shfl(pre, T - 1, T);
    int slot = cnt + pre - nh;
    while (hit) {
      const int b = __clz(hit);
      hit &= ~(0x80000000u >> b);
      if (slot < nmax) o[slot] = __float_as_int(sv[b * T].w) & ENTRY_IDX;
      ++slot;
    }
    cnt += tot;
  }
  // one pass over np staged candidates (whole rounds of 32 T); own: the row
  // atom's staged slot, or -1 to find it by index (find_self)
  template <bool IMG>
  __device__ __forceinline__ void scan(const SearchArgs& a, const RepDev& RG, const float4* st, int np, int t,
                                       int own, bool find_self, const double4& pi, float px, float py, float pz,
                                       float hi, float lo, const double3& hb) {
    const float win = hi - lo;
    const TileImage im(RG);
    for (int c0 = 0; c0 < np; c0 += 32 * T) {
      // bit 31-b <-> candidate slot c0 + t + b*T
      const float4* sv = st + c0 + t;
      // two masks with two instructions each per candidate after the
      // differences: the margin m = hi - d2 as a chain of fused
      // multiply-adds, whose sign bit (set for d2 > hi, and for the far
      // padding's -inf) shifts into the miss mask, and the sign of
      // (hi - lo) - m, set for d2 < lo (clearly inside r_cut); with PAIR the
      // candidates of list 1's and of list 2's group in two more
      unsigned miss = 0u, inside = 0u, m1 = 0u, m2 = 0u;
#pragma unroll PAIR ? 4 : 8
      for (int b = 0; b < 32; ++b) {
        const float4 v = sv[b * T];
        float dx, dy, dz;
        im.diff<IMG>(v, px, py, pz, dx, dy, dz);
        const float m = fmaf(-dx, dx, fmaf(-dy, dy, fmaf(-dz, dz, hi)));
        miss = __builtin_amdgcn_alignbit(miss, __float_as_uint(m), 31);
        inside = __builtin_amdgcn_alignbit(inside, __float_as_uint(win - m), 31);
        if constexpr (PAIR) {
          const uint32_t wb = __float_as_uint(v.w);
          m1 = __builtin_amdgcn_alignbit(m1, wb << 1, 31);
          m2 = __builtin_amdgcn_alignbit(m2, wb, 31);
        }
      }
      unsigned hit = ~miss;
      // the row atom is not its own neighbour
      const int ob = own - c0 - t;
      if (ob >= 0 && ob < 32 * T && ob % T == 0) hit &= ~(0x80000000u >> (ob / T));
      // hits inside the FP32 window: the FP64 test decides (with compacted
      // staging that is not dense every hit is also checked for the row atom)
      unsigned chk = find_self ? hit : hit & ~inside;
      while (chk) {
        const int b = __clz(chk);
        chk &= ~(0x80000000u >> b);
        const float4 v = sv[b * T];
        const int j = __float_as_int(v.w) & ENTRY_IDX;
        float dx, dy, dz;
        im.diff<IMG>(v, px, py, pz, dx, dy, dz);
        if (find_self && j == i) {
          hit &= ~(0x80000000u >> b);
        } else if (fmaf(dx, dx, fmaf(dy, dy, dz * dz)) >= lo) {
          double ex, ey, ez;
          if (!(min_image_dist2(pi, a.pos[j], hb, ex, ey, ez) < a.rc2)) hit &= ~(0x80000000u >> b);
        }
      }
      if constexpr (PAIR) {
        put(hit & m1, sv, t, out, nmax1, count);
        put(hit & m2, sv, t, out2, nmax2, count2);
      } else {
        put(hit, sv, t, out, nmax1, count);
      }
    }
  }
  // the row's lengths, and the reference's errors
  __device__ __forceinline__ void finish(const SearchArgs& a) const {
    if (row < 0) return;
    if (!active) {  // an inactive member of a growing group
      nnum1[row] = 0;
      if (PAIR) nnum2[row] = 0;
      return;
    }
    nnum1[row] = count < nmax1 ? count : nmax1;
    if (count > nmax1) raise_err(a.err, a.err_code, a.orig[i] + 1, count, a.step);
    else if (a.exact && count != nmax1) raise_err(a.err, PFM_E_GRAPHENE_NN, a.orig[i] + 1, count, a.step);
    if (PAIR) {
      nnum2[row] = count2 < nmax2 ? count2 : nmax2;
      if (count2 > nmax2) raise_err(a.err, a.err_code, a.orig[i] + 1, count2, a.step);
    }
  }
};

// every row of the cell's atoms empty: its tile holds no candidate
template <bool QUAD>
__device__ __forceinline__ void empty_rows(const SearchArgs& a, const int* __restrict__ row_of, int cs, int ncen,
                                           int first, int step) {
  for (int m = first; m < ncen; m += step) {
    const int i = a.bin ? a.bin[cs + m] : cs + m;
    if (QUAD && (a.mask[i] & a.g1mem_b)) {
      const int row = a.row_of_b[i];
      if (row >= 0) { a.nnum_b1[row] = 0; a.nnum_b2[row] = 0; }
    } else {
      empty_row(a, row_of, i);
    }
  }
}

template <int T, bool CMP, bool PAIR, bool QUAD, bool IMG>
__global__ void __launch_bounds__(256, CMP || PAIR ? 5 : 6) k_build_tile(SearchArgs a, const int* __restrict__ rank_xyz,
                                                    const int* __restrict__ row_of, int nblocks_real) {
  static_assert(TILE_MAX % (32 * T) == 0, "tile passes hold whole bitmask rounds");
  __shared__ float4 st[TILE_MAX];
  __shared__ TileCells tc;
  int c = xcd_block(nblocks_real);
  if (c < 0) return;
  if (IMG && a.cells) c = a.cells[c];
  const int ncen = a.cell_count[c];
  if (ncen == 0 || !(a.cell_grp[c] & a.g1mem)) return;  // no member of group 1 in the cell
  const RepDev& RG = a.rdev[a.cell_rep ? a.cell_rep[c] : 0];
  const int cs = a.cell_start[c];
  const int tid = threadIdx.x;
  // (cells without a row of this list, another species or another
  // replica's interactions, returned above: every group-1 member has a row)
  const int pk = rank_xyz[c];
  const int cc[3] = {pk & 1023, (pk >> 10) & 1023, (pk >> 20) & 1023};
  const double org[3] = {cc[0] * RG.clen.x, cc[1] * RG.clen.y, cc[2] * RG.clen.z};
  const double3 boxL = RG.L, hb = RG.hb;
  const int nc[3] = {RG.nc[0], RG.nc[1], RG.nc[2]};
  bool cand = false;
  if (tid < 27) {
    int q[3];
    const bool own = tile_cell<IMG>(RG, cc, tid, q);
    int r = a.cell_rank[RG.cell_base + (q[2] * nc[1] + q[1]) * nc[0] + q[0]];
    tc.start[tid] = a.cell_start[r];
    tc.cnt[tid] = own ? a.cell_count[r] : 0;
    cand = (a.cell_grp[r] & a.g2bit) != 0;
  }
  if (!__syncthreads_or(cand)) {
    // no group-2 atom in the tile: every row of the cell is empty
    empty_rows<QUAD>(a, row_of, cs, ncen, tid, 256);
    return;
  }
  if (tid == 0) {
    int off = 0;
    for (int k = 0; k < 27; ++k) { tc.off[k] = off; off += tc.cnt[k]; }
    tc.off[27] = off;
  }
  __syncthreads();
  const int R = tc.off[27];
  const float hi = (float)(a.rc2 * (1.0 + 3e-5)), lo = (float)(a.rc2 * (1.0 - 3e-5));

  // stage the group-2 atoms of tile slots [s0, s1) compacted into st (slot
  // m < R belongs to the last tile cell k with off[k] <= m; off is
  // non-decreasing, off[0] = 0), pad them to whole rounds and return that
  // length; every thread calls it.  A thread loads all its slots (every
  // 256th) before the ballots, so the pass waits on one memory latency.
  // dense: every slot was kept, so tile slots and staged slots coincide.
  constexpr int KS = TILE_MAX / 256;
  __shared__ int wsum[KS][4];
  bool dense = true;
  // slot m's record and whether its atom is in group 2
  auto load = [&](int m, float4& v) -> bool {
    int k = 0;
#pragma unroll
    for (int sft = 16; sft > 0; sft >>= 1)
      if (k + sft < 27 && tc.off[k + sft] <= m) k += sft;
    int j = tc.start[k] + (m - tc.off[k]);
    if (a.bin) j = a.bin[j];
    const double4 p = a.pos[j];
    const uint32_t mj = a.mask[j];
    v.x = (float)unwrap<IMG>(p.x - org[0], k % 3 - 1, boxL.x, nc[0]);
    v.y = (float)unwrap<IMG>(p.y - org[1], (k / 3) % 3 - 1, boxL.y, nc[1]);
    v.z = (float)unwrap<IMG>(p.z - org[2], k / 9 - 1, boxL.z, nc[2]);
    v.w = staged_w<PAIR>(a, j, mj);
    return (mj & a.g2bit) != 0;
  };
  const float4 far = make_float4(TILE_FAR, TILE_FAR, TILE_FAR, __int_as_float(-1));
  auto stage = [&](int s0, int s1) -> int {
    if constexpr (!CMP) {
      const int np = (s1 - s0 + 32 * T - 1) / (32 * T) * (32 * T);
      for (int m = s0 + tid; m < s0 + np; m += 256) {
        float4 v = far;
        if (m < s1 && !load(m, v)) v.x = v.y = v.z = TILE_FAR;
        st[m - s0] = v;
      }
      return np;
    }
    const int lane = tid & 63, w = tid >> 6;
    float4 v[KS];
    bool keep[KS];
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const int m = s0 + u * 256 + tid;
      v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      keep[u] = m < s1 && load(m, v[u]);
    }
    unsigned long long bal[KS];
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      bal[u] = __ballot(keep[u]);
      if (lane == 0) wsum[u][w] = __popcll(bal[u]);
    }
    __syncthreads();
    int base = 0;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      int off = base;
      for (int q = 0; q < w; ++q) off += wsum[u][q];
      if (keep[u]) st[off + __popcll(bal[u] & ((1ull << lane) - 1ull))] = v[u];
      base += wsum[u][0] + wsum[u][1] + wsum[u][2] + wsum[u][3];
    }
    dense = base == s1 - s0;
    const int np = (base + 32 * T - 1) / (32 * T) * (32 * T);
    for (int m = base + tid; m < np; m += 256) st[m] = far;
    return np;
  };
  const bool single = R <= TILE_MAX;
  int np = 0;
  if (single) np = stage(0, R);

  const int t = tid & (T - 1);
  for (int q0 = 0; q0 < ncen; q0 += 256 / T) {
    const int qq = q0 + tid / T;
    const bool inrow = qq < ncen;
    const int i = a.bin ? a.bin[cs + (inrow ? qq : 0)] : cs + (inrow ? qq : 0);
    RowOut<T, PAIR, QUAD> ro(a, row_of, i, inrow);
    const double4 pi = a.pos[i];
    const float px = (float)(pi.x - org[0]), py = (float)(pi.y - org[1]), pz = (float)(pi.z - org[2]);
    for (int s0 = 0; s0 < R; s0 += TILE_MAX) {
      if (!single) {
        __syncthreads();
        np = stage(s0, R < s0 + TILE_MAX ? R : s0 + TILE_MAX);
      }
      __syncthreads();
      if (!ro.active) continue;
      // the row atom's own staged slot when the pass is dense (else found by index)
      const bool find = CMP && !dense;
      const int own = find ? -1 : tc.off[13] + qq - s0;
      if (IMG && narrow_grid(RG)) ro.template scan<true>(a, RG, st, np, t, own, find, pi, px, py, pz, hi, lo, hb);
      else ro.template scan<false>(a, RG, st, np, t, own, find, pi, px, py, pz, hi, lo, hb);
    }
    if (t == 0) ro.finish(a);
  }
}

// Wave-per-cell variant of k_build_tile for sparse grids (a workgroup per
// cell would leave most of its lanes without rows): each of a workgroup's
// four waves searches one cell with its own staged tile of WTILE candidates
// per pass.  The tile order, the tests and the output are those of
// k_build_tile; the tile's cell table lives in lanes 0..26 and is read with
// shuffles, which every lane of the wave takes part in.
#define WTILE 512

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int T, bool CMP, bool PAIR, bool QUAD, bool SKIP>
__global__ void __launch_bounds__(256, 5) k_build_tile_wave(SearchArgs a, const int* __restrict__ rank_xyz,
                                                         const int* __restrict__ row_of, int ncell,
                                                         int nblocks_real) {
  static_assert(WTILE % (32 * T) == 0 && WTILE % 64 == 0, "tile passes hold whole bitmask rounds");
  constexpr int KW = WTILE / 64;
  __shared__ float4 stw[4][WTILE];
  const int lb = xcd_block(nblocks_real);
  if (lb < 0) return;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int c = lb * 4 + wv;
  if (c >= ncell) return;
  const int ncen = a.cell_count[c];
  if (ncen == 0 || !(a.cell_grp[c] & a.g1mem)) return;  // no member of group 1 in the cell
  const RepDev& RG = a.rdev[a.cell_rep ? a.cell_rep[c] : 0];
  if (SKIP && narrow_grid(RG)) return;  // searched by k_build_tile<..., IMG>
  const int cs = a.cell_start[c];
  float4* st = stw[wv];
  const int pk = rank_xyz[c];
  const int cc[3] = {pk & 1023, (pk >> 10) & 1023, (pk >> 20) & 1023};
  const double org[3] = {cc[0] * RG.clen.x, cc[1] * RG.clen.y, cc[2] * RG.clen.z};
  const double3 boxL = RG.L, hb = RG.hb;
  const int nc[3] = {RG.nc[0], RG.nc[1], RG.nc[2]};
  // the 27 tile cells in lanes 0..26: first atom, count, exclusive offset
  int kst = 0, kcn = 0;
  bool cand = false;
  if (lane < 27) {
    int q[3];
    const bool own = tile_cell<false>(RG, cc, lane, q);
    const int r = a.cell_rank[RG.cell_base + (q[2] * nc[1] + q[1]) * nc[0] + q[0]];
    kst = a.cell_start[r];
    kcn = own ? a.cell_count[r] : 0;
    cand = (a.cell_grp[r] & a.g2bit) != 0;
  }
  if (!__any(cand)) {
    empty_rows<QUAD>(a, row_of, cs, ncen, lane, 64);
    return;
  }
  int inc = kcn;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(inc, o);
    if (lane >= o) inc += v;
  }
  const int koff = inc - kcn;
  const int R = __shfl(inc, 63);
  const int koff13 = __shfl(koff, 13);
  const float hi = (float)(a.rc2 * (1.0 + 3e-5)), lo = (float)(a.rc2 * (1.0 - 3e-5));
  // tile slot m < R: the last cell k with off[k] <= m (every lane takes part)
  auto cell_of = [&](int m) -> int {
    int k = 0;
#pragma unroll
    for (int sft = 16; sft > 0; sft >>= 1) {
      const int kk = k + sft;
      const int o = __shfl(koff, kk < 27 ? kk : 0);
      if (kk < 27 && o <= m) k = kk;
    }
    return k;
  };
  // stage tile slots [s0, s1) (s1 - s0 <= WTILE): every slot, atoms outside
  // group 2 far away; with CMP only group-2 atoms, compacted in tile order.
  // Returns the staged length padded to whole rounds.
  bool dense = true;
  // slots in chunks of KC per lane (KC * 64 per wave): a tile of up to that
  // many candidates waits on one memory latency, and the registers hold one
  // chunk
  constexpr int KC = KW < 4 ? KW : 4;
  auto stage = [&](int s0, int s1) -> int {
    int base = 0;
    for (int cb = 0; cb < KW && s0 + cb * 64 < s1; cb += KC) {
      float4 v[KC];
      bool keep[KC];
#pragma unroll
      for (int u = 0; u < KC; ++u) {
        const int m = s0 + (cb + u) * 64 + lane;
        const int k = cell_of(m < s1 ? m : s0);
        const int ks = __shfl(kst, k), ko = __shfl(koff, k);
        v[u] = make_float4(TILE_FAR, TILE_FAR, TILE_FAR, __int_as_float(-1));
        keep[u] = false;
        if (m < s1) {
          int j = ks + (m - ko);
          if (a.bin) j = a.bin[j];
          const double4 p = a.pos[j];
          const uint32_t mj = a.mask[j];
          keep[u] = (mj & a.g2bit) != 0;
          const double x = unwrap<false>(p.x - org[0], k % 3 - 1, boxL.x, nc[0]);
          const double y = unwrap<false>(p.y - org[1], (k / 3) % 3 - 1, boxL.y, nc[1]);
          const double z = unwrap<false>(p.z - org[2], k / 9 - 1, boxL.z, nc[2]);
          v[u].w = staged_w<PAIR>(a, j, mj);
          if (keep[u]) { v[u].x = (float)x; v[u].y = (float)y; v[u].z = (float)z; }
        }
      }
      if constexpr (!CMP) {
#pragma unroll
        for (int u = 0; u < KC; ++u) {
          const int m = s0 + (cb + u) * 64 + lane;
          if (m < s1) st[m - s0] = v[u];
        }
      } else {
#pragma unroll
        for (int u = 0; u < KC; ++u) {
          const unsigned long long bal = __ballot(keep[u]);
          if (keep[u]) st[base + __popcll(bal & ((1ull << lane) - 1ull))] = v[u];
          base += __popcll(bal);
        }
      }
    }
    if constexpr (!CMP) base = s1 - s0;
    else dense = base == s1 - s0;
    const int np = (base + 32 * T - 1) / (32 * T) * (32 * T);
    for (int m = base + lane; m < np; m += 64) st[m] = make_float4(TILE_FAR, TILE_FAR, TILE_FAR, __int_as_float(-1));
    return np;
  };
  const bool single = R <= WTILE;
  int np = 0;
  if (single) np = stage(0, R);
  wave_sync();

  const int t = lane & (T - 1);
  for (int q0 = 0; q0 < ncen; q0 += 64 / T) {
    const int qq = q0 + lane / T;
    const bool inrow = qq < ncen;
    const int i = a.bin ? a.bin[cs + (inrow ? qq : 0)] : cs + (inrow ? qq : 0);
    RowOut<T, PAIR, QUAD> ro(a, row_of, i, inrow);
    const double4 pi = a.pos[i];
    const float px = (float)(pi.x - org[0]), py = (float)(pi.y - org[1]), pz = (float)(pi.z - org[2]);
    for (int s0 = 0; s0 < R; s0 += WTILE) {
      if (!single) {
        wave_sync();
        np = stage(s0, R < s0 + WTILE ? R : s0 + WTILE);
        wave_sync();
      }
      if (!ro.active) continue;
      // the row atom's own staged slot when the pass is dense (else found by index)
      const bool find = CMP && !dense;
      const int own = find ? -1 : koff13 + qq - s0;
      ro.template scan<false>(a, RG, st, np, t, own, find, pi, px, py, pz, hi, lo, hb);
    }
    if (t == 0) ro.finish(a);
  }
}

// One list (or with PAIR / QUAD the lists of a pair or two) by the kernel the
// list takes: one wave per cell (ListDev::wave_cells) or one workgroup.  With
// grids under three cells wide among others (a batch), the workgroup kernel
// searches all cells by its IMG form, and one wave per cell leaves it their
// cells in a launch of their own: four lists of 27,000 cells of 3.7 atoms
// beside one box of 256 atoms 81 us a rebuild (118 all one workgroup per cell,
// 89 all one wave per cell), beside one of 600 dense atoms 103 (141 and 250).
template <bool PAIR, bool QUAD>
static void launch_build(pfm_ctx* h, SearchArgs& a, const int* row_of, bool sparse, bool wave_cells) {
  const int nc = h->ncell, nbw = (nc + 3) / 4;
  const bool few = !PAIR && a.nmax <= 8;  // four lanes a row
#define BUILD_TILE(T, CMP, IMG, N)                                                                                  \
  PFM_LAUNCH(h, "build_list", (k_build_tile<T, CMP, PAIR, QUAD, IMG>), pad8(N), 256, a, h->cell_xyz, row_of, N)
#define BUILD_WAVE(T, CMP, SKIP)                                                                                    \
  PFM_LAUNCH(h, "build_list", (k_build_tile_wave<T, CMP, PAIR, QUAD, SKIP>), pad8(nbw), 256, a, h->cell_xyz,       \
             row_of, nc, nbw)
#define BUILD_AS(T, CMP)                              \
  do {                                                \
    if (wave_cells && h->n_narrow) {                  \
      BUILD_WAVE(T, CMP, true);                       \
      a.cells = h->narrow_cells;                      \
      BUILD_TILE(T, CMP, true, h->n_narrow);          \
    } else if (wave_cells) BUILD_WAVE(T, CMP, false); \
    else if (h->n_narrow) BUILD_TILE(T, CMP, true, nc); \
    else BUILD_TILE(T, CMP, false, nc);               \
  } while (0)
  if constexpr (!PAIR) {
    if (few) {
      if (sparse) BUILD_AS(4, true);
      else BUILD_AS(4, false);
      return;
    }
  }
  if (sparse) BUILD_AS(8, true);
  else BUILD_AS(8, false);
#undef BUILD_AS
#undef BUILD_WAVE
#undef BUILD_TILE
}

// Build list k (0-based) of interaction ii.  For lj/ljc/morsec, list 1 is the
// converse of list 0: same r_cut and schedule (md_interactions.f90:152-155),
// found by searching from the group-2 side, which gives the same set because
// find_distance's dr2 is symmetric in its two atoms.
// the search arguments of list k of interaction ii
static SearchArgs search_args(pfm_ctx* h, int ii, int k, int step) {
  Inter& it = h->inter[ii];
  ListDev& L = it.nl[k];
  SearchArgs a{};
  a.nrows = L.nrows;
  a.rows = h->grp.rows[L.g1];
  a.g1bit = 1u << (L.g1 - 1);
  a.g1mem = 1u << ((h->grp.shadow[L.g1] ? h->grp.shadow[L.g1] : L.g1) - 1);
  a.g2bit = 1u << (L.g2 - 1);
  a.pos = h->pos4;
  a.mask = h->mask;
  a.orig = h->orig;
  a.rdev = h->rdev;
  a.rep = h->rep;
  a.cell_rep = h->cell_rep;
  a.bin = h->bin;
  double rc = (k == 1 && has_converse(it.kind)) ? it.nl[0].rcut : L.rcut;
  a.rc2 = rc * rc;
  a.rc2_lo = a.rc2 * (1.0 - 1e-12);
  a.rc2_hi = a.rc2 * (1.0 + 1e-12);
  a.cell_rank = h->cell_rank;
  a.cell_start = h->cell_start;
  a.cell_count = h->cell_count;
  a.cell_grp = h->cell_grp;
  a.nmax = L.nmax;
  a.stride = L.stride;
  a.nnum = L.nnum;
  a.nbr = L.nbr;
  a.err = h->derr;
  a.step = step - h->step_base;
  a.err_code = PFM_E_OVERFLOW;
  a.exact = (k == 2) ? 1 : 0;
  return a;
}

static int rev_blocks(int nrows) { return (int)(((long)nrows * REV_T + 255) / 256); }

// one workgroup marks this many rows faster than a clearing launch and the
// blocks of 1,024 (4,648 rows: 4.5 us against 4.5 + 3.6)
#define MARK_ONE 8192

// what follows a list's search: tb reverse slots, the ljc/morsec metal work
// list, lj1g half-list tags
static void list_post(pfm_ctx* h, int ii, int k, int step) {
  Inter& it = h->inter[ii];
  ListDev& L = it.nl[k];
  if (L.nrows == 0) {
    L.built = true;
    return;
  }
  if (it.kind == PFM_TB || it.kind == PFM_REBOSC || (k == 2 && !(int)it.p[it.kind == PFM_LJC ? 5 : 6])) {
    PFM_LAUNCH(h, "list_rev", k_rev, rev_blocks(L.nrows), 256, L.nrows, h->grp.rows[L.g1], h->grp.row_of[L.g1], L.nnum, L.nbr,
               L.stride, L.rev, h->derr, h->orig, step - h->step_base);
  }
  if ((it.kind == PFM_LJC || it.kind == PFM_MORSEC) && k == 1) {
    if (L.nrows <= MARK_ONE) {
      PFM_LAUNCH(h, "list_rows", k_mark_rows<true>, 1, 1024, L.nrows, L.nnum, it.mrows);
    } else {
      PFM_LAUNCH(h, "list_rows", k_fill_int, 1, 64, 1, it.mrows + L.nrows, 0);
      PFM_LAUNCH(h, "list_rows", k_mark_rows<false>, (L.nrows + 1023) / 1024, 1024, L.nrows, L.nnum, it.mrows);
    }
  }
  if (it.kind == PFM_LJ1G) {
    PFM_LAUNCH(h, "list_cut", k_lj1g_cut<8>, (int)(((long)L.nrows * 8 + 255) / 256), 256, L.nrows, h->grp.rows[L.g1],
               L.nnum, L.nbr, L.stride, h->orig, h->grp.loc[L.g2], it.lc);
    PFM_LAUNCH(h, "list_cut", k_lj1g_tag, (int)(((long)L.nrows * 8 + 255) / 256), 256, L.nrows, h->grp.rows[L.g1],
               L.nnum, L.nbr, L.stride, it.lc);
  }
  L.built = true;
}

int launch_build_list(pfm_ctx* h, int ii, int k, int step) {
  ListDev& L = h->inter[ii].nl[k];
  if (L.nrows == 0) { L.built = true; return PFM_OK; }
  SearchArgs a = search_args(h, ii, k, step);
  // candidates of another species: stage only those
  launch_build<false, false>(h, a, h->grp.row_of[L.g1], 2L * h->grp.size[L.g2] < (long)h->N, L.wave_cells);
  list_post(h, ii, k, step);
  return PFM_OK;
}

// Two lists of one pair (ListDev::pair): one pass stages the union of their
// candidate groups once and writes both.
int launch_build_pair(pfm_ctx* h, int ii, int k, int jj, int kk, int step) {
  ListDev& L1 = h->inter[ii].nl[k];
  SearchArgs a = search_args(h, ii, k, step);
  SearchArgs b = search_args(h, jj, kk, step);
  if (L1.nrows > 0) {
    SearchArgs p = a;
    p.g2bit1 = a.g2bit;
    p.g2bit2 = b.g2bit;
    p.g2bit = a.g2bit | b.g2bit;
    p.nmax2 = b.nmax;
    p.stride2 = b.stride;
    p.nnum2 = b.nnum;
    p.nbr2 = b.nbr;
    launch_build<true, false>(h, p, h->grp.row_of[L1.g1], L1.pair_sparse, L1.wave_cells);
  }
  list_post(h, ii, k, step);
  list_post(h, jj, kk, step);
  return PFM_OK;
}

// Two pairs in one pass (ListDev::quad_*): the lead pair (ii, k) + (jj, kk)
// and a second pair with rows of another group whose lists take the same two
// candidate groups, (b1 for the lead's group, b2 for its partner's).
int launch_build_quad(pfm_ctx* h, int ii, int k, int jj, int kk, int b1i, int b1k, int b2i, int b2k, int step) {
  ListDev& L1 = h->inter[ii].nl[k];
  ListDev& B1 = h->inter[b1i].nl[b1k];
  SearchArgs a = search_args(h, ii, k, step);
  SearchArgs b = search_args(h, jj, kk, step);
  SearchArgs c = search_args(h, b1i, b1k, step);
  SearchArgs d = search_args(h, b2i, b2k, step);
  if (L1.nrows > 0 || B1.nrows > 0) {
    SearchArgs p = a;
    p.g2bit1 = a.g2bit;
    p.g2bit2 = b.g2bit;
    p.g2bit = a.g2bit | b.g2bit;
    p.nmax2 = b.nmax; p.stride2 = b.stride; p.nnum2 = b.nnum; p.nbr2 = b.nbr;
    p.g1bit_b = c.g1bit;
    p.g1mem_b = c.g1mem;
    p.g1mem = a.g1mem | c.g1mem;
    p.row_of_b = h->grp.row_of[B1.g1];
    p.nmax_b1 = c.nmax; p.stride_b1 = c.stride; p.nnum_b1 = c.nnum; p.nbr_b1 = c.nbr;
    p.nmax_b2 = d.nmax; p.stride_b2 = d.stride; p.nnum_b2 = d.nnum; p.nbr_b2 = d.nbr;
    launch_build<true, true>(h, p, h->grp.row_of[L1.g1], L1.pair_sparse, L1.wave_cells);
  }
  list_post(h, ii, k, step);
  list_post(h, jj, kk, step);
  list_post(h, b1i, b1k, step);
  list_post(h, b2i, b2k, step);
  return PFM_OK;
}

// nl(3) of ljc/morsec copied from the tb interaction's freshly rebuilt list
int launch_nn_from_tb(pfm_ctx* h, int ii, int step) {
  Inter& it = h->inter[ii];
  Inter& tb = h->inter[it.nn_from_tb];
  ListDev& L = it.nl[2];
  ListDev& T = tb.nl[0];
  if (L.nrows == 0) return PFM_OK;
  const int nb = (L.nrows + 255) / 256;
  PFM_LAUNCH(h, "nn_from_tb", k_nn_from_tb, nb, 256, L.nrows, h->grp.rows[L.g1], T.nnum, T.nbr, T.stride, h->pos4,
             h->rep, h->rdev, L.rcut, L.nnum, L.nbr, h->derr, h->orig, step - h->step_base);
  bool simplified = (int)it.p[it.kind == PFM_LJC ? 5 : 6];
  if (!simplified)
    PFM_LAUNCH(h, "list_rev", k_rev, rev_blocks(L.nrows), 256, L.nrows, h->grp.rows[L.g1], h->grp.row_of[L.g1], L.nnum, L.nbr,
               L.stride, L.rev, h->derr, h->orig, step - h->step_base);
  L.built = true;
  return PFM_OK;
}
