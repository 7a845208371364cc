/*
 * pfm.h -- C-ABI of libpfmds.so, the MI355X (gfx950) HIP implementation of the
 * PFMDS molecular-dynamics step.
 *
 * The reference runs its step loop inside the Fortran subroutine md()
 * (code_source/MOLECULAR_DYNAMICS/md_simulation.f90:19-275) and calls module
 * procedures whose arguments are derived types with allocatable components,
 * which are not C-interoperable.  This header replaces those procedures with a
 * handle-based interface: the caller (the Fortran front end in
 * pfmds_amd/fortran, or any C/Python host) keeps the settings file, the
 * schedule, logging and xyz output, and hands the per-step work to the GPU.
 *
 * Conventions
 *   - Every function returns an int status: PFM_OK (0) or one of PFM_E_*.
 *     pfm_last_error() returns the message, worded as the reference's
 *     "error: ..." text, so a caller can print it and stop as md() does.
 *   - Arrays of atom data are the reference's (3,N) column-major Fortran
 *     arrays, i.e. C double[N][3]; atom and group indices are 1-based.
 *   - One handle = one system and one HIP stream; a handle is not
 *     thread-safe.  Device memory is owned by the handle until pfm_destroy().
 */
#ifndef PFM_H
#define PFM_H
#ifdef __cplusplus
extern "C" {
#endif

/* status codes */
#define PFM_OK             0
#define PFM_E_OVERFLOW     1  /* "error: too many neighbours" (md_neighbours.f90:80,151) */
#define PFM_E_OUT_OF_CELL  2  /* "particle out of cell" (md_general.f90:342-364)         */
#define PFM_E_GRAPHENE_NN  3  /* "not enough / too many gr nearest neibs", "l1>3"
                                 (graphenenorm.f90:13,26,30; MorseCosine.f90:60,88)       */
#define PFM_E_NHC_PARAMS   4  /* "error: wrong nhc parameters" (md_integrators.f90:187)   */
#define PFM_E_UNKNOWN_KIND 5  /* "error: unknown interaction name" (md_interactions.f90:120) */
#define PFM_E_INVALID      6  /* argument or group layout the reference cannot run       */
#define PFM_E_HIP          7  /* HIP runtime error                                        */
#define PFM_E_NO_DEVICE    8  /* no gfx950 device visible                                 */

/* interaction kinds: the names of md_interactions.f90:70-121 */
#define PFM_LJ     1  /* 'lj'     params: eps sig R1 R2                     (LennardJones.f90:17-18)       */
#define PFM_LJ1G   2  /* 'lj1g'   params: eps sig R1 R2                     (LennardJones_1g.f90:18-19)    */
#define PFM_LJC    3  /* 'ljc'    params: eps sig delt R1 R2 simplified     (LennardJonesCosine.f90:19-21) */
#define PFM_MORSEC 4  /* 'morsec' params: d r a delt R1 R2 simplified       (MorseCosine.f90:19-21)        */
#define PFM_RJL    5  /* 'rjl'    params: A0 xi p q r0 R1 R2                (RosatoGuillopeLegrand.f90:17-18) */
#define PFM_TB     6  /* 'tb'     params: d s b r0 delt a0 c0 d0 R1 R2      (TersoffBrenner.f90:18-19)     */
#define PFM_SUR    7  /* 'sur'    params: r_c.  Learned stand-in for the graphene terms (tb + morsec):
                         no counterpart in the reference.  Lists: nl(1) g1 -> g2 (g1 = atoms that
                         carry an energy, the carbon; g2 = every atom their descriptors see,
                         g1 included), nl(2) g2 -> g1, the converse (list r_cut >= r_c).  The
                         network comes from pfm_sur_set_params.                                     */

#define PFM_REBOSC 8 /* 'rebosc' params: A Q alpha B1 B2 B3 beta1 beta2 beta3 T g1..g6 R1 R2
                         (REBOsolidcarbon.f90:17-22); forces by central differences of the energy
                         (md_interactions.f90:273-310), always in FP64                                */

/* number of surrogate parameters: mu[40] isg[40] W1[64][40] b1[64] W2[64][64] b2[64] w3[64] b3 */
#define PFM_SUR_NTHETA 6929

/* integrators: the names of md_simulation.f90:73-80 */
#define PFM_NVT  1
#define PFM_NVE  2
#define PFM_NVMS 3

/* precision of the force arithmetic */
#define PFM_FP64  0   /* all arithmetic in FP64                                        */
#define PFM_MIXED 1   /* FP32 pair arithmetic, FP64 dr, accumulation, state, reductions */

/* pfm_run events */
#define PFM_EV_DONE      0  /* ran through step_end                                            */
#define PFM_EV_CONVERGED 1  /* nvms: abs(PE-PE_prev) <= ms_de at *last_step (md_simulation.f90:142-147) */

typedef struct pfm_ctx pfm_ctx;

/* Create a system: replaces read_box_size/read_particles state setup
 * (md_read_write.f90:22-61) and the `particles` type (md_general.f90:13-17).
 * pos/vel: double[n][3]; mass: double[n] in u. */
int pfm_create(pfm_ctx** h, int n_atoms, const double box[3], const double* pos,
               const double* vel, const double* mass, int precision);

/* Create a batch of n_rep independent systems (replicas) that share every
 * pass of the step: replica r has n_atoms[r] atoms in its own periodic box
 * boxes[3r..3r+2]; pos/vel/mass hold the replicas one after another, so atom
 * numbering (groups, lists, downloads) runs over the concatenation.  Lists
 * never link atoms of different replicas, and zero_momentum, per-replica
 * energies (pfm_replica_energies) and the nvms stop test (every replica
 * within ms_de) treat each replica as if it ran alone.  Nose-Hoover chains
 * are refused in batches (a chain's group would span replicas).  No
 * counterpart in the reference, which runs one system per md() call and farms
 * systems over MPI ranks (run_md_simulation_mpi.f90:68-88); pfm_create is the
 * batch of one.
 * A replica's results are those of its own run within rounding, not bit for
 * bit: the order of its sums follows the handle's lanes per row, which start
 * by the atoms of the whole handle (pfm_set_tuning), and the order of its list
 * entries the search that the whole handle's cells lead to. */
int pfm_create_batch(pfm_ctx** h, int n_rep, const int* n_atoms, const double* boxes,
                     const double* pos, const double* vel, const double* mass, int precision);

/* Energies of every replica at the last energy evaluation: e_inter[n_rep][n_interactions],
 * pe[n_rep], ke[n_rep] (all_moving atoms of the replica) and temp[n_rep]; any
 * pointer may be NULL.  For a single system the values of pfm_energies. */
int pfm_replica_energies(pfm_ctx* h, double* e_inter, double* pe, double* ke, double* temp);

/* Define group gid (1-based) as the atom indices idx[0..n-1] (1-based) in the
 * order create_particle_group builds them (md_general.f90:57-80). */
int pfm_set_group(pfm_ctx* h, int gid, int n, const int* idx);

/* Group roles and periods of md() (md_simulation.f90:55-62,72). */
int pfm_set_roles(pfm_ctx* h, int all_moving, int xyz_moving, int z_moving,
                  int all_atoms, int zero_momentum_period, int invert_z);

/* Add one interaction, in settings order; replaces one iteration of
 * create_interactions (md_interactions.f90:68-133).  group_nums has 2*nl_n
 * entries (g1 g2 per list row); nmax/r_cut/period have nl_n entries. */
int pfm_add_interaction(pfm_ctx* h, int kind, const double* params, int n_params,
                        int nl_n, const int* group_nums, const int* nmax,
                        const double* r_cut, const int* period);

/* Add one Nose-Hoover chain; replaces create_nose_hoover_chain +
 * set_nose_hoover_chain (md_integrators.f90:165-198). */
int pfm_add_nhc(pfm_ctx* h, int group, double temperature, int M, double q1);

/* Run md steps step_begin..step_end of one integrator with time step dt;
 * replaces the body of md()'s loop (md_simulation.f90:137-231) for those
 * steps.  Energies are evaluated at step_end when energy_at_end != 0 and at
 * every step under nvms.  *last_step is the last step entered; *event is a
 * PFM_EV_* code. */
int pfm_run(pfm_ctx* h, int integrator, double dt, int step_begin, int step_end,
            int energy_at_end, double ms_de, int* last_step, int* event);

/* Energies of the last energy evaluation: e_inter[n_interactions] (eV),
 * potential, kinetic (eV), temperature (K) of the all_moving group,
 * e_nhc[n_chains], simulated time (fs).  Replaces the values md() logs at
 * md_simulation.f90:188-209. Any pointer may be NULL. */
int pfm_energies(pfm_ctx* h, double* e_inter, double* pe, double* ke, double* temp,
                 double* e_nhc, double* sim_time);

/* Potential-energy change of the last step entered, PE - PE_prev, the value
 * md() prints after an nvms run (md_simulation.f90:246). */
int pfm_pe_change(pfm_ctx* h, double* de);

/* Copy positions/velocities/forces (double[n][3], original atom order) to the
 * host; any pointer may be NULL.  Used for snapshots, trajectories and final
 * xyz (md_read_write.f90:65-107). */
int pfm_get_state(pfm_ctx* h, double* pos, double* vel, double* force);

/* Replace positions and velocities (double[n][3]).  The next pfm_run re-sorts
 * the atoms, rebuilds every list and, unless it starts at step 0 (which
 * computes forces anyway), evaluates the forces at the new positions before
 * its first half kick. */
int pfm_set_state(pfm_ctx* h, const double* pos, const double* vel);

/* Device-side transfers between two handles of the same atoms on one GPU.
 * pfm_copy_state: dst takes src's positions and velocities, as
 * pfm_set_state would take them from the host.  pfm_force_rmse: the RMSE
 * (eV/A) over the 3n force components of group `group` (of handle b) between
 * a's and b's forces.  They serve a run that checks one potential against
 * another at the same positions (the surrogate's judge).  No counterpart in
 * the reference. */
int pfm_copy_state(pfm_ctx* dst, pfm_ctx* src);
int pfm_force_rmse(pfm_ctx* a, pfm_ctx* b, int group, double* rmse);

/* pfm_force_rmse without allocation.  No counterpart in the reference: it is
 * for callers that cannot allocate device memory (code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc).  Same
 * arguments and result as pfm_force_rmse (bit-identical), but its staging
 * and partial sums live in a fixed device array of the library (32 MiB per
 * device, held until the process ends) instead of memory the library
 * allocates, and it calls no hipMalloc/hipFree.  At most 1,048,576 atoms
 * (PFM_E_INVALID beyond).  All handles on one device share that array:
 * calls that overlap on one device (threads) race. */
int pfm_force_rmse_noalloc(pfm_ctx* a, pfm_ctx* b, int group, double* rmse);

/* Positions x[M] and velocities v[M] of Nose-Hoover chain c (1-based, in
 * pfm_add_nhc order): the `nose_hoover_chain` state (md_general.f90:24-28)
 * that md() carries from step to step.  pfm_set_chain takes them over (after
 * the first pfm_run), e.g. to continue a run in another handle; the chain's
 * masses stay those of pfm_add_nhc. */
int pfm_get_chain(pfm_ctx* h, int c, double* x, double* v);
int pfm_set_chain(pfm_ctx* h, int c, const double* x, const double* v);

/* Download neighbour list k (1-based) of interaction inter (1-based) in the
 * reference layout of type neighbour_list (md_general.f90:30-35): n_rows,
 * nnum[row], nlist[row*stride+p] = 1-based group2-local index, lessnnum[row].
 * Entries of a row are in ascending group2 order, as find_neighbours
 * (md_neighbours.f90:56-100) produces them. */
int pfm_get_list(pfm_ctx* h, int inter, int k, int* n_rows, int* nnum, int* nlist,
                 int* lessnnum, int stride);

/* Per-row energies of interaction inter (1-based) at the last energy
 * evaluation, one per row of its first list in the handle's row order;
 * *n_rows their number (e_row may be NULL to ask for it).  Their sum is the
 * interaction's energy (a compensated sum, as every energy and kinetic
 * energy reduction of the library).  The reference keeps no per-row
 * energies (its *_energy routines sum directly, e.g.
 * RosatoGuillopeLegrand.f90:23-49); for inspection and tests. */
int pfm_row_energies(pfm_ctx* h, int inter, int* n_rows, double* e_row);

/* Graphene normals gr_norm(3,N_g1) of a ljc/morsec interaction
 * (graphenenorm.f90:38-56), double[N_g1][3] in group order. */
int pfm_get_normals(pfm_ctx* h, int inter, double* gr_norm);

/* Kernel timing.  pfm_set_timing(h,1) brackets every launch with HIP events on
 * the handle's stream; pfm_kernel_time() returns the launch count and the
 * mean duration (ms) of the kernels whose name contains `name`. */
int pfm_set_timing(pfm_ctx* h, int on);
int pfm_kernel_time(pfm_ctx* h, const char* name, int* count, double* mean_ms);

/* Shape of the pair passes: lanes per atom row (1,2,4,8,16,32) and
 * workgroup size (64..1024); 0 keeps the current value.  A handle starts
 * with 8 lanes (16 up to 15,000 atoms in FP64 and 8,192 in the mixed path)
 * and 256.  No counterpart in the reference (launch-shape control for tuning
 * and benchmarks). */
int pfm_set_tuning(pfm_ctx* h, int lanes_per_row, int block);

/* Co-scheduled passes (default on).  For graphene on a metal -- exactly
 * rjl, tb and a ljc/morsec fed by that tb list, with the rjl rows, the
 * graphene rows and the metal rows of ljc/morsec sharing no atom -- passes
 * over disjoint atoms share launches: the rjl density pass with the tb
 * bond-order pass, the rjl force pass with the graphene pass of ljc/morsec,
 * the tb force pass (with the normal-derivative terms) with the metal rows.
 * When every interaction is lj, lj1g or rjl, passes whose rows share no
 * atom share launches in phases (a binary gas's lj1g A and B, then its lj
 * rows of both directions; the rjl passes of a batch beside them).  The
 * surrogate's descriptor, network and backward passes run as one kernel
 * (the same bits as three).  Results equal the separate launches' up to
 * the order of the FP64 force sums.  pfm_set_fusion(h, 0) launches every pass on its own.  No
 * counterpart in the reference (launch schedule). */
int pfm_set_fusion(pfm_ctx* h, int on);

/* Lanes per row (1,2,4,8,16,32) of the row passes of interaction `inter`
 * (1-based, settings order) when they are launched on their own; 0 returns
 * it to the count of pfm_set_tuning.  Co-scheduled launches take the
 * pfm_set_tuning count for all of their passes.  No counterpart in the
 * reference (launch-shape control for the autotuner). */
int pfm_set_pass_lanes(pfm_ctx* h, int inter, int lanes);

/* Captured steps (default on).  pfm_run records a block of steps whose list
 * and zero-momentum schedule repeats (the least common multiple of the list
 * periods, up to 64 steps) and that holds no energy step as one HIP graph,
 * and replays it for every later such block; results are identical to
 * launching the steps one by one.  pfm_set_graphs(h, 0) launches every step
 * directly.  No counterpart in the reference (launch mechanics). */
int pfm_set_graphs(pfm_ctx* h, int on);
/* nvms blocks (default on).  Under nvms md() tests abs(PE-PE_prev) <= ms_de
 * at every step (md_simulation.f90:142-147), which needs each step's
 * energies on the host.  pfm_run instead runs blocks of steps (the list
 * schedule's period, up to 32, else 16; captured like other blocks) that keep
 * every step's energies and state in device memory, reads the energies back
 * once per block, and on the first step whose test holds restores the state
 * of the step before it; the lists are rebuilt from a fresh sort at the next
 * step.  Results, exit step and energies are those of testing every step.
 * Systems without group changes, batches included (a batch stops when every
 * replica meets the test); pfm_set_speculation(h, 0) tests every step on
 * the host.  No counterpart in the reference. */
int pfm_set_speculation(pfm_ctx* h, int on);

/* Blocks captured and blocks launched from graphs since the handle was made. */
int pfm_graph_count(pfm_ctx* h, long* captured, long* launched);

/* Output records.  md() stops at every log, out, snapshot and trajectory
 * step to compute energies and write files (md_simulation.f90:188-229,
 * md_read_write.f90:65-107).  With records set, pfm_run takes these values
 * on the device at the steps they are due, without leaving the run:
 *   energy record at every step some energy period divides: interaction
 *     energies, kinetic energy and temperature of all_moving, chain
 *     energies, and the out block's sums (calculate_force_sum,
 *     calculate_mass_center, calculate_mass_center_velocity over all_atoms,
 *     md_general.f90:184-234,277-298; find_max_velocity over every atom,
 *     md_general.f90:366-380);
 *   frame at every step some frame period divides: positions and velocities
 *     of every atom, double[n][3] each in original order.
 * The record kernels run in the step's launch sequence (inside captured
 * blocks too) and write each record into a slot of pinned host memory
 * (256 energy slots, frame_slots frames); pfm_run passes the records to fn
 * in step order as their slots complete, while later steps run, and waits
 * for the oldest when a ring is full.  The pointers in the record are valid
 * during the call only.  The trajectory is identical to stopping at
 * every recorded step.  Every record of a pfm_run call is delivered before it
 * returns; a nonzero return from fn ends the run with PFM_E_INVALID.
 * Periods <= 0 are ignored; no periods, or fn NULL, turns records off.
 * Single systems only (not batches).  No counterpart in the reference, which
 * computes and writes these synchronously inside the step loop. */
typedef struct pfm_record {
  int step;              /* md_step of the record                          */
  int integrator;        /* PFM_NVT / PFM_NVE / PFM_NVMS                   */
  int has_energy;        /* the energy fields below are set                */
  int has_frame;         /* pos and vel are set                            */
  double sim_time;       /* simulated time after the step (fs)             */
  double pe, ke, temp;   /* sum of e_inter; all_moving kinetic energy (eV), temperature (K) */
  double force_sum[3];   /* sum of forces over all_atoms (eV/A)            */
  double mass_center[3]; /* centre of mass of all_atoms (A)                */
  double mass_center_vel[3]; /* centre-of-mass velocity of all_atoms (A/fs) */
  double max_vel;        /* largest |v| over every atom (A/fs)             */
  const double* e_inter; /* [n_interactions] (eV)                          */
  const double* e_nhc;   /* [n_chains] chain energies (eV)                 */
  const double* pos;     /* double[n][3] or NULL                           */
  const double* vel;     /* double[n][3] or NULL                           */
  const int* group_n;    /* [33]: active atoms of group g at the step (pfm_group_count) */
} pfm_record;
typedef int (*pfm_record_fn)(void* user, const pfm_record* rec);
int pfm_set_records(pfm_ctx* h, int n_energy_periods, const int* energy_periods, int n_frame_periods,
                    const int* frame_periods, int frame_slots, pfm_record_fn fn, void* user);

/* Runtime group growth: one change_group line of the settings
 * (md_simulation.f90:63-70), applied at the top of every step as md() does
 * (md_simulation.f90:116-119) with change_particle_group_N
 * (md_general.f90:82-94): up to step ts1 group `to` holds as many of its
 * atoms as group `from` does (one more at ts1), then one more every frec
 * steps before ts2, never more than its members; the active atoms are the
 * first n in the group's order.  Everything that reads the group sees only
 * its active atoms: integration, kinetic energy and temperature, zero
 * momentum, chains, and the list search (rows of inactive members stay
 * empty until the first rebuild after they join, as in find_neighbours).
 * Taken for role and chain groups and the groups of lj, lj1g, rjl, tb,
 * rebosc and ljc/morsec lists (not surrogate lists: PFM_E_INVALID at the
 * first run).  In a batch the rule applies to every replica's own counts
 * (each replica is its own md() run).  Changes are added before the first
 * pfm_run.
 * pfm_group_count gives the active atoms of a group after the last step. */
int pfm_add_group_change(pfm_ctx* h, int from, int to, int ts1, int ts2, int frec);
int pfm_group_count(pfm_ctx* h, int gid, int* n);

/* Learned surrogate (interaction kind PFM_SUR).  None of these has a
 * counterpart in the reference; they serve the training and inference of a
 * per-atom network that stands in for TB_forces + MorseC_forces
 * (TersoffBrenner.f90:74-150, MorseCosine.f90:53-139) on graphene over a
 * metal.  E = sum over g1 atoms of NN((G_i - mu) * isg), G_i the 40
 * descriptors of atom i, NN a 40-64-64-1 tanh perceptron on BF16 MFMA.
 *
 * pfm_sur_set_params: the network, in the PFM_SUR_NTHETA layout
 *   mu[40] isg[40] W1[64][40] b1[64] W2[64][64] b2[64] w3[64] b3.
 * pfm_sur_descriptors: G of every g1 atom at the current positions,
 *   double[N_g1][40] in group order (lists from the last step).
 * pfm_sur_loss_grad: at the current positions (lists from the last step),
 *   the loss of one reference frame
 *     L = w_e ((E - e_ref)/N_g1)^2 + w_f/(3 N_g2) sum_{a in g2} |F_a - f_ref,a|^2,
 *   F the surrogate's own forces (they replace the handle's forces), f_ref
 *   double[n_atoms][3] in original order; loss[3] = {L, energy term, force
 *   term}; grad[PFM_SUR_NTHETA] = dL/dtheta (zero for mu and isg). */
int pfm_sur_set_params(pfm_ctx* h, int inter, const double* theta, int n_theta);
int pfm_sur_descriptors(pfm_ctx* h, int inter, double* G);
int pfm_sur_loss_grad(pfm_ctx* h, int inter, const double* f_ref, double e_ref, double w_e, double w_f,
                      double* loss, double* grad);

int  pfm_last_error(pfm_ctx* h, char* buf, int len);
int  pfm_destroy(pfm_ctx* h);

#ifdef __cplusplus
}
#endif
#endif
