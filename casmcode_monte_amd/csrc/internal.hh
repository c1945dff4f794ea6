// internal.hh -- device data layout shared by the kernels and the C ABI host code.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "../../include/casm_mi355x/mcgpu.h"
#include "rng.hh"

namespace mcg {

// ---------------------------------------------------------------------------
// EXACT mode: a chain per workgroup, of one wave (scalar walk) or five (block walk).
// ---------------------------------------------------------------------------

// Number of (old spin, neighbour sum) classes of the 2D square NN Ising flip:
// class k = (s_old > 0) * 5 + (nbr_sum + 4) / 2.
constexpr int EXACT_NCLASS = 10;

// Read-only per-chain parameters (built on the host).
struct ExactParams {
  int32_t rows, cols;  // shape[0], shape[1]
  int32_t n;           // sites
  int32_t fold;        // 1: compute the row/column-fold formation energy at samples
  int32_t self_nb;     // neighbour slots that are the site itself (rows==1, cols==1)
  uint32_t mark_mask;  // conflict marks of the block walk: entry (site & mark_mask)
  uint64_t div_magic;  // floor(l / rows) = (l * div_magic) >> 40 for l < 2^24
  uint64_t thr[EXACT_NCLASS];  // accept a drawn word x iff x < thr[k]
  uint32_t neg_mask;   // bit k: dE < 0, accept without drawing (metropolis.hh:28-30)
  uint32_t full_mask;  // bit k: every drawn word accepts (thr == 2^64)
  double dq[EXACT_NCLASS];  // fl(dE_k / n_unitcells), occupation_metropolis.hh:141
  double negJ;               // -J, for the row/column fold
  int64_t lat_off;           // byte offset of this chain's lattice in the pool
  int64_t block_from;        // launches of fewer attempts take the scalar walk on HBM
};

// The block walk's lattice: a site's class in four bits, so at most 2^18 sites
// (the records' site field) of two per byte.
constexpr int64_t EXACT_BLOCK_MAX_SITES = int64_t(1) << 18;
constexpr uint32_t EXACT_WALK_FIXED_LDS = 14704;  // engine, records and the other fixed parts
// LDS bytes of one chain in the block walk (classes, fixed parts, conflict
// marks, fold scratch) and in the scalar walk (one byte per site, fold scratch).
inline int64_t exact_block_lds_bytes(const ExactParams &P) {
  return 4 * ((((int64_t)P.n + 7) / 8 + 3) & ~int64_t(3)) + (int64_t)EXACT_WALK_FIXED_LDS +
         4 * ((int64_t)P.mark_mask + 1) +
         (P.fold ? 4 * ((int64_t)P.rows + P.cols) : 0);
}
inline int64_t exact_scalar_lds_bytes(const ExactParams &P) {
  return (((int64_t)P.n + 15) & ~int64_t(15)) + 4 * ((int64_t)P.rows + P.cols);
}

// The most dynamic LDS that launches of kernel fn ask for; refused if it does not fit a
// workgroup's 160 KB beside what fn has static, which is nothing if fn takes its dynamic
// array to start at LDS address 0 (walk.hh).
inline hipError_t set_dynamic_lds(const void *fn, int bytes, bool at_zero) {
  hipFuncAttributes a;
  const hipError_t e = hipFuncGetAttributes(&a, fn);
  if (e != hipSuccess) return e;
  if (a.sharedSizeBytes > (at_zero ? size_t(0) : size_t(160 * 1024 - bytes)))
    return hipErrorInvalidDeviceFunction;
  return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

// Read-write per-chain state of the sequential modes: the engine's words, and the rest,
// which the host reads after a run (its bytes follow one another).
struct EngineState {
  uint64_t mt[MT_N];  // std::mt19937_64 state words
};
struct ChainState {
  int64_t pos;        // index of the next output (312: twist first)
  int64_t n_pass, n_accept, n_reject;
  int64_t S, M;       // exact bond sum and magnetisation
  double e_run;       // running potential energy per unit cell (NFOLD: the total rate
                      // at the pending event's selection)
  int64_t n_samples;  // records the run produced (written while below the capacity)
  // NFOLD
  double time;           // simulated time
  int64_t pending_site;  // event selected at the end of a sampled pass, or -1
  double pending_dt;     // its time increment
  int64_t next_k;        // next time-grid sample index (sample at next_k * period)
  int64_t frozen;        // NFOLD: the total rate reached 0 on the time grid; OCCUPANT: the
                         // swap types ran out of events
  // EXACT: attempts done in the current pass (0 <= step < n; runs of whole
  // passes keep it, runs of single steps move it); OCCUPANT: steps done in the
  // current pass (0 <= step < n_mut); NFOLD and KMC: events done in the
  // current pass
  int64_t step;
  // OCCUPANT: sites of each asymmetric unit holding its occupant 0
  int32_t occ_cnt0[8];
  // KMC: attempts since the last event, and the sums over atoms of dx^2 +
  // dy^2, dx and dy (time, next_k and frozen are shared with NFOLD)
  int64_t kmc_k;
  int64_t kmc_sum_sq, kmc_sum_dx, kmc_sum_dy;
  // KMC pending event (pending_site >= 0): its direction and attempts; its
  // time is in pending_dt
  int64_t kmc_pdir, kmc_pk;
};
struct ExactState : EngineState, ChainState {};
static_assert(sizeof(ExactState) == sizeof(EngineState) + sizeof(ChainState) &&
              sizeof(ChainState) % 8 == 0);

// Every active chain makes n_passes * n + n_steps attempts from where it stands.
void launch_exact(const ExactParams *P, ExactState *S, int8_t *lat_pool, mcg_sample *series,
                  int64_t series_cap, const uint8_t *active, int n_chains, int64_t n_passes,
                  int64_t n_steps, int64_t sample_period, int lds_bytes, bool lattice_in_lds,
                  bool block_walk, hipStream_t stream);

// ---------------------------------------------------------------------------
// OCCUPANT mode: occupant events over an OccLocation with several asymmetric
// units (semi-grand canonical single-site events or canonical pair swaps),
// a chain per workgroup of two (general kernel) or five waves.
// ---------------------------------------------------------------------------
constexpr int OCC_MAX_ASYM = 8;
constexpr int OCC_MAX_CAND = 2 * OCC_MAX_ASYM;
constexpr int OCC_MAX_SWAPS = 16;
// classes: swap type i, neighbour sum of a, and (pairs) of b after a changed,
// k = i * 25 + ((Sa + 4) / 2) * 5 + (Sb + 4) / 2
constexpr int OCC_NCLASS = OCC_MAX_SWAPS * 25;

struct OccParams {
  int32_t rows, cols, n, n_mut;
  int32_t canonical;  // 1: pair swaps (propose_canonical_event), 0: single sites
  int32_t n_asym, n_cand, n_swaps;
  int32_t window;     // stream positions evaluated per block
  int32_t pad;
  uint64_t div_magic; // floor(l / rows) = (l * div_magic) >> 40
  // per unit: segment of the list array (units with one occupant: size 0)
  int32_t asym_off[OCC_MAX_ASYM], asym_size[OCC_MAX_ASYM];
  // per candidate (OccCandidateList order): unit and occupant index
  int32_t cand_asym[OCC_MAX_CAND], cand_occ[OCC_MAX_CAND];
  // swap types: candidate indices (cand_a, cand_b)
  int32_t swap_a[OCC_MAX_SWAPS], swap_b[OCC_MAX_SWAPS];
  int64_t lat_off;    // lattice byte offset; the lists start at entry lat_off of the list pool
};

// per chain: the class thresholds (first word whose canonical double reaches
// exp(-beta dE)), fl(dE / n_unitcells), and flags (bit 0: dE < 0, accepted
// without a draw; bit 1: every word accepts)
struct OccTables {
  uint64_t thr[OCC_NCLASS];
  double dq[OCC_NCLASS];
  uint8_t flags[OCC_NCLASS];
};

// LDS bytes of one chain: lattice and the list array (occupant_sgc_kernel: behind
// its fixed parts, nothing static).
constexpr int OCC_MAX_SITES_LDS = 40000;
constexpr uint32_t OCC_SGC_FIXED_LDS = 30032;
inline int occ_lds_bytes(const OccParams &P) {
  return ((P.n + 15) & ~15) + ((2 * P.n_mut + 15) & ~15);
}

// Every active chain makes n_passes * n_mut + n_steps steps from where it
// stands (fewer if its swap types run out of events: ExactState::frozen).
// asym_pool: every site's asymmetric unit at the lattice offsets.  sgc_units: the
// pairs of swap types of occupant_sgc_kernel, or 0 for the general kernel.
void launch_occupant(const OccParams *P, const OccTables *T, ExactState *S, int8_t *lat_pool,
                     int32_t *list_pool, const int8_t *asym_pool, mcg_sample *series,
                     int64_t series_cap, const uint8_t *active, int n_chains, int64_t n_passes,
                     int64_t n_steps, int64_t sample_period, bool canonical, int n_swaps,
                     int sgc_units, int lds_bytes, hipStream_t stream);
// Dynamic LDS limits of the general kernel (its static LDS is ~23 KB) and of
// occupant_sgc_kernel.
hipError_t occupant_set_max_lds(int general_bytes, int sgc_bytes);

// ---------------------------------------------------------------------------
// KMC mode: kinetic Monte Carlo with atom tracking for a square lattice gas,
// a chain per workgroup of two (general kernel) or five waves.
// ---------------------------------------------------------------------------
// classes of a hop: a - b + 3 (a, b: atoms next to the origin other than at
// the target, next to the target other than at the origin), dE = J (a - b)
constexpr int KMC_NCLASS = 7;

struct KmcParams {
  int32_t rows, cols, n, n_atoms;
  int32_t window;      // stream positions evaluated per block
  uint32_t draw_mask;  // bit k: dE > 0, the class draws an acceptance word
  uint32_t full_mask;  // bit k: every drawn word accepts
  int32_t pad;
  uint64_t div_magic;  // floor(l / rows) = (l * div_magic) >> 40
  double attempt_rate; // R = 4 * n_atoms: attempts per unit time
  double time_period;  // > 0: samples at k * time_period; 0: by pass
  double J;
  int64_t spin_limit;  // attempts without an event after which a chain stops (frozen)
  int64_t lat_off;     // lattice byte offset; the lists start at entry lat_off of the
                       // list pool, the atoms (4 int32 each) at entry 4 lat_off of the atom pool
  uint64_t thr[KMC_NCLASS];
  // hop correlations (0: off): every hop_every-th jump of an atom is recorded,
  // at most hop_max per atom; record k of atom a at hop pool entry
  // hop_off + k * n + a, the atoms' record counts at count pool entry lat_off + a
  int32_t hop_every, hop_max;
  int64_t hop_off;
};

// One hop-correlation record: the atom's displacement since its occupation was
// set, the step within the pass and the pass of the event, and its time.
struct KmcHop {
  int32_t dx, dy;
  int64_t step, pass;
  double time;
};

// LDS bytes of one chain: list, positions and site atoms (16-bit), atom
// displacements and jumps (32-bit).
inline int kmc_lds_bytes(int n) {
  const int a = (n + 7) & ~7;
  return 3 * 2 * a + 3 * 4 * a;
}

// LDS bytes of kmc_walk_kernel: fixed parts, sites (word and mark), list, atoms.
constexpr uint32_t KMC_WALK_FIXED_LDS = 21088;
inline int kmc_walk_lds_bytes(int n) { return (int)KMC_WALK_FIXED_LDS + 22 * ((n + 7) & ~7); }

// Every active chain applies its pending event, if any, then makes events up
// to n_passes * n + n_steps in all (fewer if it freezes: ExactState::frozen).
// An event whose time reaches stop_time is left pending instead of applied
// (the chain stops there); with select_at_end a chain that reached the count
// selects one more event and leaves it pending.  walk: by kmc_walk_kernel, which
// takes launches without a stop time, select_at_end, pending events or hop
// correlations, at spin limits below 2^31, of chains that fit it
// (kmc_walk_lds_bytes).
void launch_kmc(const KmcParams *P, ExactState *S, int8_t *lat_pool, int32_t *list_pool,
                int32_t *atom_pool, KmcHop *hop_pool, int32_t *hop_count_pool,
                mcg_sample *series, int64_t series_cap, const uint8_t *active, int n_chains,
                int64_t n_passes, int64_t n_steps, int64_t sample_period, double stop_time,
                int select_at_end, bool walk, int lds_bytes, hipStream_t stream);
hipError_t kmc_set_max_lds(int general_bytes, int walk_bytes);

// ---------------------------------------------------------------------------
// CANONICAL mode: pair swaps at fixed composition, a chain per workgroup of five waves.
// ---------------------------------------------------------------------------

// Classes of a swap (site a: -1 -> +1, then site b: +1 -> -1): the neighbour
// sum of a before the swap and the neighbour sum of b after a has flipped,
// k = ((Sa + 4) / 2) * 5 + (Sb + 4) / 2.
constexpr int CANON_NCLASS = 25;

struct CanonParams {
  int32_t rows, cols, n;
  int32_t nA, nB;        // sizes of the species-0 (spin -1) and species-1 (+1) lists
  int32_t fold;          // 1: compute the row/column-fold formation energy at samples
  int32_t self_nb;       // neighbour slots that are the site itself
  int32_t window;        // 1: step by step
  uint32_t mark_mask;    // conflict marks: 4-byte entry (site's address & mark_mask)
  uint32_t neg_mask;     // bit k: dE < 0, accept without drawing
  uint32_t full_mask;    // bit k: every drawn word accepts
  int32_t pad;
  uint64_t thr[CANON_NCLASS];
  double dq[CANON_NCLASS];  // fl(dE_k / n_unitcells)
  double negJ;
  int64_t lat_off;       // lattice byte offset; the lists start at entry lat_off of the list pool
};

// What a chain is accepted by: lattice, lists, up to 8192 marks and the fold scratch
// within EXACT_LDS_MAX.
inline int canon_lds_bytes(const CanonParams &P) {
  int marks = 64;
  while (marks < P.n && marks < 8192) marks <<= 1;
  return ((P.n + 15) & ~15) + 4 * marks + ((2 * P.n + 15) & ~15) + 4 * (P.rows + P.cols);
}
// LDS bytes of the kernel (nothing static): fixed parts, lists, lattice, conflict
// marks, fold scratch.
constexpr uint32_t CANON_FIXED_LDS = 20304;
inline int canon_walk_lds_bytes(const CanonParams &P) {
  return (int)CANON_FIXED_LDS + ((2 * P.n + 15) & ~15) + ((P.n + 15) & ~15) +
         4 * (int)(P.mark_mask + 1) + 4 * (P.rows + P.cols);
}

void launch_canonical(const CanonParams *P, ExactState *S, int8_t *lat_pool, int32_t *list_pool,
                      mcg_sample *series, int64_t series_cap, const uint8_t *active,
                      int n_chains, int64_t n_passes, int64_t sample_period, int lds_bytes,
                      hipStream_t stream);
// Dynamic LDS limit of the canonical kernel.
hipError_t canonical_set_max_lds(int bytes);

// ---------------------------------------------------------------------------
// NFOLD mode: rejection-free single-site flips, one chain per wavefront.
// ---------------------------------------------------------------------------
struct NfoldParams {
  int32_t rows, cols, n;
  int32_t pad;
  uint64_t div_magic;   // floor(l / rows) = (l * div_magic) >> 40
  double rate[10];      // Metropolis rate of class k = (s > 0) * 5 + (nbr_sum + 4) / 2
  double time_period;   // > 0: samples on the time grid k * time_period; else by pass
  int64_t lat_off;      // lattice byte offset; the class array starts at entry lat_off
  int32_t sample_start; // by pass: also sample pass 0 (the first event selected then)
  int32_t pad2;
};

// class array and positions (16-bit each; a position's bit 15 is the spin)
inline int nfold_lds_bytes(const NfoldParams &P) { return 4 * P.n + 64; }

// max_events >= 0: event by event (no records, n_passes ignored): apply the
// pending event unless its time reaches stop_time, then up to max_events
// events, leaving pending the one that reaches stop_time or, with
// select_at_end, the one after the last; max_events < 0: whole passes.
// general: some active chain is 1 or 2 wide.
void launch_nfold(const NfoldParams *P, ExactState *S, int8_t *lat_pool, int32_t *list_pool,
                  mcg_sample *series, int64_t series_cap, const uint8_t *active, int n_chains,
                  int64_t n_passes, int64_t sample_period, int sample_now, int64_t max_events,
                  double stop_time, int select_at_end, bool general, int lds_bytes,
                  hipStream_t stream);
hipError_t nfold_set_max_lds(int bytes);

// ---------------------------------------------------------------------------
// CHECKERBOARD mode
// ---------------------------------------------------------------------------

// Acceptance classes: (old spin, NN sum, NNN sum).  For coordination numbers
// z1 (NN) and z2 (NNN) the sums take z+1 values each (steps of 2).
struct CheckerParams {
  int32_t L0, L1, L2;      // shape
  int32_t ncolor;          // 2, 4 or 8
  int32_t z1, z2;          // coordination numbers (z2 = 0 without J2)
  int32_t ndim;            // 2 or 3
  int32_t quad_only;       // 1: use the 4-site path even when 16-site chunks fit
  uint32_t key0, key1;     // Philox key (chain seed)
  int64_t n;               // sites
  int64_t lat_off;         // byte offset in the lattice pool
  int64_t tab_off;         // offset of the chain's threshold table (uint32 entries)
  // HBM paths: the chain's observable changes of a pass (S1, S2, M, accepted), summed
  // over CHECKER_PARTS slots, for each of the passes between two record launches; zero
  // after one
  int64_t *parts;
};

// Workgroups add their changes to slot (index % CHECKER_PARTS), 64 bytes apart:
// additions to one address take ~10 ns each whoever makes them (MI355X: 4096 to the
// four fields of one state 41 us, whatever else the launch did).
constexpr int CHECKER_PARTS = 64;
constexpr int CHECKER_PART_STRIDE = 8;  // int64 per slot
constexpr int CHECKER_PASS_PARTS = CHECKER_PARTS * CHECKER_PART_STRIDE;
// Passes between two record launches at most: the launches are told how far ahead of the
// state's pass counter they are.
constexpr int CHECKER_AHEAD = 8;

// Acceptance table of a chain: entry (b << 7) | (c1 << 4) | c2 for old spin
// bit b and up-neighbour counts c1 <= 6, c2 <= 12 (unused entries 0), so the
// class bytes of four sites come from one packed-word shift-and-add.
constexpr int CHECKER_NTAB = 256;
__host__ __device__ inline int checker_class(int b, int c1, int c2) {
  return (b << 7) | (c1 << 4) | c2;
}

struct CheckerState {
  int64_t n_pass;
  int64_t n_accept;
  int64_t S1, S2, M;       // exact integer observables (FCC: P1, P2, N1)
  int64_t n_samples;
  int64_t S3, T3;          // FCC: P3 and the triangle count
};

// A chain's parameters in a launch `ahead` passes ahead of the state's counter: its
// changes go to that pass's slots.
__device__ __forceinline__ CheckerParams checker_ahead(const CheckerParams *Pp, int chain,
                                                       int ahead) {
  CheckerParams P = Pp[chain];
  P.parts += ahead * CHECKER_PASS_PARTS;
  return P;
}

// A workgroup's observable changes into its slot of the chain's (by one thread).
__device__ __forceinline__ void checker_add_part(const CheckerParams &P, int index, long long a1,
                                                 long long a2, long long am, long long an) {
  unsigned long long *p = reinterpret_cast<unsigned long long *>(P.parts) +
                          (index & (CHECKER_PARTS - 1)) * CHECKER_PART_STRIDE;
  if (a1) atomicAdd(p, (unsigned long long)a1);
  if (a2) atomicAdd(p + 1, (unsigned long long)a2);
  if (am) atomicAdd(p + 2, (unsigned long long)am);
  if (an) atomicAdd(p + 3, (unsigned long long)an);
}

void launch_checker_lds(const CheckerParams *P, CheckerState *St, int8_t *lat_pool,
                        const uint32_t *tables, mcg_sample *series, int64_t series_cap,
                        const uint8_t *active, int n_chains, int64_t n_passes,
                        int64_t sample_period, int lds_bytes, int block, hipStream_t stream);

void launch_checker_color(const CheckerParams *P, CheckerState *St, int8_t *lat_pool,
                          const uint32_t *tables, const int32_t *work, int n_work_items,
                          int color, int upt, int ahead, hipStream_t stream);

// Chains with an odd edge (checker_ring.hip): ring colourings, natural layout.
void launch_checker_ring_lds(const CheckerParams *P, CheckerState *St, int8_t *lat_pool,
                             const uint32_t *tables, mcg_sample *series, int64_t series_cap,
                             const uint8_t *active, int n_chains, int64_t n_passes,
                             int64_t sample_period, int lds_bytes, int block,
                             hipStream_t stream);
// the class launches of one HBM pass of the listed chains (the pass counter and
// the record follow in launch_checker_record)
void launch_checker_ring_pass(const CheckerParams *P, CheckerState *St, int8_t *lat_pool,
                              const uint32_t *tables, const int32_t *chains, int n_ring,
                              int per_chain, int ndim, int ahead, hipStream_t stream);
hipError_t checker_ring_set_max_lds(int bytes);

// Spins (+1/-1, site order) of sites [first, first + count) of one lattice into
// out (16-byte aligned); L0: its line length when lines hold their even sites
// first, 0 when sites are in order.
void launch_checker_spins(const int8_t *lat, int64_t L0, int64_t first, int64_t count, int8_t *out,
                          hipStream_t stream);
// Every chain's sample count to 0: of the sequential chains' states, or (xs null) of
// the checkerboard ones'.
void launch_clear_samples(ExactState *xs, CheckerState *cs, int n_chains, hipStream_t stream);
// Words [first, first + count) of the chains' ChainStates, one after another, into out.
void launch_chain_states(const ExactState *xs, int64_t first, int64_t count, int64_t *out,
                         hipStream_t stream);

// the state, counter and records of the last `passes` passes (at most CHECKER_AHEAD)
void launch_checker_record(CheckerState *St, int64_t *parts, mcg_sample *series,
                           int64_t series_cap, const uint8_t *active, int n_chains,
                           int64_t sample_period, int passes, hipStream_t stream);

// Bit-packed path (checker_bits.hip): 2D lattices of lines of up to 4096 sites
// streamed in bands, 3D J1+J2 ones a plane per workgroup.  An item is a wave's bands
// (chain, first line of the first, lines of each, bands) or a pair of planes (chain,
// first plane); off: the chain's first word in `bits` (bit_words of them: 2D two
// buffers, used in turn by passes).
struct BitItem {
  int32_t chain, j0, H, n_groups;
  int64_t off;
};
struct BitPass {
  uint32_t *bits = nullptr;
  const BitItem *items = nullptr;
  int n_items = 0;
  bool four = false;                   // 2D: 4 colours (else 2)
  int plane_lds = 0, plane_block = 0;  // 3D, 8 colours (else 0): LDS bytes, threads
  bool cube = false;                   // 3D, 2 colours
  int oct = 4;                         // a thread takes 8 oct sites of a word
};
struct BitLaunch {  // arguments: parameters, states, bits, tables, items, last, passes ahead
  void *fn;
  unsigned grid, block, lds;
  int last;
};
constexpr int CHECKER_PLANE_MAX_LDS = 144 * 1024;
bool bit_fits(const CheckerParams &P);
int64_t bit_words(const CheckerParams &P);
int bit_groups(const CheckerParams &P, int oct);  // 2D: bands a wave takes side by side
int bit_waves();                         // 2D: items of a workgroup, all of one chain
int64_t bit_cube_blocks(const CheckerParams &P, int oct);
int bit_plane_lds(const CheckerParams &P);
int bit_plane_block(const CheckerParams &P, int oct);
int bit_pass_launches(const BitPass &b, BitLaunch (&L)[2]);
void launch_bit_pass(const CheckerParams *P, const CheckerState *St, const uint32_t *tables,
                     const BitPass &b, int ahead, hipStream_t stream);
// the listed chains' lattices (items' chain and off) into bits and back; max_words:
// the most words of one lattice
void launch_bit_pack(const CheckerParams *P, const CheckerState *St, const int8_t *lat_pool,
                     uint32_t *bits, const BitItem *chains, int n_chains, int64_t max_words,
                     hipStream_t stream);
void launch_bit_unpack(const CheckerParams *P, const CheckerState *St, int8_t *lat_pool,
                       const uint32_t *bits, const BitItem *chains, int n_chains,
                       int64_t max_words, hipStream_t stream);
hipError_t bit_set_max_lds();

// 2D chains that fit a workgroup, as bits in LDS (checker_bits.hip): words of 8 oct
// sites, threads, LDS bytes.  word_tasks: the most words of one class.
struct WordPlan {
  int oct = 0, block = 0, lds = 0;  // oct 0: not used
};
constexpr int WORDS_MAX_LDS = 96 * 1024;
int word_lds(int L0, int L1, int oct);
int word_tasks(int L0, int L1, bool ring, bool nnn, int oct);
void launch_checker_words(const CheckerParams *P, CheckerState *St, int8_t *lat_pool,
                          const uint32_t *tables, mcg_sample *series, int64_t series_cap,
                          const uint8_t *active, int n_chains, int64_t n_passes,
                          int64_t sample_period, bool ring, bool nnn, const WordPlan &w,
                          hipStream_t stream);
hipError_t words_set_max_lds();

hipError_t checker_graph_add_passes(hipGraph_t g, const CheckerParams *P, CheckerState *St,
                                    int8_t *lat_pool, const uint32_t *tables,
                                    const int32_t *work, int n_work_items, int ncolor, int upt,
                                    mcg_sample *series, int64_t series_cap,
                                    const uint8_t *active, int n_chains, int64_t sample_period,
                                    int passes, const int32_t *band_work, int n_bands,
                                    int ring_bytes, const BitPass &bit, int64_t *parts,
                                    const int32_t *pair_work,
                                    int n_pairs, int pair_lds, int tile_grid);

// Line-class path (4 and 8 colourings): one launch per line class, both
// halves of each line.  lds_bytes == 0: items (chain, first colour-class line,
// lines, 0) read straight from HBM, one workgroup per item.  lds_bytes > 0:
// tiles (chain, jh0, kh0, TJ | TK << 16) of class lines staged with their
// neighbour lines in LDS ((2TJ+1) x (2TK+1) x L0 bytes, 2D (2TJ+1) x L0, at
// most checker_tile_max_bytes()), tile_grid persistent workgroups.
void launch_checker_pair(const CheckerParams *P, CheckerState *St, int8_t *lat_pool,
                         const uint32_t *tables, const int32_t *pair_work, int n_items,
                         int line_class, int lds_bytes, int tile_grid, int ahead, hipStream_t stream);
hipError_t checker_pair_set_max_lds(int bytes);
int checker_pair_block();
int checker_tile_max_bytes();

// 2D band path: one launch over (chain, first line, lines) bands, then the
// band-edge launch; ring_bytes = checker_band_ring_lines() * L0 (largest chain).
void launch_checker_band(const CheckerParams *P, CheckerState *St, int8_t *lat_pool,
                         const uint32_t *tables, const int32_t *band_work, int n_bands,
                         int ring_bytes, int ahead, hipStream_t stream);
int checker_band_ring_lines();
hipError_t checker_band_set_max_lds(int bytes);


// FCC cluster expansion (fcc.hip): CheckerParams with ncolor = 64, tab_off in
// doubles into the per-chain acceptance tables, tri = the 4096-entry
// triangle-count table of the nearest-neighbour occupancy mask.
// bit_lines: the bit-line kernels (every chain L0 <= 64, lattice in LDS as one
// 64-bit word per line, tri_lines the triangle table in its mask bit order);
// class_lines (with bit_lines, every chain L0 <= 32): one thread per class
// line with bit-sliced counts, else 4-site units
struct FccSched;
void launch_fcc(const CheckerParams *P, CheckerState *St, int8_t *lat_pool, const double *tables,
                const uint8_t *tri, const uint8_t *tri_lines, const FccSched *sched,
                mcg_sample *series, int64_t series_cap, const uint8_t *active, int n_chains,
                int64_t n_passes, int64_t sample_period, int lds_bytes, bool lattice_in_lds,
                bool bit_lines, bool wide_lines, bool class_lines, int block,
                hipStream_t stream);
// the triangle pairs of the class-line kernel against the host's table in the
// bit-line mask order (true: they agree for every mask)
bool fcc_tri_pairs_check(const std::vector<uint8_t> &tri_lines);

// ---------------------------------------------------------------------------
// Statistics on the device sample series
// ---------------------------------------------------------------------------
struct ObsParams {
  int64_t n_sites;
  double negJ1, negJ2;
  double mu;
  int32_t fold;  // use e_fold as E_f
  int32_t observable;
  int32_t fcc;   // FCC cluster expansion: E_f from the counts and coef
  int32_t running;  // OCCUPANT: the potential energy is the record's running e_run
  double coef[6];  // FCC: V0, V1, V2/6, V3/3, V4/12, Vt/8
};

void launch_stats(const mcg_sample *series, int64_t first, int64_t count, ObsParams op,
                  double *d_out, hipStream_t stream);

void launch_weighted_stats(const mcg_sample *series, int64_t first, int64_t count, ObsParams op,
                           int method, int64_t n_resamples, double *d_out, hipStream_t stream);
void launch_equilibration(const mcg_sample *series, int64_t count, ObsParams op, double prec,
                          int weighted, int64_t *d_out, hipStream_t stream);
// Equilibration and statistics of n chains in one launch (check_batch_kernel).
void launch_check_batch(const mcg_sample *series, int64_t series_cap, const int64_t *chains,
                        const int64_t *counts, const ObsParams *ops, const int64_t *scratch_off,
                        int n, double prec, double *scratch, double *out, hipStream_t stream);
// Device address of the fixed statistics scratch (MCG_STATS_NOALLOC_MAX doubles)
// on device `dev`: looked up once per device by the init call, with that
// device current; nullptr before it.
hipError_t stats_noalloc_scratch_init(int dev);
double *stats_noalloc_scratch(int dev);

}  // namespace mcg
