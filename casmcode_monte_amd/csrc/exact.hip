// exact.hip -- EXACT mode: the reference's sequential random-site Metropolis
// chain, reproduced bit for bit by one walking wavefront per chain.
//
// Reference: the main loop of basic_occupation_metropolis.hh:381-422 driving the
// SGC Ising calculator (basic_semigrand_canonical.hh:308-320 propose/apply,
// :178-192 potential delta, model.hh:305-345 formation-energy delta) with
// metropolis_acceptance (metropolis.hh:25-35) and RandomNumberGenerator over
// std::mt19937_64 (RandomNumberGenerator.hh:31-41).
//
// Layout: one chain per workgroup.  The chain's int8 lattice (column-major,
// l = i + rows*j) lives in LDS when it fits, else in HBM.  The scalar walk
// (exact_kernel) is one 64-lane wavefront that twists the MT19937-64 state in
// LDS itself (two dependency-free phases of 156 words) and executes every other
// step in lockstep with scalar (readfirstlane) operands.  The block walk
// (exact_block_kernel) keeps the lattice in LDS as four-bit classes and has five
// wavefronts: one walks, one adds energies, three twist the engine's next
// generation.
//
// Exactness: a site is drawn by Lemire's method on one engine word; the
// Metropolis decision for class k (old spin, neighbour sum) is either "dE < 0,
// accept without a draw" or "draw one word x and accept iff x < thr[k]", where
// thr[k] is the first word whose libstdc++ canonical double is >= exp(-dE*beta)
// (computed on the host with the same std::exp), so no exp and no
// int->double conversion happens per attempt.  The FP64 tails (running energy
// and the row/column formation-energy fold) use explicitly rounded operations.
#include <cstddef>

#include "internal.hh"
#include "walk.hh"

namespace mcg {

// Twist of the 312-word state by one wavefront.  Phase 1 (k < 156) reads only
// old words; phase 2 (k >= 156) reads old x[k], x[k+1] and new x[k-156], x[0].
// Within a phase all reads complete before any write.
__device__ void twist_wave(uint64_t *mt, int lane) {
  const int a0 = lane, a1 = lane + 64, a2 = lane + 128;
  uint64_t v0 = mt_twist_word(mt[a0], mt[a0 + 1], mt[a0 + MT_M]);
  uint64_t v1 = mt_twist_word(mt[a1], mt[a1 + 1], mt[a1 + MT_M]);
  uint64_t v2 = 0;
  if (a2 < MT_N - MT_M) v2 = mt_twist_word(mt[a2], mt[a2 + 1], mt[a2 + MT_M]);
  __syncthreads();
  mt[a0] = v0;
  mt[a1] = v1;
  if (a2 < MT_N - MT_M) mt[a2] = v2;
  __syncthreads();
  const int b0 = 156 + lane, b1 = 220 + lane, b2 = 284 + lane;
  v0 = mt_twist_word(mt[b0], mt[b0 + 1], mt[b0 - MT_M]);
  v1 = mt_twist_word(mt[b1], mt[b1 + 1], mt[b1 - MT_M]);
  if (b2 < MT_N) v2 = mt_twist_word(mt[b2], mt[b2 == MT_N - 1 ? 0 : b2 + 1], mt[b2 - MT_M]);
  __syncthreads();
  mt[b0] = v0;
  mt[b1] = v1;
  if (b2 < MT_N) mt[b2] = v2;
  __syncthreads();
}

template <bool LDS_LATTICE>
__global__ __launch_bounds__(64) void exact_kernel(const ExactParams *__restrict__ Pp,
                                                   ExactState *__restrict__ Sp,
                                                   int8_t *__restrict__ lat_pool,
                                                   mcg_sample *__restrict__ series,
                                                   int64_t series_cap,
                                                   const uint8_t *__restrict__ active,
                                                   int64_t n_passes, int64_t n_steps,
                                                   int64_t sample_period) {
  const int c = blockIdx.x;
  if (!active[c]) return;
  const int lane = threadIdx.x;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ uint64_t mt[MT_N];

  const ExactParams *P = Pp + c;
  ExactState *St = Sp + c;
  const int32_t rows = P->rows, cols = P->cols, n = P->n;
  // attempts of this launch: n_passes whole passes and n_steps more, from the
  // chain's position `step` in its current pass
  const int64_t total = n_passes * (int64_t)n + n_steps;
  if (!LDS_LATTICE && total >= P->block_from) return;  // exact_block_kernel's
  const uint64_t magic = P->div_magic;
  const uint32_t neg_mask = P->neg_mask, full_mask = P->full_mask;
  const int fold = P->fold;
  const int self_nb = P->self_nb;
  int8_t *g_lat = lat_pool + P->lat_off;
  const int lat_bytes_al = (n + 15) & ~15;
  int8_t *lat = LDS_LATTICE ? reinterpret_cast<int8_t *>(smem) : g_lat;
  int32_t *scratch = reinterpret_cast<int32_t *>(smem + (LDS_LATTICE ? lat_bytes_al : 0));

  for (int i = lane; i < MT_N; i += 64) mt[i] = St->mt[i];
  if (LDS_LATTICE)
    for (int i = lane; i < n; i += 64) lat[i] = g_lat[i];
  __syncthreads();

  int pos = (int)St->pos;
  int64_t n_pass = St->n_pass, n_acc = St->n_accept, n_rej = St->n_reject;
  int64_t S = St->S, M = St->M, n_samples = St->n_samples;
  double e_run = St->e_run;
  const uint64_t N64 = (uint64_t)n;

  auto next_word = [&]() -> uint64_t {
    if (pos >= MT_N) {
      twist_wave(mt, lane);
      pos = 0;
    }
    uint64_t w = rfl64(mt[pos]);
    ++pos;
    return mt_temper(w);
  };

  int32_t step = (int32_t)St->step;
  for (int64_t done = 0; done < total; ++done) {
    {
      // propose: l = uniform_int_distribution<long>(0, n-1) (Lemire)
      uint64_t x = next_word();
      uint64_t lo = x * N64;
      uint64_t hi = __umul64hi(x, N64);
      if (lo < N64) {
        const uint64_t t = (0ULL - N64) % N64;
        while (lo < t) {
          x = next_word();
          lo = x * N64;
          hi = __umul64hi(x, N64);
        }
      }
      const uint32_t l = (uint32_t)hi;
      const uint32_t j = (uint32_t)(((uint64_t)l * magic) >> 40);
      const uint32_t i = l - j * (uint32_t)rows;
      const uint32_t iu = (i + 1 == (uint32_t)rows) ? 0u : i + 1;
      const uint32_t id = (i == 0) ? (uint32_t)rows - 1 : i - 1;
      const uint32_t ju = (j + 1 == (uint32_t)cols) ? 0u : j + 1;
      const uint32_t jd = (j == 0) ? (uint32_t)cols - 1 : j - 1;
      const int s = rfl32(lat[l]);
      const int nsum = rfl32(lat[iu + rows * j] + lat[id + rows * j] + lat[i + rows * ju] +
                             lat[i + rows * jd]);
      const int k = (s > 0 ? 5 : 0) + ((nsum + 4) >> 1);
      bool acc;
      if ((neg_mask >> k) & 1u) {
        acc = true;
      } else {
        const uint64_t x2 = next_word();
        acc = ((full_mask >> k) & 1u) || (x2 < P->thr[k]);
      }
      if (acc) {
        if (lane == 0) lat[l] = (int8_t)(-s);
        if (!LDS_LATTICE) __threadfence();
        // the bond sum's self terms (a 1-wide lattice is its own neighbour) never
        // change; the reference's dE keeps them (model.hh:312-314), S does not
        S += -2LL * s * (nsum - self_nb * s);
        M += -2LL * s;
        e_run = __dadd_rn(e_run, P->dq[k]);
        ++n_acc;
      } else {
        ++n_rej;
      }
    }
    if (++step < n) continue;
    step = 0;
    ++n_pass;
    if (n_pass % sample_period == 0) {
      double ef = 0.0;
      if (fold) {
        __syncthreads();
        for (int r = lane; r < rows; r += 64) {
          const int ru = (r + 1 == rows) ? 0 : r + 1;
          int d = 0;
          for (int q = 0; q < cols; ++q) d += lat[r + rows * q] * lat[ru + rows * q];
          scratch[r] = d;
        }
        for (int q = lane; q < cols; q += 64) {
          const int qu = (q + 1 == cols) ? 0 : q + 1;
          int d = 0;
          for (int r = 0; r < rows; ++r) d += lat[r + rows * q] * lat[r + rows * qu];
          scratch[rows + q] = d;
        }
        __syncthreads();
        if (lane == 0) {
          // model.hh:276-285: sequential fold of fl(-J * dot) over rows, then columns
          double e = 0.0;
          for (int r = 0; r < rows + cols; ++r)
            e = __dadd_rn(e, __dmul_rn(P->negJ, (double)scratch[r]));
          ef = e;
        }
        __syncthreads();
      }
      if (lane == 0 && n_samples < series_cap) {
        mcg_sample rec = {};
        rec.pass = n_pass;
        rec.S1 = S;
        rec.S2 = 0;
        rec.M = M;
        rec.e_fold = ef;
        rec.e_run = e_run;
        series[(int64_t)c * series_cap + n_samples] = rec;
      }
      ++n_samples;
    }
  }

  __syncthreads();
  for (int i = lane; i < MT_N; i += 64) St->mt[i] = mt[i];
  if (LDS_LATTICE)
    for (int i = lane; i < n; i += 64) g_lat[i] = lat[i];
  if (lane == 0) {
    St->pos = pos;
    St->step = step;
    St->n_pass = n_pass;
    St->n_accept = n_acc;
    St->n_reject = n_rej;
    St->S = S;
    St->M = M;
    St->e_run = e_run;
    St->n_samples = n_samples;
  }
}

// ---------------------------------------------------------------------------
// Block-speculative walk (lattice classes in LDS).
//
// The stream is consumed in blocks of up to 64 positions.  For a block starting
// at stream position P, lane t evaluates position P+t as if it were a site
// draw, from the block-start lattice: the class k of its site, whether the
// attempt would draw a uniform (dE >= 0) and whether it would accept.  The real
// sequence follows in closed form: position t is an attempt; the next attempt
// is at t+1, or t+2 when t drew a uniform.  An attempt sees another lattice
// than the block-start one only when an earlier accepted attempt of the block
// flipped its site or one of its neighbours; the block stops before the first
// such attempt (it becomes lane 0 of the next block, on the updated lattice).
// Hence every attempt the block executes saw exactly the lattice the sequential
// chain would see.
//
// What bounds it is the latency of one dependent chain per wavefront (a
// dependent instruction costs 8 cycles, an LDS round trip 76 or more), so
// everything that does not depend on the lattice is moved off the walking wave:
//   waves 2-4 (walk_producer) twist the engine's next generation and turn each
//     of its words x into a 32-bit record: the site x would draw (Lemire), the
//     site's wrap flags, and for each of the 10 classes whether x accepts it
//     (one wave for all of it took 4500 cycles a generation and set the pace);
//   wave 1 (walk_energy) adds the accepted attempts' FP64 running energy in
//     attempt order and the integer observables, from the classes the walk
//     leaves in a ring of bytes, and writes the sample records;
//   wave 0 reads a position's record and the next one's, then one lattice
//     nibble: the lattice holds each site's class, 5 (s > 0) + up neighbours, in
//     four bits, so an attempt reads one nibble instead of five spins, and a
//     flip adds to five nibbles.  Sums of nibble changes are exact modulo 2^32
//     whatever order the adds of a block meet in.
// The waves meet at one workgroup barrier per engine generation (walk.hh).
//
// Conflicts: every position that would accept marks its site and the four
// neighbours with its lane (minimum) in a table of 32-bit entries indexed by
// site & mark_mask, while the scalar unit works out the attempt positions; an
// attempt whose own site holds a lower lane is a conflict.  A mark is
// 64 * epoch + lane with an epoch one lower in every block, so marks of earlier
// blocks are larger than any of this one and nothing is cleared.  Positions
// that turn out to be uniform draws, and sites that share an entry, only end a
// block early.  Marks of accepted lanes alone keep whole windows on small lattices
// too (marks of every attempt stopped a 25x25 block after ~2 attempts).
//
// Measured on MI355X, kernel time per attempt and chain at 2.4 GHz: 128x128, 64
// chains over 500-3000 K, 27 cycles (73 with one byte per site, the engine's raw
// words and the energy on the walking wave); one 25x25 chain 28 to 51 (826:
// marks of all attempts); 450x389 with the fold 26 (1260: the scalar walk on HBM).
// A block of 64 positions is ~100 instructions at 5 cycles or more each and two
// LDS round trips, most of them filled.
// ---------------------------------------------------------------------------
// A record: bits 2..19 the site (so the masked record is the bit address of
// the site's nibble), bits 20..29 accepted at class k, and the wrap flags of the
// neighbours site + 1 (bit 30), - 1 (31), + rows (0), - rows (1).  All four
// flags: the word needs Lemire's rejection test (a 1x1 lattice, where they
// would be the site's own, takes the scalar walk).
constexpr uint32_t REC_SITE = 0xFFFFCu;
constexpr int REC_ACC = 20, REC_UP = 30, REC_DN = 31, REC_RT = 0, REC_LF = 1;
constexpr uint32_t REC_SPECIAL = 0xC0000003u;
constexpr int EXACT_THREADS = 5 * 64;
constexpr uint32_t NO_MARK = 0xFFFFFFFFu;
constexpr uint32_t FIRST_EPOCH = 0x3FFFFFEu;  // 64 * it + 63 is below NO_MARK
// The block walk's fixed LDS parts, at LDS address 0 (the kernel has no static
// LDS); the conflict marks follow, then the lattice and the fold scratch.  The
// walk computes LDS byte addresses itself: the parts' offsets become immediates.
struct ExactWalkLds {
  uint32_t rec[REC_RING + REC_MIRROR];
  uint64_t raw[3][MT_N];
  double dq[EXACT_NCLASS];
  int32_t dS[EXACT_NCLASS], dM[EXACT_NCLASS];
  uint8_t fifo[FIFO];
  int done;
  uint32_t pub;
};
static_assert(sizeof(ExactWalkLds) <= EXACT_WALK_FIXED_LDS, "the marks start behind it");
// The record of engine word x.
__device__ __forceinline__ uint32_t exact_record(uint64_t x, const ExactParams *__restrict__ P,
                                                 uint32_t always) {
  const uint32_t rows = (uint32_t)P->rows, cols = (uint32_t)P->cols, n = (uint32_t)P->n;
  // x * n from two 32x32->64 products: site = high word, lo = low
  const uint64_t p0 = (uint64_t)(uint32_t)x * n;
  const uint64_t p1 = (uint64_t)(uint32_t)(x >> 32) * n + (p0 >> 32);
  const uint64_t lo = (p1 << 32) | (uint32_t)p0;
  const uint32_t site = (uint32_t)(p1 >> 32);
  const uint32_t j = (uint32_t)(((uint64_t)site * P->div_magic) >> 40);
  const uint32_t i = site - j * rows;
  uint32_t acc = always;
#pragma unroll
  for (int k = 0; k < EXACT_NCLASS; ++k) acc |= (x < P->thr[k] ? 1u : 0u) << k;
  uint32_t r = (site << 2) | (acc << REC_ACC);
  r |= (i + 1 == rows ? 1u : 0u) << REC_UP;
  r |= (i == 0 ? 1u : 0u) << REC_DN;
  r |= (j + 1 == cols ? 1u : 0u) << REC_RT;
  r |= (j == 0 ? 1u : 0u) << REC_LF;
  return lo < (uint64_t)n ? REC_SPECIAL | (acc << REC_ACC) : r;
}

__global__ __launch_bounds__(EXACT_THREADS) void exact_block_kernel(const ExactParams *__restrict__ Pp,
                                                         ExactState *__restrict__ Sp,
                                                         int8_t *__restrict__ lat_pool,
                                                         mcg_sample *__restrict__ series_pool,
                                                         int64_t series_cap,
                                                         const uint8_t *__restrict__ active,
                                                         int64_t n_passes, int64_t n_steps,
                                                         int64_t sample_period) {
  const int c = blockIdx.x;
  if (!active[c]) return;
  const int lane = threadIdx.x & 63;
  const int wave = rfl32(threadIdx.x >> 6);
  extern __shared__ __align__(16) unsigned char smem[];

  const ExactParams *P = Pp + c;
  ExactState *St = Sp + c;
  mcg_sample *series = series_pool + (int64_t)c * series_cap;
  const int32_t rows = P->rows, cols = P->cols, n = P->n;
  const int64_t total = n_passes * (int64_t)n + n_steps;
  if (total < P->block_from) return;  // exact_kernel's
  const uint64_t magic = P->div_magic;
  const uint32_t neg_mask = P->neg_mask, full_mask = P->full_mask, mmask = P->mark_mask;
  const uint32_t always = neg_mask | full_mask;
  const int fold = P->fold;
  int8_t *g_lat = lat_pool + P->lat_off;
  const int n_words = (n + 7) >> 3;
  ExactWalkLds &L = *reinterpret_cast<ExactWalkLds *>(smem);
  uint64_t(*raw)[MT_N] = L.raw;
  uint32_t *rec = L.rec;
  uint8_t *fifo = L.fifo;
  volatile lds_u32 *done = lds_at(offsetof(ExactWalkLds, done));
  volatile lds_u32 *pub = lds_at(offsetof(ExactWalkLds, pub));
  uint32_t *marks = reinterpret_cast<uint32_t *>(smem + EXACT_WALK_FIXED_LDS);
  const uint32_t lat_base = EXACT_WALK_FIXED_LDS + 4 * (mmask + 1);
  uint32_t *lat = reinterpret_cast<uint32_t *>(smem + lat_base);
  int32_t *scratch = reinterpret_cast<int32_t *>(lat + ((n_words + 3) & ~3));
  auto add_nibble = [&](uint32_t l, uint32_t v) { atomicAdd(&lat[l >> 3], v << ((l & 7u) * 4u)); };

  // spins first (5 per up site), then every up site adds one to the neighbours
  for (int w = threadIdx.x; w < n_words; w += EXACT_THREADS) {
    uint32_t v = 0;
    for (int e = 0; e < 8; ++e)
      if (8 * w + e < n && g_lat[8 * w + e] > 0) v |= 5u << (4 * e);
    lat[w] = v;
  }
  for (uint32_t i = threadIdx.x; i <= mmask; i += EXACT_THREADS) marks[i] = NO_MARK;
  for (int i = threadIdx.x; i < MT_N; i += EXACT_THREADS) {
    raw[0][i] = St->mt[i];
    rec[i] = exact_record(mt_temper(St->mt[i]), P, always);
  }
  if (threadIdx.x < EXACT_NCLASS) {
    // a flip of spin s with neighbour sum m changes S by -2 s (m - self_nb s): the
    // bond sum's self terms (a 1-wide lattice is its own neighbour) never change
    const int c = threadIdx.x, s = c >= 5 ? 1 : -1, m = 2 * (c % 5) - 4;
    L.dq[c] = P->dq[c];
    L.dS[c] = -2 * s * (m - P->self_nb * s);
    L.dM[c] = -2 * s;
  }
  if (threadIdx.x == 0) {
    *done = 0;
    *pub = 0;
  }
  const int64_t pos0 = St->pos;
  const int32_t step0 = (int32_t)St->step;
  __syncthreads();
  for (int l = threadIdx.x; l < n; l += EXACT_THREADS) {
    if (g_lat[l] <= 0) continue;
    const uint32_t j = (uint32_t)(((uint64_t)l * magic) >> 40);
    const uint32_t i = (uint32_t)l - j * (uint32_t)rows;
    add_nibble(((i + 1 == (uint32_t)rows) ? 0u : i + 1) + (uint32_t)rows * j, 1u);
    add_nibble(((i == 0) ? (uint32_t)rows - 1 : i - 1) + (uint32_t)rows * j, 1u);
    add_nibble(i + (uint32_t)rows * ((j + 1 == (uint32_t)cols) ? 0u : j + 1), 1u);
    add_nibble(i + (uint32_t)rows * ((j == 0) ? (uint32_t)cols - 1 : j - 1), 1u);
  }
  __syncthreads();
  if (wave >= 2) {
    walk_producer(raw, done, wave - 2, lane, [&](int slot, int k, uint64_t x, int) {
      const uint32_t r = exact_record(mt_temper(x), P, always);
      rec[slot * MT_N + k] = r;
      if (slot == 0) rec[REC_RING + k] = r;
    });
    return;
  }
  if (wave == 1) {
    walk_energy(St, series, series_cap, sample_period, total, fold, fifo, L.dq, L.dS, L.dM, pub,
                done, lane);
    return;
  }

  WalkRing ring{(int)pos0};
  uint32_t pushed = 0;  // entries written to fifo
  int64_t n_pass = St->n_pass, n_samples = St->n_samples;  // as wave 1 counts them (fold)
  int64_t remaining = total;
  int32_t step = step0;
  int seg = 0, left = 0;  // attempts up to the end of the pass or launch, and those to go
  auto ensure = [&](int upto) { ring.ensure(upto, pushed, pub, lane); };
  const uint32_t nd_mask = ~neg_mask, m4 = 4u * mmask;
  const uint32_t r_wrap = 4u * (uint32_t)rows, c_wrap = 4u * (uint32_t)rows * (uint32_t)cols;
  uint32_t my_mark = FIRST_EPOCH * 64u + (uint32_t)lane;
  uint32_t r0 = 0, r1 = 0;
  auto fetch = [&]() {
    r0 = rec[ring.rp + lane];
    r1 = rec[ring.rp + lane + 1];
  };
  // the end of the pass or of the launch (first: of nothing); false: all done
  auto segment_end = [&]() -> bool {
    step += seg;
    remaining -= seg;
    if (step == n) {
      step = 0;
      ++n_pass;
      if (lane == 0) fifo[pushed & (FIFO - 1)] = FIFO_PASS_END;
      ++pushed;
      if (fold && n_pass % sample_period == 0) {
        auto spin = [&](uint32_t l) { return ((lat[l >> 3] >> ((l & 7u) * 4u)) & 15u) >= 5u ? 1 : -1; };
        for (int r = lane; r < rows; r += 64) {
          const int ru = (r + 1 == rows) ? 0 : r + 1;
          int d = 0;
          for (int q = 0; q < cols; ++q) d += spin(r + rows * q) * spin(ru + rows * q);
          scratch[r] = d;
        }
        for (int q = lane; q < cols; q += 64) {
          const int qu = (q + 1 == cols) ? 0 : q + 1;
          int d = 0;
          for (int r = 0; r < rows; ++r) d += spin(r + rows * q) * spin(r + rows * qu);
          scratch[rows + q] = d;
        }
        asm volatile("" ::: "memory");
        if (lane == 0 && n_samples < series_cap) {
          double e = 0.0;  // model.hh:276-285
          for (int r = 0; r < rows + cols; ++r)
            e = __dadd_rn(e, __dmul_rn(P->negJ, (double)scratch[r]));
          series[n_samples].e_fold = e;
        }
        asm volatile("" ::: "memory");
        ++n_samples;
      }
    }
    seg = left = (int)(remaining < (int64_t)(n - step) ? remaining : (int64_t)(n - step));
    // a segment's blocks take at most one epoch per attempt
    if ((my_mark >> 6) <= (uint32_t)left) {
      for (uint32_t i = lane; i <= mmask; i += 64) marks[i] = NO_MARK;
      my_mark = FIRST_EPOCH * 64u + (uint32_t)lane;
      asm volatile("" ::: "memory");
    }
    return remaining > 0;
  };
  // one attempt with the full Lemire rejection loop, every lane alike
  auto special_attempt = [&]() {
    auto word_at = [&]() -> uint64_t {  // the engine word at pos, which is passed
      ensure(1);
      const uint64_t x = ring.word(raw);
      ++ring.rp;
      return x;
    };
    const uint64_t N64 = (uint64_t)n;
    uint64_t xs = word_at();
    const uint64_t th = (0ULL - N64) % N64;
    while (xs * N64 < th) xs = word_at();
    const uint32_t l = (uint32_t)__umul64hi(xs, N64);
    const uint32_t jj = (uint32_t)(((uint64_t)l * magic) >> 40);
    const uint32_t ii = l - jj * (uint32_t)rows;
    const uint32_t kk = (uint32_t)rfl32((int32_t)((lat[l >> 3] >> ((l & 7u) * 4u)) & 15u));
    bool a = true;
    if (!((neg_mask >> kk) & 1u)) {
      const uint64_t x2 = word_at();
      a = ((full_mask >> kk) & 1u) || (x2 < P->thr[kk]);
    }
    if (a) {
      if (lane == 0) {
        const bool up = kk >= 5;
        const uint32_t dn = up ? 0xFFFFFFFFu : 1u;
        add_nibble(l, up ? 0u - 5u : 5u);
        add_nibble(((ii + 1 == (uint32_t)rows) ? 0u : ii + 1) + (uint32_t)rows * jj, dn);
        add_nibble(((ii == 0) ? (uint32_t)rows - 1 : ii - 1) + (uint32_t)rows * jj, dn);
        add_nibble(ii + (uint32_t)rows * ((jj + 1 == (uint32_t)cols) ? 0u : jj + 1), dn);
        add_nibble(ii + (uint32_t)rows * ((jj == 0) ? (uint32_t)cols - 1 : jj - 1), dn);
        fifo[pushed & (FIFO - 1)] = (uint8_t)kk;
      }
      ++pushed;
    }
    asm volatile("" ::: "memory");
    --left;
  };
  auto specials = [&]() -> uint64_t { return __ballot((r0 & REC_SPECIAL) == REC_SPECIAL); };
  while (left > 0 || segment_end()) {
    ensure(65);
    fetch();
    uint64_t SP = specials();
    if (SP & 1ull) {
      special_attempt();
      continue;
    }
    // the blocks up to the end of the segment or of the readable positions
    for (;;) {
      // bit addresses of the site's nibble and (wrapped) of its neighbours', and
      // the mark entries, while the class arrives
      const uint32_t b0 = r0 & REC_SITE;
      const uint32_t w0 = nibble_word(b0, lat_base);
      const uint32_t word = *lds_at(w0);
      __builtin_amdgcn_sched_barrier(0);  // the read goes out before the rest
      auto flag = [&](int bit) { return (uint32_t)__builtin_amdgcn_sbfe((int)r0, bit, 1); };
      const uint32_t b1 = b0 + 4u - (flag(REC_UP) & r_wrap);
      const uint32_t b2 = b0 - 4u + (flag(REC_DN) & r_wrap);
      const uint32_t b3 = b0 + r_wrap - (flag(REC_RT) & c_wrap);
      const uint32_t b4 = b0 - r_wrap + (flag(REC_LF) & c_wrap);
      uint32_t m0 = b0 & m4, m1 = b1 & m4, m2 = b2 & m4, m3 = b3 & m4, mm4 = b4 & m4;
      uint32_t accs = r1 >> REC_ACC;
      my_mark -= 64u;
      asm volatile("" : "+v"(m0), "+v"(m1), "+v"(m2), "+v"(m3), "+v"(mm4), "+v"(accs));
      uint32_t k;
      asm("v_lshrrev_b32 %0, %1, %2" : "=v"(k) : "v"(b0), "v"(word));
      k &= 15u;
      const bool acc = (accs >> k) & 1u;
      const uint64_t AC = __ballot(acc);
      const uint64_t ND = __ballot((nd_mask >> k) & 1u) & ~SP;
      uint32_t mk = my_mark;
      if (AC) {
        if (acc) {
          lds_min(EXACT_WALK_FIXED_LDS + m0, my_mark);
          lds_min(EXACT_WALK_FIXED_LDS + m1, my_mark);
          lds_min(EXACT_WALK_FIXED_LDS + m2, my_mark);
          lds_min(EXACT_WALK_FIXED_LDS + m3, my_mark);
          lds_min(EXACT_WALK_FIXED_LDS + mm4, my_mark);
        }
        // the wave's LDS operations execute in issue order; the asm keeps the
        // compiler from moving the read above the marks
        asm volatile("" ::: "memory");
        mk = *lds_at(EXACT_WALK_FIXED_LDS + m0);
      }
      // the words of the neighbours' nibbles while the mark arrives
      uint32_t w1 = nibble_word(b1, lat_base), w2 = nibble_word(b2, lat_base);
      uint32_t w3 = nibble_word(b3, lat_base), w4 = nibble_word(b4, lat_base);
      const uint32_t up_v = k >= 5 ? 0xFFFFFFFFu : 1u;  // a neighbour's change
      uint32_t v0 = nibble_place(b0, k >= 5 ? 0u - 5u : 5u), v1 = nibble_place(b1, up_v);
      uint32_t v2 = nibble_place(b2, up_v), v3 = nibble_place(b3, up_v), v4 = nibble_place(b4, up_v);
      // Attempt positions of the window in closed form: position t is a uniform
      // draw iff t-1 is an attempt that draws (ND), so inside every run of ND bits
      // the attempts sit at even offsets from the run start.  E = attempts that
      // draw, E << 1 = uniform positions, attempts = the others.
      const uint64_t ALT = 0x5555555555555555ull;
      const uint64_t run_start = ND & ~(ND << 1);
      const uint64_t odd_runs = ND & ~(ND + (run_start & ~ALT));
      const uint64_t E = ND & (ALT ^ odd_runs);
      const uint64_t A = ~(E << 1);  // (bits above the window's first stop are not used)
      asm volatile("" : "+v"(mk), "+v"(w1), "+v"(w2), "+v"(w3), "+v"(w4), "+v"(v0), "+v"(v1),
                   "+v"(v2), "+v"(v3), "+v"(v4));
      const uint64_t STOP = SP | __ballot(mk < my_mark);
      // the block stops before its first conflict, else behind the window
      // (lane 0 is never one: its mark is the block's lowest, and not special)
      const uint64_t stops = A & STOP;
      uint64_t exec = A & (stops - 1) & ~stops;
      int t = (int)min((uint32_t)lowest_bit(stops), 64u + (uint32_t)(E >> 63));
      int attempts = __popcll(exec);
      if (attempts > left) {  // the pass or the launch ends inside the block
        uint64_t rest = exec;
        for (int r = 0; r < left; ++r) rest &= rest - 1;
        exec ^= rest;
        attempts = left;
        const int last = 63 - __builtin_clzll(exec);
        t = last + 1 + (int)((ND >> last) & 1ull);
      }
      const uint64_t F = exec & AC;
      ring.rp += t;
      left -= attempts;
      // the next block's records are read before this block's flips go out
      const bool more = ((ring.end - 65 - ring.rp) | (left - 1)) >= 0;
      if (more) fetch();
      asm volatile("" ::: "memory");
      if (__builtin_amdgcn_inverse_ballot_w64(F)) {
        lds_add(w0, v0);
        lds_add(w1, v1);
        lds_add(w2, v2);
        lds_add(w3, v3);
        lds_add(w4, v4);
        const uint32_t at = pushed + __builtin_amdgcn_mbcnt_hi((uint32_t)(F >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)F, 0u));
        lds_byte(offsetof(ExactWalkLds, fifo) + (at & (FIFO - 1)), k);
      }
      pushed += (uint32_t)__popcll(F);
      asm volatile("" ::: "memory");
      if (!more) break;
      SP = specials();
      if (SP & 1ull) break;
    }
  }

  // release the other waves: the final barrier's number goes into done
  if (lane == 0) {
    *pub = pushed;
    *done = (uint32_t)(ring.nbar + 1);
  }
  __syncthreads();
  // write back in the std::mt19937_64 layout: the generation holding the last
  // consumed output, with index in (0, 312]
  const int64_t pos = ring.position();
  int64_t g_fin = 0, p_fin = pos0;
  if (pos != pos0) {
    g_fin = (pos - 1) / MT_N;
    p_fin = pos - (int64_t)MT_N * g_fin;
  }
  for (int i = lane; i < MT_N; i += 64) St->mt[i] = raw[g_fin % 3][i];
  for (int w = lane; w < n_words; w += 64) {
    const uint32_t v = lat[w];
    for (int e = 0; e < 8; ++e)
      if (8 * w + e < n) g_lat[8 * w + e] = ((v >> (4 * e)) & 15u) >= 5u ? (int8_t)1 : (int8_t)-1;
  }
  if (lane == 0) {
    St->pos = p_fin;
    St->step = step;
  }
}

void launch_exact(const ExactParams *P, ExactState *S, int8_t *lat_pool, mcg_sample *series,
                  int64_t series_cap, const uint8_t *active, int n_chains, int64_t n_passes,
                  int64_t n_steps, int64_t sample_period, int lds_bytes, bool lattice_in_lds,
                  bool block_walk, hipStream_t stream) {
  if (lattice_in_lds && block_walk) {
    hipLaunchKernelGGL(exact_block_kernel, dim3(n_chains), dim3(EXACT_THREADS), lds_bytes, stream, P, S,
                       lat_pool, series, series_cap, active, n_passes, n_steps, sample_period);
  } else if (lattice_in_lds) {
    hipLaunchKernelGGL(exact_kernel<true>, dim3(n_chains), dim3(64), lds_bytes, stream, P, S,
                       lat_pool, series, series_cap, active, n_passes, n_steps, sample_period);
  } else {
    hipLaunchKernelGGL(exact_kernel<false>, dim3(n_chains), dim3(64), lds_bytes, stream, P, S,
                       lat_pool, series, series_cap, active, n_passes, n_steps, sample_period);
  }
}

// block_bytes, scalar_bytes: the most dynamic LDS a block walk and a scalar walk
// ask for.
hipError_t exact_set_max_lds(int block_bytes, int scalar_bytes) {
  hipError_t e =
      set_dynamic_lds(reinterpret_cast<const void *>(exact_block_kernel), block_bytes, true);
  if (e != hipSuccess) return e;
  e = hipFuncSetAttribute(reinterpret_cast<const void *>(exact_kernel<true>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, scalar_bytes);
  if (e != hipSuccess) return e;
  return hipFuncSetAttribute(reinterpret_cast<const void *>(exact_kernel<false>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, scalar_bytes);
}

}  // namespace mcg
