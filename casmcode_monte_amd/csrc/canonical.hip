// canonical.hip -- CANONICAL mode: the reference's canonical pair-swap chain
// (Kawasaki exchanges between any two sites of different species), reproduced
// bit for bit by one walking wavefront per chain; the workgroup's other waves do
// what does not depend on the chain's state (walk.hh).
//
// Reference: the generic loop of occupation_metropolis.hh:87-153 with
// propose_canonical_event (OccEventProposal.hh:109-236) over an OccLocation
// (OccLocation.hh:254-259 choose_mol; OccLocation.cc:216-283 apply) and
// metropolis_acceptance (metropolis.hh:25-35), on a binary lattice with one
// asymmetric unit: species 0 = spin -1, species 1 = spin +1, one canonical
// swap type ((0,0),(0,1)).  The potential is the square-lattice Ising
// formation energy with the multi-site delta of model.hh:354-379.
//
// Per step the reference draws: one word for the swap-type choice (with a
// single swap type it always picks it), one Lemire word for the position in
// the species-0 list (site a), one for the species-1 list (site b), and one
// more only when dE >= 0.  dE depends on (Sa, Sb'): the neighbour sum of a
// before the swap and of b after a has flipped, so the acceptance is a per-class
// word threshold as in the EXACT mode.
//
// Device OccLocation: the two candidate lists as 16-bit site indices in LDS
// (species 0 at [0, nA), species 1 at [nA, n)); Mol ids equal site indices
// because every site mutates.  An accepted swap (a at list-0 slot ia, b at
// list-1 slot ib) leaves list0[ia] = old list0[nA-1], list0[nA-1] = b and
// list1[ib] = a, which is what the reference's remove-by-swap-with-back then
// push_back sequence gives.
//
// Both list sizes are fixed, so waves 2-4 turn each engine word into a record:
// the slot it gives in either list and the swap classes it accepts.  A site's
// class is a byte, 5 (species) + up neighbours, so a step reads two list entries,
// two bytes and one record, and an accepted one adds to ten bytes.  Wave 1 adds
// energies and bond sums in step order and writes the samples (walk_energy).
//
// Block-speculative walk: lane t evaluates stream position P+t as if a step
// started there, from the block-start state.  Steps take 3 or 4 words; the real
// starts follow from the "draws a uniform" ballot (WindowStarts).  Positions that
// would accept mark the ten sites whose bytes they change, and the species-0
// list's last entry (a hash of 4-byte entries, 64 * epoch + lane as in exact.hip);
// the block stops before the first step whose own two sites hold a lower lane.
// Only earlier accepted steps can flag a step, so all steps before the first
// flagged one saw the sequential chain's state.
//
// Measured on MI355X, 64 chains of 128x128 sites at 8 T x 8 compositions, 327680
// steps each: 34.3 ms by a walk that read ten sites' spins a step and added energies
// itself, 15.2 ms so (70 cycles a step of the coldest chain at 2.4 GHz, 113 of the one
// that accepts 43 %): ~255 instructions a block of up to 18 steps, which one wave
// issues in ~5 cycles each.  1024 chains of 64x64, 10 passes: 9.0 and 4.1 ms; one of
// 150x150, 4 passes: 8.0 and 3.3 ms.
#include <cstddef>

#include "internal.hh"
#include "walk.hh"

namespace mcg {

namespace {

constexpr int CANON_THREADS = 5 * 64;
constexpr uint32_t NO_MARK = 0xFFFFFFFFu;
constexpr uint32_t FIRST_EPOCH = NO_MARK / 64u - 1u;
// a class's index in masks and tables: 5 (byte of a) + (byte of b) + links, where
// b's byte holds its species' 5
constexpr int CLASS0 = 5;

// fixed LDS parts at address 0; the lists, the class bytes, the marks and the fold
// scratch follow
struct CanonWalkLds {
  uint32_t slots[REC_RING + REC_MIRROR];  // the word's entry for a; for b << 16
  uint32_t acc[REC_RING + REC_MIRROR];    // accepted classes, bit CLASS0 + class
  uint64_t raw[3][MT_N];
  double dq[32];
  int32_t dS[32], dM[32];
  uint8_t fifo[FIFO];
  uint32_t bs[64];  // a block's accepted steps' b, in order
  uint32_t done, pub;
  int32_t rejecting;  // the newest generation with a word that a Lemire draw may reject
};
static_assert(sizeof(CanonWalkLds) <= CANON_FIXED_LDS, "the lists start behind it");
static_assert(CLASS0 + CANON_NCLASS <= 32, "a class's bit");

}  // namespace

__global__ __launch_bounds__(CANON_THREADS) void canonical_kernel(
    const CanonParams *__restrict__ Pp, ExactState *__restrict__ Sp,
    int8_t *__restrict__ lat_pool, int32_t *__restrict__ list_pool,
    mcg_sample *__restrict__ series_pool, int64_t series_cap,
    const uint8_t *__restrict__ active, int64_t n_passes, int64_t sample_period) {
  const int c = blockIdx.x;
  if (!active[c]) return;
  const int lane = threadIdx.x & 63;
  const int wave = rfl32(threadIdx.x >> 6);
  extern __shared__ __align__(16) unsigned char smem[];

  const CanonParams *P = Pp + c;
  ExactState *St = Sp + c;
  mcg_sample *series = series_pool + (int64_t)c * series_cap;
  const uint32_t rows = (uint32_t)P->rows, cols = (uint32_t)P->cols, n = (uint32_t)P->n;
  const uint32_t nA = (uint32_t)P->nA, nB = (uint32_t)P->nB, mmask = P->mark_mask;
  const int fold = P->fold;
  const bool scalar = P->window == 1;
  int8_t *g_lat = lat_pool + P->lat_off;
  int32_t *g_list = list_pool + P->lat_off;
  CanonWalkLds &L = *reinterpret_cast<CanonWalkLds *>(smem);
  volatile lds_u32 *done = lds_at(offsetof(CanonWalkLds, done));
  volatile lds_u32 *pub = lds_at(offsetof(CanonWalkLds, pub));
  volatile lds_u32 *rejecting = lds_at(offsetof(CanonWalkLds, rejecting));
  const uint32_t cls_base = CANON_FIXED_LDS + ((2u * n + 15u) & ~15u);
  const uint32_t mark_base = cls_base + ((n + 15u) & ~15u);
  uint16_t *list = reinterpret_cast<uint16_t *>(smem + CANON_FIXED_LDS);
  uint8_t *cls = smem + cls_base;
  uint32_t *marks = reinterpret_cast<uint32_t *>(smem + mark_base);
  int32_t *scratch = reinterpret_cast<int32_t *>(smem + mark_base + 4u * (mmask + 1u));

  const uint32_t nd_mask = (~P->neg_mask & ((1u << CANON_NCLASS) - 1u)) << CLASS0;
  const uint32_t always = (P->neg_mask | P->full_mask) << CLASS0;
  // one word's record in generation g (slot: its place in the ring)
  auto put = [&](int slot, int k, uint64_t raw_word, int g) {
    const uint64_t x = mt_temper(raw_word);
    const uint32_t s = (uint32_t)__umul64hi(x, (uint64_t)nA) |
                       ((nA + (uint32_t)__umul64hi(x, (uint64_t)nB)) << 16);
    uint32_t acc = always;
#pragma unroll
    for (int e = 0; e < CANON_NCLASS; ++e) acc |= (x < P->thr[e] ? 1u : 0u) << (CLASS0 + e);
    if (x * nA < nA || x * nB < nB) *rejecting = (uint32_t)g;
    L.slots[slot * MT_N + k] = s;
    L.acc[slot * MT_N + k] = acc;
    if (slot == 0) {
      L.slots[REC_RING + k] = s;
      L.acc[REC_RING + k] = acc;
    }
  };
  // floor(l / rows): 2 l * 2 rows < 2^32 for the lattices that fit
  const uint32_t magic = (uint32_t)(((1ull << 32) + 2u * rows - 1u) / (2u * rows));
  // a site's four neighbours, as sites' byte addresses
  const uint32_t row_wrap = rows, col_wrap = rows * cols;
  auto neighbours = [&](uint32_t l, uint32_t (&x)[4]) __attribute__((always_inline)) {
    const uint32_t j = __umulhi(2u * l, magic), i = l - j * rows, at = l + cls_base;
    x[0] = at + (i == rows - 1u ? 1u - row_wrap : 1u);
    x[1] = at + (i == 0u ? row_wrap - 1u : 0u - 1u);
    x[2] = at + (j == cols - 1u ? rows - col_wrap : rows);
    x[3] = at + (j == 0u ? col_wrap - rows : 0u - rows);
  };
  auto add_byte = [&](uint32_t at, uint32_t v) __attribute__((always_inline)) {
    lds_add(at & ~3u, v << ((at & 3u) * 8u));
  };

  // classes without neighbours first, then every up site adds one to the four
  for (uint32_t i = threadIdx.x; i < ((n + 15u) & ~15u); i += CANON_THREADS)
    cls[i] = i < n && g_lat[i] > 0 ? 5 : 0;
  for (uint32_t i = threadIdx.x; i < n; i += CANON_THREADS) list[i] = (uint16_t)g_list[i];
  for (uint32_t i = threadIdx.x; i <= mmask; i += CANON_THREADS) marks[i] = NO_MARK;
  if (threadIdx.x == 0) {
    *done = 0;
    *pub = 0;
    *rejecting = (uint32_t)-4;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < MT_N; i += CANON_THREADS) {
    L.raw[0][i] = St->mt[i];
    put(0, (int)i, St->mt[i], 0);
  }
  if (threadIdx.x < CANON_NCLASS) {
    const int k = threadIdx.x;
    L.dq[CLASS0 + k] = P->dq[k];
    L.dS[CLASS0 + k] = 4 * (k / 5 - k % 5) + 4 * P->self_nb;  // 2 (Sa - Sb) + 4 self_nb
    L.dM[CLASS0 + k] = 0;
  }
  for (uint32_t l = threadIdx.x; l < n; l += CANON_THREADS) {
    if (g_lat[l] <= 0) continue;
    uint32_t x[4];
    neighbours(l, x);
    for (int e = 0; e < 4; ++e) add_byte(x[e], 1u);
  }
  __syncthreads();
  const int64_t total = n_passes * (int64_t)n;
  if (wave >= 2) {
    walk_producer(L.raw, done, wave - 2, lane, put);
    return;
  }
  if (wave == 1) {
    walk_energy(St, series, series_cap, sample_period, total, fold, L.fifo, L.dq, L.dS, L.dM, pub,
                done, lane);
    return;
  }

  const int64_t pos0 = St->pos;
  WalkRing ring{(int)pos0};
  uint32_t pushed = 0;
  int64_t n_pass = St->n_pass, n_samples = St->n_samples;  // as wave 1 counts them (fold)
  int64_t passes = -1;
  int left = 0;  // steps up to the end of the pass
  uint32_t back0 = (uint32_t)rfl32((int32_t)list[nA - 1u]);  // the species-0 list's last entry
  const uint32_t back_at = CANON_FIXED_LDS + 2u * (nA - 1u);
  uint32_t my_mark = FIRST_EPOCH * 64u + (uint32_t)lane;
  auto ensure = [&](int upto) { ring.ensure(upto, pushed, pub, lane); };
  auto put_list = [&](uint32_t at, uint32_t l) __attribute__((always_inline)) {
    *(volatile __attribute__((address_space(3))) uint16_t *)(uintptr_t)at = (uint16_t)l;
  };
  auto push = [&](uint32_t rank, uint32_t v) __attribute__((always_inline)) {
    lds_byte(offsetof(CanonWalkLds, fifo) + ((pushed + rank) & (FIFO - 1)), v);
  };
  // the end of a pass (first: of nothing); false: all done
  auto pass_end = [&]() -> bool {
    if (++passes > 0) {
      if (lane == 0) push(0, FIFO_PASS_END);
      ++pushed;
      ++n_pass;
      if (fold && n_pass % sample_period == 0) {
        auto spin = [&](uint32_t l) { return cls[l] >= 5 ? 1 : -1; };
        for (uint32_t r = lane; r < rows; r += 64) {
          const uint32_t ru = r + 1 == rows ? 0 : r + 1;
          int d = 0;
          for (uint32_t q = 0; q < cols; ++q) d += spin(r + rows * q) * spin(ru + rows * q);
          scratch[r] = d;
        }
        for (uint32_t q = lane; q < cols; q += 64) {
          const uint32_t qu = q + 1 == cols ? 0 : q + 1;
          int d = 0;
          for (uint32_t r = 0; r < rows; ++r) d += spin(r + rows * q) * spin(r + rows * qu);
          scratch[rows + q] = d;
        }
        asm volatile("" ::: "memory");
        if (lane == 0 && n_samples < series_cap) {
          double e = 0.0;  // model.hh:276-285
          for (uint32_t r = 0; r < rows + cols; ++r)
            e = __dadd_rn(e, __dmul_rn(P->negJ, (double)scratch[r]));
          series[n_samples].e_fold = e;
        }
        asm volatile("" ::: "memory");
        ++n_samples;
      }
    }
    left = (int)n;
    if ((my_mark >> 6) <= n) {  // a block takes at most one epoch
      for (uint32_t i = lane; i <= mmask; i += 64) marks[i] = NO_MARK;
      my_mark = FIRST_EPOCH * 64u + (uint32_t)lane;
      asm volatile("" ::: "memory");
    }
    return passes < n_passes;
  };
  // an accepted step's bytes, by the calling lane: a and b with their neighbours
  auto apply = [&](uint32_t a, uint32_t b, const uint32_t (&xa)[4], const uint32_t (&xb)[4])
      __attribute__((always_inline)) {
    add_byte(a + cls_base, 5u);
    add_byte(b + cls_base, 0u - 5u);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      add_byte(xa[e], 1u);
      add_byte(xb[e], 0u - 1u);
    }
  };
  auto links = [&](uint32_t a, const uint32_t (&xb)[4]) __attribute__((always_inline)) {
    const uint32_t at = a + cls_base;
    return (xb[0] == at) + (xb[1] == at) + (xb[2] == at) + (xb[3] == at);
  };
  // one step with the full Lemire rejection loops, every lane alike
  auto scalar_step = [&]() {
    auto next_word = [&]() -> uint64_t {
      ensure(1);
      const uint64_t x = ring.word(L.raw);
      ++ring.rp;
      return x;
    };
    auto slot_of = [&](uint64_t m) -> uint32_t {
      uint64_t x = next_word();
      if (x * m < m) {
        const uint64_t th = (0ULL - m) % m;
        while (x * m < th) x = next_word();
      }
      return (uint32_t)__umul64hi(x, m);
    };
    next_word();  // the swap type
    const uint32_t pa = CANON_FIXED_LDS + 2u * slot_of(nA);
    const uint32_t pb = CANON_FIXED_LDS + 2u * (nA + slot_of(nB));
    const uint32_t a = list[(pa - CANON_FIXED_LDS) >> 1], b = list[(pb - CANON_FIXED_LDS) >> 1];
    uint32_t xa[4], xb[4];
    neighbours(a, xa);
    neighbours(b, xb);
    const uint32_t k = (uint32_t)rfl32((int32_t)(5u * cls[a] + cls[b] + links(a, xb)));
    bool ok = true;
    if ((nd_mask >> k) & 1u)
      ok = next_word() < P->thr[k - CLASS0] || ((always >> k) & 1u);
    asm volatile("" ::: "memory");
    if (ok) {
      if (lane == 0) {
        apply(a, b, xa, xb);
        put_list(pa, back0);
        put_list(pb, a);
        put_list(back_at, b);
        push(0, k);
      }
      ++pushed;
      back0 = (uint32_t)rfl32((int32_t)b);
    }
    asm volatile("" ::: "memory");
    --left;
  };
  auto bits_below = [&](uint64_t m) __attribute__((always_inline)) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  };

  WindowStarts<3> starts;
  uint32_t sa = 0, sb = 0, acc = 0;
  auto fetch = [&]() __attribute__((always_inline)) {
    sa = L.slots[ring.rp + lane + 1];
    sb = L.slots[ring.rp + lane + 2];
    acc = L.acc[ring.rp + lane + 3];
  };
  while (left > 0 || pass_end()) {
    ensure(67);
    // the newest two generations hold every word from here on
    if (scalar || rfl32((int32_t)*rejecting) + 2 > ring.nbar) {
      scalar_step();
      continue;
    }
    fetch();
    for (;;) {
      const uint32_t pa = CANON_FIXED_LDS + 2u * (sa & 0xFFFFu);
      const uint32_t pb = CANON_FIXED_LDS + 2u * (sb >> 16);
      const uint32_t a = *(const __attribute__((address_space(3))) uint16_t *)(uintptr_t)pa;
      const uint32_t b = *(const __attribute__((address_space(3))) uint16_t *)(uintptr_t)pb;
      const uint32_t ca = cls[a], cb = cls[b];
      __builtin_amdgcn_sched_barrier(0);
      uint32_t xa[4], xb[4];
      neighbours(b, xb);
      uint32_t k = links(a, xb);
      neighbours(a, xa);
      asm volatile(""
                   : "+v"(xa[0]), "+v"(xa[1]), "+v"(xa[2]), "+v"(xa[3]), "+v"(xb[0]), "+v"(xb[1]),
                     "+v"(xb[2]), "+v"(xb[3]), "+v"(k));
      k += 5u * ca + cb;
      const uint32_t kbit = 1u << k;
      const uint64_t AC = __ballot((acc & kbit) != 0u);
      const uint64_t ND = __ballot((nd_mask & kbit) != 0u);
      uint64_t exec = starts(__builtin_amdgcn_inverse_ballot_w64(ND));
      uint64_t F = exec & AC;
      if (F) {
        auto mark_of = [&](uint32_t at) __attribute__((always_inline)) {
          return mark_base + 4u * (at & mmask);  // (of a site's byte address)
        };
        const uint32_t ma = mark_of(a + cls_base), mb = mark_of(b + cls_base);
        if (__builtin_amdgcn_inverse_ballot_w64(F)) {
          lds_min(ma, my_mark);
          lds_min(mb, my_mark);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            lds_min(mark_of(xa[e]), my_mark);
            lds_min(mark_of(xb[e]), my_mark);
          }
          // for the steps of the list's last entry (an address that the compiler
          // does not know to be one: it would reduce the values first)
          uint32_t m0 = mark_of(back0 + cls_base);
          asm("" : "+v"(m0));
          lds_min(m0, my_mark);
        }
        asm volatile("" ::: "memory");
        const uint32_t m0 = *lds_at(ma), m1 = *lds_at(mb);
        asm volatile("" ::: "memory");
        const uint64_t HIT = exec & __ballot((m0 < m1 ? m0 : m1) < my_mark);
        if (HIT) {
          exec &= (HIT & (0ull - HIT)) - 1ull;
          F &= exec;
        }
        my_mark -= 64u;
      }
      int steps = __popcll(exec);
      if (__builtin_expect(steps >= left, 0)) {  // up to the pass's last step
        uint64_t rest = exec;
        for (int r = 0; r < left; ++r) rest &= rest - 1;
        exec ^= rest;
        F &= exec;
        steps = left;
      }
      const int last = 63 - __builtin_clzll(exec);
      ring.rp += last + 3 + (int)((ND >> last) & 1ull);
      left -= steps;
      const bool more = ((ring.end - 67 - ring.rp) | (left - 1)) >= 0;
      if (more) fetch();
      asm volatile("" ::: "memory");
      if (F) {
        const int lf = 63 - __builtin_clzll(F);
        if (__builtin_amdgcn_inverse_ballot_w64(F)) {
          const uint32_t rank = bits_below(F);
          constexpr uint32_t BS = offsetof(CanonWalkLds, bs);
          *(volatile lds_u32 *)lds_at(BS + 4u * rank) = b;
          uint32_t back = *(volatile lds_u32 *)lds_at(BS + 4u * (rank ? rank - 1u : 0u));
          push(rank, k);
          apply(a, b, xa, xb);
          put_list(pb, a);
          back = rank ? back : back0;
          put_list(pa, back);
          if (lane == lf) put_list(back_at, b);
        }
        back0 = (uint32_t)__builtin_amdgcn_readlane((int)b, lf);
        pushed += (uint32_t)__popcll(F);
      }
      asm volatile("" ::: "memory");
      if (!more) break;
    }
  }

  // release the other waves
  if (lane == 0) {
    *pub = pushed;
    *done = (uint32_t)(ring.nbar + 1);
  }
  __syncthreads();
  const int64_t pos = ring.position();
  int64_t g_fin = 0, p_fin = pos0;
  if (pos != pos0) {
    g_fin = (pos - 1) / MT_N;
    p_fin = pos - (int64_t)MT_N * g_fin;
  }
  for (int i = lane; i < MT_N; i += 64) St->mt[i] = L.raw[g_fin % 3][i];
  for (uint32_t i = lane; i < n; i += 64) {
    g_lat[i] = cls[i] >= 5 ? (int8_t)1 : (int8_t)-1;
    g_list[i] = (int32_t)list[i];
  }
  if (lane == 0) St->pos = p_fin;
}

void launch_canonical(const CanonParams *P, ExactState *S, int8_t *lat_pool, int32_t *list_pool,
                      mcg_sample *series, int64_t series_cap, const uint8_t *active,
                      int n_chains, int64_t n_passes, int64_t sample_period, int lds_bytes,
                      hipStream_t stream) {
  hipLaunchKernelGGL(canonical_kernel, dim3(n_chains), dim3(CANON_THREADS), lds_bytes, stream, P,
                     S, lat_pool, list_pool, series, series_cap, active, n_passes, sample_period);
}

hipError_t canonical_set_max_lds(int bytes) {
  return set_dynamic_lds(reinterpret_cast<const void *>(canonical_kernel), bytes, true);
}

}  // namespace mcg
