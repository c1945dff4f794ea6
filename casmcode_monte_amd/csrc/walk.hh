// walk.hh -- wavefront helpers shared by the sequential-chain kernels (EXACT
// single-site flips, canonical pair swaps, occupant events, KMC, N-fold way): scalar
// broadcasts, the out-of-place MT19937-64 twist, and the hand-offs by which other
// waves of the workgroup work beside the walking one: one that twists the engine into
// a ring of tempered outputs (the general OCCUPANT and KMC kernels), or three that
// twist it and leave a record per word, and one that adds energies and writes samples.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.hh"
#include "rng.hh"

namespace mcg {

// Two generations of tempered outputs: the walk reads stream positions
// [312(G-1), 312(G+1)) while generation G is the newest.
constexpr int RING = 2 * MT_N;

__device__ __forceinline__ uint64_t rfl64(uint64_t v) {
  uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ int32_t rfl32(int32_t v) {
  return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ double readlane_f64(double v, int lane) {
  uint64_t u = __double_as_longlong(v);
  uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, lane);
  uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), lane);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Out-of-place twist of generation src into dst; each new word k also goes to
// emit(k, x).  Lane L owns words L, L+64, L+128 (the first 156, which read only
// old words) and L+156, L+220, L+284 (the rest, each of which reads the new word
// 156 below it: one this lane computed).  Word 311 also reads the new word 0.
// All reads go out before any arithmetic, and since src and dst differ no write
// can disturb a read: one LDS round trip per generation.
// Column `col` (0, 1, 2) of it: words L + 64 col and L + 64 col + 156.
template <typename Emit>
__device__ __forceinline__ void mt_twist_column(const uint64_t *src, uint64_t *dst, int L,
                                                int col, Emit emit) {
  const int k = L + 64 * col;
  if (k >= MT_N - MT_M) return;  // column 2 has 28 lanes
  const bool wraps = k == MT_N - MT_M - 1;  // its second word is 311
  const uint64_t a = src[k], an = src[k + 1], b = src[k + MT_M];
  const uint64_t z0 = src[0], z1 = src[1], zm = src[MT_M];
  const uint64_t bn = wraps ? mt_twist_word(z0, z1, zm) : src[k + MT_M + 1];
  const uint64_t d = mt_twist_word(a, an, b), e = mt_twist_word(b, bn, d);
  dst[k] = d;
  emit(k, d);
  dst[k + MT_M] = e;
  emit(k + MT_M, e);
}

// All three columns by one wavefront, into a ring slot of tempered outputs.  The
// wave's LDS operations execute in issue order, so the caller's later reads see
// these writes.
__device__ __forceinline__ void twist_gen(const uint64_t *src, uint64_t *dst, uint64_t *slot, int L) {
  const bool third = L < MT_N - MT_M - 128;  // words L+128 and L+284 exist (L < 28)
  const bool wraps = L == MT_N - MT_M - 128 - 1;  // L+284 == 311
  const uint64_t a0 = src[L], a0n = src[L + 1], a1 = src[L + 64], a1n = src[L + 65];
  const uint64_t b0 = src[L + 156], b0n = src[L + 157], b1 = src[L + 220], b1n = src[L + 221];
  uint64_t a2 = 0, a2n = 0, b2 = 0, b2n = 0;
  if (third) {
    a2 = src[L + 128];
    a2n = src[L + 129];
    b2 = src[L + 284];
    if (!wraps) b2n = src[L + 285];
  }
  const uint64_t d0 = mt_twist_word(a0, a0n, b0);
  const uint64_t d1 = mt_twist_word(a1, a1n, b1);
  const uint64_t d2 = mt_twist_word(a2, a2n, b2);
  const uint64_t new0 = ((uint64_t)__builtin_amdgcn_readlane((uint32_t)(d0 >> 32), 0) << 32) |
                        (uint32_t)__builtin_amdgcn_readlane((uint32_t)d0, 0);
  const uint64_t e0 = mt_twist_word(b0, b0n, d0);
  const uint64_t e1 = mt_twist_word(b1, b1n, d1);
  const uint64_t e2 = mt_twist_word(b2, wraps ? new0 : b2n, d2);
  dst[L] = d0;
  dst[L + 64] = d1;
  dst[L + 156] = e0;
  dst[L + 220] = e1;
  slot[L] = mt_temper(d0);
  slot[L + 64] = mt_temper(d1);
  slot[L + 156] = mt_temper(e0);
  slot[L + 220] = mt_temper(e1);
  if (third) {
    dst[L + 128] = d2;
    dst[L + 284] = e2;
    slot[L + 128] = mt_temper(d2);
    slot[L + 284] = mt_temper(e2);
  }
  asm volatile("" ::: "memory");
}

// The engine's generations come from a second wavefront of the workgroup.
// raw[g % 3] holds generation g untempered and ring[g % 3] its tempered
// outputs.  The walk reads two generations at a time (G-1 and G, G the newest
// it has), so the producer can write generation G+1 into the third slot while
// the walk works.  The waves meet at one workgroup barrier per generation:
//   B_g: generation g+1 is in its slots; the walk passes it when its window
//   first needs generation g+1, the producer after writing it.
// The producer twists generation g right after B_{g-2}: by then the walk's
// window reaches into generation g-1, so its last consumed word lies in
// generation g-2 or later and the slots of generation g-3 are free.  Both waves
// count the barriers.  When the walk is done it writes the number its final
// barrier will have into `done` and passes that barrier, which is the one the
// producer waits at; the producer returns after the barrier whose number equals
// `done` (a read that races ahead of the final barrier sees a larger number and
// goes on to the final barrier).
__device__ inline void mt_producer(uint64_t (*raw)[MT_N], uint64_t (*ring)[MT_N],
                            volatile const int *done, int L) {
  int nbar = 0;
  for (int64_t g = 1;; ++g) {
    twist_gen(raw[(g - 1) % 3], raw[g % 3], ring[g % 3], L);
    __syncthreads();  // B_{g-1}
    if (*done == ++nbar) return;
  }
}

// The walking wave's side of the hand-off: G is the newest generation it may
// read (the slots hold G-1 and G), nbar the barriers passed.
struct MtRing3 {
  int64_t G = 0;
  int sG = 0;  // G % 3
  int nbar = 0;
  // make stream positions < upto readable
  __device__ __forceinline__ void ensure(int64_t upto) {
    while (upto > (int64_t)MT_N * (G + 1)) {
      __syncthreads();  // B_G: generation G+1 is in its slots
      ++nbar;
      ++G;
      sG = sG == 2 ? 0 : sG + 1;
    }
  }
  // offset of stream position q, 312(G-1) <= q < 312(G+1), in ring[3][MT_N]:
  // generation G sits in slot sG, generation G-1 in slot (sG + 2) % 3, so a
  // negative r lands at r + 312 sG except when sG = 0 (slot 2: r + 936); one
  // select, no branch
  __device__ __forceinline__ int index(int64_t q) const {
    const int r = (int)(q - (int64_t)MT_N * G);
    return r + MT_N * sG + ((r < 0 && sG == 0) ? 3 * MT_N : 0);
  }
  // the walk is done: release the producer (lane 0 writes the final barrier's
  // number; every lane of the walking wave passes the barrier)
  __device__ __forceinline__ void finish(int *done, int lane) {
    if (lane == 0) *done = nbar + 1;
    __syncthreads();
  }
};

// ---- LDS addressed by byte -------------------------------------------------------
// Kernels whose only LDS is one dynamic array (it starts at address 0; set_dynamic_lds
// refuses one with static LDS) compute byte addresses themselves: the offsets of their
// fixed parts become immediates.
using lds_u32 = __attribute__((address_space(3))) uint32_t;
__device__ __forceinline__ lds_u32 *lds_at(uint32_t byte) { return (lds_u32 *)(uintptr_t)byte; }
__device__ __forceinline__ void lds_add(uint32_t byte, uint32_t v) {
  __hip_atomic_fetch_add(lds_at(byte), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// nibbles: the LDS byte address of the word holding bit address b, and v moved
// to the nibble's place in it (a shift takes the low five bits of its amount by
// itself); one and two instructions, which the compiler does not find
__device__ __forceinline__ uint32_t nibble_word(uint32_t b, uint32_t base) {
  uint32_t w;
  asm("v_lshl_add_u32 %0, %1, 2, %2" : "=v"(w) : "v"(b >> 5), "s"(base));
  return w;
}
__device__ __forceinline__ uint32_t nibble_place(uint32_t b, uint32_t v) {
  uint32_t d;
  asm("v_lshlrev_b32 %0, %1, %2" : "=v"(d) : "v"(b), "v"(v));
  return d;
}
__device__ __forceinline__ void lds_byte(uint32_t byte, uint32_t v) {
  *(__attribute__((address_space(3))) uint8_t *)(uintptr_t)byte = (uint8_t)v;
}
// the lowest set bit's place, 0xFFFFFFFF if there is none
__device__ __forceinline__ uint32_t lowest_bit(uint64_t v) {
  uint32_t r;
  asm("s_ff1_i32_b64 %0, %1" : "=s"(r) : "s"(v));
  return r;
}
__device__ __forceinline__ void lds_min(uint32_t byte, uint32_t v) {
  __hip_atomic_fetch_min(lds_at(byte), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ---- accepted attempts and samples on a wave of their own --------------------------
// The walking wave leaves the classes of the accepted attempts, one byte each
// and in order, in a ring of bytes, and a marker per pass end; it publishes
// their count before each of its barriers.  At most 2 x 377 entries come between
// two barriers, and the adding wave is at most one generation (and 63 entries)
// behind.
constexpr int FIFO = 2048;
constexpr uint8_t FIFO_PASS_END = 0x80u;

__device__ __forceinline__ int64_t walk_sum(int64_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += (int64_t)__shfl_xor((long long)v, o, 64);
  return v;
}

// The adding wave: FP64 running energy in attempt order (class c adds dq[c]), the
// integer observables (dS[c], dM[c]), the sample records, and at the end the
// chain's counters.  Whole chunks of 64 entries are added as they come; the rest
// of a generation waits for more, or for the end.  fold: the walking wave writes
// the records' e_fold.  total: attempts of the launch.
__device__ inline void walk_energy(ExactState *St, mcg_sample *__restrict__ series,
                                   int64_t series_cap, int64_t sample_period, int64_t total,
                                   bool fold, const uint8_t *fifo, const double *dq,
                                   const int32_t *dS, const int32_t *dM,
                                   const volatile lds_u32 *pub, const volatile lds_u32 *done,
                                   int lane) {
  double e_run = St->e_run;
  int64_t S = St->S, M = St->M, n_pass = St->n_pass, n_samples = St->n_samples;
  int64_t n_acc = 0;
  int64_t accS = 0, accM = 0;  // this lane's share since the last reduction
  uint32_t head = 0;
  int nbar = 0;
  for (bool last = false; !last;) {
    __syncthreads();
    last = rfl32((int32_t)*done) == ++nbar;
    const uint32_t end = (uint32_t)rfl32((int32_t)*pub);
    asm volatile("" ::: "memory");  // the entries are read after the count
    while (end != head) {
      const uint32_t left = end - head;
      if (left < 64u && !last) break;
      const int m = left < 64u ? (int)left : 64;
      const uint32_t v = fifo[(head + lane) & (FIFO - 1)];
      const bool in = lane < m;
      const bool flip = in && v < FIFO_PASS_END;
      const int c = flip ? (int)v : 0;
      const double q = dq[c];
      const int s = flip ? dS[c] : 0, g = flip ? dM[c] : 0;
      uint64_t marks = __ballot(in && v == FIFO_PASS_END);
      if (m == 64 && !marks) {
#pragma unroll
        for (int j = 0; j < 64; ++j) e_run = __dadd_rn(e_run, readlane_f64(q, j));
        accS += s;
        accM += g;
        n_acc += 64;
      } else {
        for (int j = 0;;) {
          const int e = marks ? __builtin_ctzll(marks) : m;
          if (lane >= j && lane < e) {
            accS += s;
            accM += g;
          }
          n_acc += e - j;
          for (; j < e; ++j) e_run = __dadd_rn(e_run, readlane_f64(q, j));
          if (e == m) break;
          marks &= marks - 1;
          j = e + 1;
          if (++n_pass % sample_period != 0) continue;
          S += walk_sum(accS);
          M += walk_sum(accM);
          accS = accM = 0;
          if (lane == 0 && n_samples < series_cap) {
            mcg_sample *rec = series + n_samples;
            rec->pass = n_pass;
            rec->S1 = S;
            rec->S2 = 0;
            rec->M = M;
            if (!fold) rec->e_fold = 0.0;
            rec->e_run = e_run;
            rec->S3 = 0;
            rec->T3 = 0;
            rec->time = 0.0;
            rec->weight = 0.0;
          }
          ++n_samples;
        }
      }
      head += (uint32_t)m;
    }
  }
  S += walk_sum(accS);
  M += walk_sum(accM);
  if (lane == 0) {
    St->n_pass = n_pass;
    St->n_accept += n_acc;
    St->n_reject += total - n_acc;
    St->S = S;
    St->M = M;
    St->e_run = e_run;
    St->n_samples = n_samples;
  }
}

// A producing wave: its column of generation g into raw[g % 3], each word also to
// emit(slot, k, x, g), in step with the walk's barriers as mt_producer.
template <typename Emit>
__device__ __forceinline__ void walk_producer(uint64_t (*raw)[MT_N], const volatile lds_u32 *done,
                                              int col, int L, Emit emit) {
  int nbar = 0;
  int s = 0;  // (g - 1) % 3
  for (;;) {
    const int d = s == 2 ? 0 : s + 1;
    mt_twist_column(raw[s], raw[d], L, col, [&](int k, uint64_t x) { emit(d, k, x, nbar + 1); });
    s = d;
    __syncthreads();
    if ((int)*done == ++nbar) return;
  }
}

// The walking wave's place in a ring of three generations of per-word records
// (slot 0 once more behind the ring's end): rp the place of the next stream
// position (position % 936, or in the mirror), end that of the first position
// not readable yet.
constexpr int REC_RING = 3 * MT_N;
constexpr int REC_MIRROR = MT_N;
struct WalkRing {
  int rp, end = MT_N, nbar = 0;
  // `upto` positions from rp on readable; *pub gets the FIFO's count first
  __device__ __forceinline__ void ensure(int upto, uint32_t pushed, volatile lds_u32 *pub,
                                         int lane) {
    while (end - rp < upto) {
      if (lane == 0) *pub = pushed;
      __syncthreads();
      ++nbar;
      end += MT_N;
      if (rp >= REC_RING) {
        rp -= REC_RING;
        end -= REC_RING;
      }
    }
  }
  __device__ __forceinline__ int64_t position() const {
    return (int64_t)MT_N * (nbar + 1) - (end - rp);
  }
  // the raw engine word at rp, tempered
  __device__ __forceinline__ uint64_t word(const uint64_t (*raw)[MT_N]) const {
    const int slot = rp / MT_N;
    return mt_temper(rfl64(raw[slot % 3][rp - slot * MT_N]));
  }
};

// Starts of the attempts in a window of W stream words (bit t: an attempt
// starts at word t) when an attempt takes two words or, if it draws (bit t of
// ND), three: 0, then 2 or 3 words on, up to the first start in SX (excluded:
// the walk stops before it) or in SI (included: the walk stops after it).
// Starts keep their parity until one draws, so they are taken a segment at a
// time, one iteration per drawing attempt instead of one per attempt.
__device__ __forceinline__ uint64_t window_starts2(uint64_t ND, uint64_t SX, uint64_t SI, int W) {
  const uint64_t win = W >= 64 ? ~0ull : ((1ull << W) - 1ull);
  uint64_t A = 0;
  int t = 0;
  while (t < W) {
    const uint64_t res = (t & 1) ? 0xAAAAAAAAAAAAAAAAull : 0x5555555555555555ull;
    const uint64_t cand = res & (~0ull << t) & win;
    const uint64_t stop = cand & (SX | SI | ND);
    if (!stop) {
      A |= cand;
      break;
    }
    const int f = __builtin_ctzll(stop);
    const uint64_t below = (1ull << f) - 1ull;
    if ((SX >> f) & 1ull) {
      A |= cand & below;
      break;
    }
    A |= cand & (below | (1ull << f));
    if ((SI >> f) & 1ull) break;
    t = f + 3;
  }
  return A;
}

// All starts of a window of 64 when an attempt takes WORDS words (two or three) or,
// if it draws (nd), one more.  Word t maps the words left to the next start (0 to
// WORDS; one byte each) to those left after it, and a prefix composition of the 64 maps -- a byte
// permutation a step -- gives every word's, whatever draws: ~25 instructions, where
// window_starts2 takes ~12 for each attempt that draws.  A step's lanes without a
// partner keep what `far` held before: the identity, in a register per step.
template <int WORDS>
struct WindowStarts {
  static constexpr int ID = 0x03020100;
  int far[6] = {ID, ID, ID, ID, ID, ID};
  template <int CTRL, int ROWS>
  __device__ __forceinline__ int step(int f, int s) {
    far[s] = __builtin_amdgcn_update_dpp(far[s], f, CTRL, ROWS, 0xf, false);
    return (int)__builtin_amdgcn_perm((uint32_t)f, (uint32_t)f, (uint32_t)far[s]);
  }
  __device__ __forceinline__ uint64_t operator()(bool nd) {
    int f = nd ? 0x02010000 + WORDS : 0x02010000 + WORDS - 1;
    f = step<0x111, 0xf>(f, 0);  // row_shr 1, 2, 4, 8
    f = step<0x112, 0xf>(f, 1);
    f = step<0x114, 0xf>(f, 2);
    f = step<0x118, 0xf>(f, 3);
    f = step<0x142, 0xa>(f, 4);  // row_bcast 15, 31
    f = step<0x143, 0xc>(f, 5);
    return (__ballot((f & 3) == 0) << 1) | 1ull;
  }
};

}  // namespace mcg
