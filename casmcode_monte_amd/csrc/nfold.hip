// nfold.hip -- NFOLD mode: the N-fold way (rejection-free kinetic Monte Carlo)
// for the SGC square-lattice Ising model, one sequential chain per wavefront.
//
// Reference: the main loop of nfold.hh:78-149 (select an event and its time
// increment, sample by count with the increment as weight or on the time grid,
// apply, advance time, count a step).  The event selector is defined here:
// a site's rate is its Metropolis probability for the SGC potential delta of
// its class k = (s > 0) * 5 + (nbr_sum + 4) / 2 (the EXACT mode's classes,
// basic_semigrand_canonical.hh:178-192, model.hh:305-345); sites are kept in
// one array partitioned by class, class k at [start[k], start[k+1]).  Per
// event: R = sum_k n_k r_k in class order; the class is the first whose
// running sum exceeds u1 * R; the site is arr[start[k] + p] with p a Lemire
// draw over n_k; dt = -log1p(-u3) / R.  After the flip the site and its four
// neighbours (+i, -i, +j, -j, in that order) move to their new classes: down
// a class by swapping with the first entry of the segment left, up by
// swapping with the last.
//
// Layout: workgroup = one 64-lane wavefront = one chain.  LDS holds the class
// array and each site's position in it (16-bit each; bit 15 of a position is
// the site's spin, which its class also fixes: 4 bytes a site, so two 128x128
// chains share a CU) and the MT19937-64 ring.  The segment starts live in
// registers (lane k holds start[k]); the rates likewise (lane k, k < 10).
// The walk is sequential, and the latency of one event's dependent chain bounds
// it (5 cycles or more an instruction, ~76 an LDS round trip), so an event is
// three round trips and few instructions (select, apply_event):
//   the class: running rate sums by ten lane shifts, one ballot;
//   round trip 1: the site's entry together with the entries at the five segment
//     boundaries its move crosses (its class fixes them);
//   round trip 2: the four neighbours' positions and spins and their
//     neighbours' spins, one entry in each of 20 lanes, counted from one ballot;
//   round trip 3: the boundary entries the four neighbours swap with.
// The neighbours of a flipped site all cross one boundary in the same direction
// as the site, so their swaps are read and written together; the rare event
// whose swaps touch each other's entries is put in order in registers.  Lattices
// 1 or 2 wide, where a neighbour can be listed twice, and an event left pending
// by another launch take the general moves one by one (apply).
// Measured on MI355X, 64 chains of 128x128 over 500-3000 K: 1490 to 1640 cycles an
// event at 2.4 GHz (4400 with the moves one by one, each a round trip, and the
// sums by lane reads); the next event's words read ahead of the moves: 2% slower.
#include <type_traits>

#include "internal.hh"
#include "walk.hh"

// every lambda below is inlined: a call would put the walk's state into memory
#define MCG_INLINE __attribute__((always_inline))

namespace mcg {

namespace {

// pos[l] holds l's position in the class array (bits 0..14) and its spin
// (bit 15: 1 = +1)
constexpr uint16_t SPIN_BIT = 0x8000u;
__device__ __forceinline__ int spin_at(const uint16_t *pos, uint32_t l) {
  return (pos[l] & SPIN_BIT) ? 1 : -1;
}

__device__ __forceinline__ void nbrs(uint32_t l, int32_t rows, int32_t cols, uint64_t magic,
                                     uint32_t out[4]) {
  const uint32_t j = (uint32_t)(((uint64_t)l * magic) >> 40);
  const uint32_t i = l - j * (uint32_t)rows;
  const uint32_t iu = (i + 1 == (uint32_t)rows) ? 0u : i + 1;
  const uint32_t id = (i == 0) ? (uint32_t)rows - 1 : i - 1;
  const uint32_t ju = (j + 1 == (uint32_t)cols) ? 0u : j + 1;
  const uint32_t jd = (j == 0) ? (uint32_t)cols - 1 : j - 1;
  out[0] = iu + (uint32_t)rows * j;
  out[1] = id + (uint32_t)rows * j;
  out[2] = i + (uint32_t)rows * ju;
  out[3] = i + (uint32_t)rows * jd;
}

__device__ __forceinline__ int class_of(const uint16_t *pos, uint32_t l, int32_t rows,
                                        int32_t cols, uint64_t magic) {
  uint32_t nb[4];
  nbrs(l, rows, cols, magic, nb);
  const int nsum = spin_at(pos, nb[0]) + spin_at(pos, nb[1]) + spin_at(pos, nb[2]) +
                   spin_at(pos, nb[3]);
  return (spin_at(pos, l) > 0 ? 5 : 0) + ((nsum + 4) >> 1);
}

// A cross-lane read only sees lanes that are active when it executes.  The
// empty asm consumes the result where the call stands (all 64 lanes active),
// so the compiler cannot sink the read into a branch that masks off its
// source lanes.
template <typename T>
__device__ __forceinline__ T pinned(T v) {
  asm volatile("" : "+v"(v));
  return v;
}
// lane k receives lane k+1's value (row_shl:1) / lane k-1's (row_shr:1)
// within its row of 16 lanes; the walk uses lanes 0..10
__device__ __forceinline__ int row_shl1(int v) {
  return pinned(__builtin_amdgcn_update_dpp(0, v, 0x101, 0xf, 0xf, false));
}
__device__ __forceinline__ int row_shr1(int v) {
  return pinned(__builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));
}
// The running sums of lanes 0..9's values in lane order, all within the row of
// lanes 0..15: lane k ends with fl(..fl(v_0 + v_1).. + v_k), lanes 9..15 with the
// whole sum.  Step j adds lane j's value, broadcast over the row, times on[j],
// which is 1.0 in the lanes from j on and 0.0 below: an exact product, so each
// fused step rounds as one addition.  (Ten dependent fused adds; shifting the
// sums along took three instructions and two waits a step.)
__device__ __forceinline__ double running_sums(double v, const double (&on)[10]) {
  double run = 0.0;
  asm("s_nop 1\n"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %3 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %4 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %5 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %6 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %7 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %8 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %9 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %10 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %1, %11 row_newbcast:9 row_mask:0xf bank_mask:0xf"
      : "+v"(run)
      : "v"(v), "v"(on[0]), "v"(on[1]), "v"(on[2]), "v"(on[3]), "v"(on[4]), "v"(on[5]),
        "v"(on[6]), "v"(on[7]), "v"(on[8]), "v"(on[9]));
  return run;
}
// lane 9's value in every lane of its row
__device__ __forceinline__ double row_lane9(double v) {
  double d;
  asm("s_nop 1\nv_mov_b64_dpp %0, %1 row_newbcast:9 row_mask:0xf bank_mask:0xf" : "=v"(d) : "v"(v));
  return d;
}
// canonical_from_word (rng.hh) in fewer steps: hi 2^32 + lo rounds once, as the
// conversion does; the clamp of 1.0 is one of 2^64 to the double below it
__device__ __forceinline__ double canonical_of(uint64_t w) {
  const double x = __fma_rn((double)(uint32_t)(w >> 32), 4294967296.0, (double)(uint32_t)w);
  return (x < 18446744073709549568.0 ? x : 18446744073709549568.0) * 0x1p-64;
}
// lane k receives lane k - D's value within its row of 16 lanes (0 if none)
template <int D>
__device__ __forceinline__ uint32_t row_shr(uint32_t v) {
  return (uint32_t)pinned(__builtin_amdgcn_update_dpp(0, (int)v, 0x110 + D, 0xf, 0xf, true));
}
constexpr int RING_MIRROR = 2;  // the ring's first words once more behind its end
// the four neighbours' lanes in apply_event
constexpr uint64_t NEIGHBOUR_LANES = 0x8421ull;

}  // namespace

// GENERAL: lattices 1 or 2 wide among the chains, or event by event; the other
// instance keeps only what whole passes of wider lattices need (with both in one
// kernel its loop spilled scalar registers).
template <bool GENERAL>
__global__ __launch_bounds__(64) void nfold_kernel(const NfoldParams *__restrict__ Pp,
                                                   ExactState *__restrict__ Sp,
                                                   int8_t *__restrict__ lat_pool,
                                                   int32_t *__restrict__ list_pool,
                                                   mcg_sample *__restrict__ series,
                                                   int64_t series_cap,
                                                   const uint8_t *__restrict__ active,
                                                   int64_t n_passes, int64_t sample_period,
                                                   int sample_now, int64_t max_events,
                                                   double stop_time, int select_at_end) {
  const int c = blockIdx.x;
  if (!active[c]) return;
  const int lane = threadIdx.x;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ uint64_t raw[2][MT_N];
  __shared__ uint64_t ring[RING + RING_MIRROR];
  __shared__ int hist[16];

  const NfoldParams *P = Pp + c;
  ExactState *St = Sp + c;
  const int32_t rows = P->rows, cols = P->cols, n = P->n;
  const uint64_t magic = P->div_magic;
  const double period = P->time_period;
  const bool by_time = period > 0.0;
  int8_t *g_lat = lat_pool + P->lat_off;
  int32_t *g_arr = list_pool + P->lat_off;
  uint16_t *arr = reinterpret_cast<uint16_t *>(smem);
  uint16_t *pos = arr + n;

  for (int i = lane; i < MT_N; i += 64) {
    raw[0][i] = St->mt[i];
    ring[i] = mt_temper(raw[0][i]);
  }
  if (lane < 16) hist[lane] = 0;
  for (int i = lane; i < n; i += 64) {
    const uint32_t l = (uint32_t)g_arr[i];
    arr[i] = (uint16_t)l;
    pos[l] = (uint16_t)(i | (g_lat[l] > 0 ? SPIN_BIT : 0u));
  }
  __syncthreads();
  for (int l = lane; l < n; l += 64) atomicAdd(&hist[class_of(pos, l, rows, cols, magic)], 1);
  __syncthreads();
  // lane k holds start[k] (k <= 10) and rate[k] (k < 10)
  int startv = 0;
  for (int k = 0; k < 10; ++k)
    if (k < lane) startv += hist[k];
  const double ratev = lane < 10 ? P->rate[lane] : 0.0;

  const int64_t pos0 = St->pos;
  int64_t G = 0;
  int64_t n_pass = St->n_pass, n_ev = St->n_accept, n_samples = St->n_samples;
  int64_t S = St->S, M = St->M, next_k = St->next_k;
  double time = St->time;
  int64_t pending = St->pending_site;
  double pending_dt = St->pending_dt;
  int pending_kk = 0, pending_pos = -1;  // known when this launch selected it
  double pending_R = St->e_run;  // the total rate at the pending event's selection
  int64_t step = St->step;       // events done in the current pass
  const int self_nb = 2 * (rows == 1) + 2 * (cols == 1);
  const bool narrow = GENERAL && (rows <= 2 || cols <= 2);  // a neighbour can be listed twice
  bool frozen = false;  // total rate 0: the next event never comes

  // rs: ring slot of the next word; avail: readable words from it on
  int rs = (int)pos0, avail = MT_N - (int)pos0;
  auto ensure = [&](int upto) MCG_INLINE {
    while (__builtin_expect(avail < upto, 0)) {
      const int s = (int)((G + 1) & 1);
      twist_gen(raw[G & 1], raw[s], ring + s * MT_N, lane);
      if (s == 0 && lane < RING_MIRROR) ring[RING + lane] = ring[lane];
      ++G;
      avail += MT_N;
    }
  };
  auto take = [&](int words) MCG_INLINE {
    rs += words;
    avail -= words;
    if (rs >= RING) rs -= RING;
  };
  auto word = [&]() MCG_INLINE -> uint64_t {
    ensure(1);
    const uint64_t w = rfl64(ring[rs]);
    take(1);
    return w;
  };
  // select an event: its class and position in the class array, the
  // time-increment word w3 and the total rate R.  Lane k (k < 10) holds n_k and
  // the running rate sum up to class k, formed in class order (an empty class
  // adds +0.0).
  double on[10];
#pragma unroll
  for (int k = 0; k < 10; ++k) on[k] = lane >= k ? 1.0 : 0.0;
  auto select = [&](int &kk, int &site_pos, uint64_t &w3, double &R) MCG_INLINE {
    ensure(3);
    // the usual three words arrive while the rates are summed
    const uint64_t w0 = ring[rs], w1 = ring[rs + 1];
    w3 = ring[rs + 2];
    const int nxt = row_shl1(startv);
    const int nv = lane < 10 ? nxt - startv : 0;
    const double tv = __dmul_rn((double)nv, ratev);
    const double run = running_sums(tv, on);
    R = readlane_f64(run, 9);
    const double target = __dmul_rn(canonical_of(w0), row_lane9(run));  // (lanes 0..9 count)
    const uint64_t some = __ballot(nv > 0), hit = some & __ballot(target < run);
    kk = __builtin_ctzll(hit | (1ull << 63));
    if (__builtin_expect(hit == 0, 0))  // rounding left none: the last non-empty class
      kk = 63 - __clzll((unsigned long long)some);
    const uint32_t nk = (uint32_t)__builtin_amdgcn_readlane(nv, kk);
    const int st = __builtin_amdgcn_readlane(startv, kk);
    // Lemire over nk < 2^16: w1 * nk from two 32x32->64 products
    const uint64_t p0 = (uint64_t)(uint32_t)w1 * nk;
    const uint64_t p1 = (uint64_t)(uint32_t)(w1 >> 32) * nk + (p0 >> 32);
    site_pos = st + rfl32((int32_t)(p1 >> 32));
    take(3);
    if (__builtin_expect(rfl32((int32_t)p1) == 0, 0)) {  // the low word may be below nk
      uint64_t x = rfl64(w1);
      const uint64_t th = (0ULL - (uint64_t)nk) % (uint64_t)nk;
      if (x * nk < th) {
        rs = rs == 0 ? RING - 1 : rs - 1;  // the third word was not the time's
        ++avail;
        do {
          x = word();
        } while (x * nk < th);
        w3 = word();
      }
      site_pos = st + (int)__umul64hi(x, (uint64_t)nk);
    }
  };
  // Move site x from class a to class b at position p.  Going up, x swaps in
  // turn with the last entry of segments a, a+1, .., b-1 (each of which then
  // starts one lower); going down, with the first entry of segments a, a-1,
  // .., b+1 (each then starts one higher).  The chain of swaps is a rotation:
  // lane k holds the boundary between segments k-1 and k, reads the entry
  // there and writes it into the previous hole, all lanes at once; a boundary
  // that coincides with the previous one (empty segment) is a swap of x with
  // itself and writes nothing.
  auto move = [&](uint32_t x, int a, int b, int p_known) MCG_INLINE {
    const bool up = a < b;
    // lane k: the last entry of segment k-1 (up) or the first of segment k (down)
    const int q = up ? startv - 1 : startv;
    const int from_below = row_shr1(q), from_above = row_shl1(q);
    const bool act = up ? (lane > a && lane <= b) : (lane > b && lane <= a);
    uint32_t y = arr[act ? q : 0], px = pos[x];
    asm volatile("" : "+v"(y), "+v"(px));  // both reads issued before either is used
    const int p = p_known >= 0 ? p_known : rfl32((int32_t)(px & 0x7fffu));
    int qp = lane == (up ? a + 1 : a) ? p : up ? from_below : from_above;
    const int qx = __builtin_amdgcn_readlane(q, up ? b : b + 1);
    // an entry keeps its class (k - 1 going up, k going down), which fixes its
    // spin; lane 11 (outside the segment lanes) carries x to its final slot,
    // in class b, in the same writes
    int cls = up ? lane - 1 : lane;
    bool wr = act && q != qp;
    if (lane == 11) {
      y = x;
      qp = qx;
      cls = b;
      wr = true;
    }
    if (wr) {
      arr[qp] = (uint16_t)y;
      pos[y] = (uint16_t)(qp | (cls >= 5 ? SPIN_BIT : 0u));
    }
    startv += act ? (up ? -1 : 1) : 0;
    // the wave's LDS operations execute in issue order; keep the compiler from
    // moving the next move's reads above these writes
    asm volatile("" ::: "memory");
  };
  int dS = 0, dM = 0;  // changes not yet in S and M, in units of 4 and 2
  auto settle = [&]() MCG_INLINE {
    S += 4 * (int64_t)dS;
    M += 2 * (int64_t)dM;
    dS = dM = 0;
  };
  // a by-pass record also keeps the total rate R in e_run
  auto record = [&](double t, double w, double R) MCG_INLINE {
    if (lane == 0 && n_samples < series_cap) {
      mcg_sample rec = {};
      rec.pass = n_pass;
      rec.S1 = S;
      rec.M = M;
      rec.e_run = R;
      rec.time = t;
      rec.weight = w;
      series[(int64_t)c * series_cap + n_samples] = rec;
    }
    ++n_samples;
  };
  // by pass: select the pending event and sample the state with its increment
  auto sample_pass = [&]() MCG_INLINE {
    int kk, l_pos;
    uint64_t w3;
    double R;
    select(kk, l_pos, w3, R);
    pending_dt = -log1p(-canonical_of(w3)) / R;
    pending = rfl32((int32_t)arr[l_pos]);
    pending_kk = kk;
    pending_pos = l_pos;
    pending_R = R;
    record(time, pending_dt, R);
  };
  // the pass-0 sample, or a sample of the current pass asked for by the host,
  // unless this pass's first event is already selected
  if (max_events < 0 && !by_time && pending < 0 &&
      (sample_now || (P->sample_start && n_pass == 0 && n_samples == 0)))
    sample_pass();

  // Deferred time increments: lane j holds event j of the current batch (its
  // word and R, or its known increment's bits with R = -1, and the state before it).
  // A flush turns them into increments on all lanes at once, adds them to the
  // time in event order and, on the time grid, writes the batch's records.
  uint64_t bu = 0;
  double bR = 1.0;
  int bS = 0, bM = 0;  // (as changes from S and M)
  int nb_ev = 0;
  auto flush = [&]() MCG_INLINE {
    if (nb_ev == 0) return;
    const double dtv = bR < 0.0 ? __longlong_as_double((long long)bu)
                                : -log1p(-canonical_of(bu)) / bR;
    double tend = 0.0;
    if (!by_time && nb_ev == 64) {
#pragma unroll
      for (int j = 0; j < 64; ++j) time = __dadd_rn(time, readlane_f64(dtv, j));
    } else {
      for (int j = 0; j < nb_ev; ++j) {
        time = __dadd_rn(time, readlane_f64(dtv, j));
        tend = lane == j ? time : tend;
      }
    }
    if (by_time) {
      // first grid index k >= next_k with k * period >= t_end (the predicate
      // decides at the edge); t_end is non-decreasing, so each lane can
      // search from the batch's starting index
      int64_t k = next_k;
      const bool never = lane < nb_ev && !(tend <= 1.79769313486231570815e308);
      if (__ballot(never)) frozen = true;
      if (lane < nb_ev && !never) {
        k = (int64_t)ceil(tend / period);
        if (k < next_k) k = next_k;
        while (k > next_k && (double)(k - 1) * period >= tend) --k;
        while ((double)k * period < tend) ++k;
      }
      const int64_t ku = pinned(__shfl_up(k, 1));
      const int64_t kp = lane == 0 ? next_k : ku;
      const int64_t m = lane < nb_ev ? k - kp : 0;
      const uint64_t rec = __ballot(m > 0);
      if (m > 0) {
        const int64_t ns =
            n_samples + __popcll((unsigned long long)rec & ((1ULL << lane) - 1ULL));
        if (ns < series_cap) {
          mcg_sample r = {};
          r.pass = n_pass;
          r.S1 = S + 4 * (int64_t)bS;
          r.M = M + 2 * (int64_t)bM;
          r.time = (double)kp * period;
          r.weight = (double)m;
          series[(int64_t)c * series_cap + ns] = r;
        }
      }
      n_samples += __popcll((unsigned long long)rec);
      const int32_t klo = __builtin_amdgcn_readlane((int32_t)k, nb_ev - 1);
      const int32_t khi = __builtin_amdgcn_readlane((int32_t)(k >> 32), nb_ev - 1);
      next_k = ((int64_t)khi << 32) | (uint32_t)klo;
    }
    nb_ev = 0;
  };

  // flip site l (at position l_pos when known, else -1), update S and M, and
  // re-class it and its four neighbours
  auto apply = [&](uint32_t l, int l_pos) MCG_INLINE {
    // lanes 0..4 take l, +i, -i, +j, -j: their spin, neighbour sum, and how
    // many of their neighbour slots hold l
    const uint32_t lj = (uint32_t)(((uint64_t)l * magic) >> 40);
    const uint32_t li = l - lj * (uint32_t)rows;
    uint32_t xi = li, xj = lj;
    if (lane == 1) xi = li + 1 == (uint32_t)rows ? 0u : li + 1;
    if (lane == 2) xi = li == 0 ? (uint32_t)rows - 1 : li - 1;
    if (lane == 3) xj = lj + 1 == (uint32_t)cols ? 0u : lj + 1;
    if (lane == 4) xj = lj == 0 ? (uint32_t)cols - 1 : lj - 1;
    const uint32_t xs = xi + (uint32_t)rows * xj;
    const uint32_t xu = xi + 1 == (uint32_t)rows ? 0u : xi + 1;
    const uint32_t xd = xi == 0 ? (uint32_t)rows - 1 : xi - 1;
    const uint32_t yu = xj + 1 == (uint32_t)cols ? 0u : xj + 1;
    const uint32_t yd = xj == 0 ? (uint32_t)cols - 1 : xj - 1;
    const uint32_t xn[4] = {xu + (uint32_t)rows * xj, xd + (uint32_t)rows * xj,
                            xi + (uint32_t)rows * yu, xi + (uint32_t)rows * yd};
    const int sx = spin_at(pos, xs);
    const int nsx = spin_at(pos, xn[0]) + spin_at(pos, xn[1]) + spin_at(pos, xn[2]) +
                    spin_at(pos, xn[3]);
    const int mx = (xn[0] == l) + (xn[1] == l) + (xn[2] == l) + (xn[3] == l);
    const int s_old = __builtin_amdgcn_readlane(sx, 0);
    const int nsum = __builtin_amdgcn_readlane(nsx, 0);
    const int c_pre = (sx > 0 ? 5 : 0) + ((nsx + 4) >> 1);
    const int sp = xs == l ? -sx : sx;
    const int nsp = nsx - 2 * s_old * mx;
    const int c_post = (sp > 0 ? 5 : 0) + ((nsp + 4) >> 1);
    dS += -s_old * (nsum - self_nb * s_old) / 2;
    dM -= s_old;
    // the flip itself is written with l's move (its spin bit follows its class)
    // (only narrow lattices take these moves event after event: 1x3000, two passes 10.0 ms
    // in a loop and 7.5 unrolled)
    constexpr int UNROLL = GENERAL ? 5 : 1;
#pragma unroll UNROLL
    for (int t = 0; t < 5; ++t) {
      const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)xs, t);
      const int a = __builtin_amdgcn_readlane(c_pre, t), b = __builtin_amdgcn_readlane(c_post, t);
      bool dup = false;  // listed twice (a lattice 1 or 2 sites wide): moved once
      if (narrow)
        for (int u = 0; u < t; ++u) dup |= (uint32_t)__builtin_amdgcn_readlane((int)xs, u) == x;
      if (dup || a == b) continue;
      move(x, a, b, t == 0 ? l_pos : -1);
    }
  };

  // Lanes 5t + e: neighbour t (+i, -i, +j, -j) of the flipped site (e = 0) and its
  // own four neighbours (e = 1..4), as offsets on the ring of rows and columns.
  const int nt = lane / 5, ne = lane - 5 * nt;
  const uint32_t off_i = lane < 20 ? (uint32_t)(((nt == 0) - (nt == 1) + (ne == 1) - (ne == 2) + 2 * rows) % rows) : 0u;
  const uint32_t off_j = lane < 20 ? (uint32_t)(((nt == 2) - (nt == 3) + (ne == 3) - (ne == 4) + 2 * cols) % cols) : 0u;
  // The event of class kk at position site_pos (lattices at least 3 wide): the
  // site flips, which moves it five classes, and its neighbours one, all down
  // (an up spin flips) or all up, in the order of apply's moves.
  auto apply_dir = [&](auto dir, int kk, int site_pos) MCG_INLINE {
    constexpr bool down = decltype(dir)::value;
    const int nup = down ? kk - 5 : kk;
    dS += down ? 2 - nup : nup - 2;
    dM += down ? -1 : 1;
    // round trip 1.  The site's move is a rotation (see apply's move): lane k in
    // the five boundaries crossed holds the segment entry there; lane 11 the site.
    const int q = down ? startv : startv - 1;
    const int from_below = row_shr1(q), from_above = row_shl1(q);
    const int first = down ? kk - 4 : kk + 1;  // the crossed boundaries' lanes
    const bool act = (uint32_t)(lane - first) < 5u;
    uint32_t y = arr[lane == 11 ? site_pos : act ? q : 0];
    int qp = lane == (down ? kk : kk + 1) ? site_pos : down ? from_above : from_below;
    const int qx = __builtin_amdgcn_readlane(q, down ? first : first + 4);
    const bool site_lane = lane == 11;
    int cls = down ? lane : lane - 1;
    cls = site_lane ? (down ? kk - 5 : kk + 5) : cls;
    const uint64_t wr = (__ballot(act) & __ballot(q != qp)) | (1ull << 11);
    qp = site_lane ? qx : qp;
    if (__builtin_amdgcn_inverse_ballot_w64(wr)) {
      arr[qp] = (uint16_t)y;
      pos[y] = (uint16_t)(qp | (cls >= 5 ? SPIN_BIT : 0u));
    }
    startv += act ? (down ? 1 : -1) : 0;
    asm volatile("" ::: "memory");
    // round trip 2: pos entries (after the site's move, its new spin among them)
    const uint32_t x0 = (uint32_t)__builtin_amdgcn_readlane((int)y, 11);
    const uint32_t lj = (uint32_t)(((uint64_t)x0 * magic) >> 40);
    const uint32_t li = x0 - lj * (uint32_t)rows;
    uint32_t xi = li + off_i, xj = lj + off_j;
    xi = min(xi, xi - (uint32_t)rows);  // off the end: the other is huge
    xj = min(xj, xj - (uint32_t)cols);
    const uint32_t x = xi + (uint32_t)rows * xj;
    const uint32_t w = pos[x];
    const uint32_t up_bits = (uint32_t)__ballot(w & SPIN_BIT);
    const uint32_t spin = w & SPIN_BIT;
    uint32_t p = w & 0x7fffu;
    // the boundary neighbour t crosses: its class after the flip, one more going
    // down; entries before it in t's order have moved the boundary already
    const int kb = (int)__popc(__builtin_amdgcn_ubfe(up_bits, (uint32_t)lane + 1u, 4u)) +
                   (spin ? 5 : 0) + (down ? 1 : 0);
    int qn = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = __builtin_amdgcn_readlane(kb, 5 * u);
      const int s = __builtin_amdgcn_readlane(startv, k);
      qn = lane == 5 * u ? (down ? s : s - 1) : qn;
      startv += lane == k ? (down ? 1 : -1) : 0;
    }
    // round trip 3: the entries they swap with
    uint32_t yn = arr[qn];
    // an earlier swap (t) may have put its entry at this one's place (qn == p of
    // t) or moved this neighbour (x == yn of t)
    const uint32_t c1 = min((uint32_t)qn ^ row_shr<5>(p), x ^ row_shr<5>(yn));
    const uint32_t c2 = min((uint32_t)qn ^ row_shr<10>(p), x ^ row_shr<10>(yn));
    const uint32_t c3 = min((uint32_t)qn ^ row_shr<15>(p), x ^ row_shr<15>(yn));
    uint64_t live = NEIGHBOUR_LANES;  // their entry yn ends at p
    if (__builtin_expect((__ballot(min(c1, min(c2, c3)) == 0u) & NEIGHBOUR_LANES & ~1ull) != 0, 0)) {
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        const uint32_t pu = (uint32_t)__builtin_amdgcn_readlane((int)p, 5 * u);
        const uint32_t yu = (uint32_t)__builtin_amdgcn_readlane((int)yn, 5 * u);
        const uint64_t later = NEIGHBOUR_LANES & (~0ull << (5 * u + 1));
        const uint64_t there = __ballot((uint32_t)qn == pu) & later;
        const uint64_t moved = __ballot(x == yu) & later;
        yn = __builtin_amdgcn_inverse_ballot_w64(there) ? yu : yn;
        p = __builtin_amdgcn_inverse_ballot_w64(moved) ? pu : p;
        if (there | moved) live &= ~(1ull << (5 * u));
      }
    }
    if (__builtin_amdgcn_inverse_ballot_w64(live)) {
      arr[p] = (uint16_t)yn;
      pos[yn] = (uint16_t)(p | spin);  // its class is the neighbour's old one: the same spin
    }
    asm volatile("" ::: "memory");
    if (__builtin_amdgcn_inverse_ballot_w64(NEIGHBOUR_LANES)) {
      arr[qn] = (uint16_t)x;
      pos[x] = (uint16_t)((uint32_t)qn | spin);
    }
    asm volatile("" ::: "memory");
  };
  auto apply_event = [&](int kk, int site_pos) MCG_INLINE {
    if (kk >= 5)
      apply_dir(std::true_type{}, kk, site_pos);
    else
      apply_dir(std::false_type{}, kk, site_pos);
  };

  // Event by event (max_events >= 0; no records: the host samples), the
  // select-then-sample protocol of nfold.hh:121-141: the pending event is
  // applied first unless its time reaches stop_time; then events are selected
  // and, each time increment formed at once, applied until max_events are
  // done; an event whose time reaches stop_time, or (select_at_end) the one
  // after the last, is selected and left pending with its increment and the
  // total rate at its selection.  A total rate of 0 (no event ever comes)
  // stops the chain as frozen.
  if (GENERAL && max_events >= 0) {
    int64_t done = 0;
    bool stopped = false;
    auto bump = [&]() MCG_INLINE {
      ++n_ev;
      ++done;
      if (++step == n) {
        step = 0;
        ++n_pass;
      }
    };
    if (pending >= 0) {
      const double et = __dadd_rn(time, pending_dt);
      if (et >= stop_time) {
        stopped = true;
      } else {
        apply((uint32_t)pending, -1);
        time = et;
        pending = -1;
        bump();
      }
    }
    while (!stopped) {
      const bool select_only = done >= max_events;
      if (select_only && !select_at_end) break;
      int kk, l_pos;
      uint64_t w3;
      double R;
      select(kk, l_pos, w3, R);
      const uint32_t l = (uint32_t)rfl32((int32_t)arr[l_pos]);
      const double dt = -log1p(-canonical_of(w3)) / R;
      const double et = __dadd_rn(time, dt);
      if (!(et <= 1.79769313486231570815e308)) {
        frozen = true;
        break;
      }
      if (select_only || et >= stop_time) {
        pending = l;
        pending_dt = dt;
        pending_R = R;
        stopped = true;
      } else {
        if (narrow)
          apply(l, l_pos);
        else
          apply_event(kk, l_pos);
        time = et;
        bump();
      }
    }
    settle();
    n_passes = 0;
  }

  // the event goes into the batch of deferred time increments
  auto defer = [&](uint64_t w, double R) MCG_INLINE {
    const bool mine = lane == nb_ev;
    bu = mine ? w : bu;
    bR = mine ? R : bR;
    bS = mine ? dS : bS;
    bM = mine ? dM : bM;
    ++nb_ev;
  };
  for (int64_t pp = 0; pp < n_passes; ++pp) {
    // a pass begun by event-by-event advances ends at its boundary
    int32_t st = pp == 0 ? (int32_t)step : 0;
    step = 0;
    n_ev += n - st;
    if (pending >= 0 && st < n) {
      defer((uint64_t)__double_as_longlong(pending_dt), -1.0);
      if (pending_pos >= 0 && !narrow)
        apply_event(pending_kk, pending_pos);
      else
        apply((uint32_t)pending, -1);
      pending = -1;
      ++st;
      if (nb_ev == 64) flush();
    }
    for (; st < n && !frozen; ++st) {
      int kk, l_pos;
      uint64_t w3;
      double R;
      select(kk, l_pos, w3, R);
      defer(w3, R);
      if (narrow)
        apply((uint32_t)rfl32((int32_t)arr[l_pos]), l_pos);
      else
        apply_event(kk, l_pos);
      if (__builtin_expect(nb_ev == 64, 0)) flush();
    }
    n_ev -= n - st;  // (frozen: the events that did not come)
    flush();
    settle();
    if (frozen) break;
    ++n_pass;
    if (!by_time && n_pass % sample_period == 0) sample_pass();
  }

  __syncthreads();
  const int64_t pos_mt = (int64_t)MT_N * (G + 1) - avail;
  int64_t g_fin = 0, p_fin = pos0;
  if (pos_mt != pos0) {
    g_fin = (pos_mt - 1) / MT_N;
    p_fin = pos_mt - (int64_t)MT_N * g_fin;
  }
  for (int i = lane; i < MT_N; i += 64) St->mt[i] = raw[g_fin & 1][i];
  for (int i = lane; i < n; i += 64) {
    g_lat[i] = (pos[i] & SPIN_BIT) ? (int8_t)1 : (int8_t)-1;
    g_arr[i] = (int32_t)arr[i];
  }
  if (lane == 0) {
    St->pos = p_fin;
    St->n_pass = n_pass;
    St->n_accept = n_ev;
    St->S = S;
    St->M = M;
    St->n_samples = n_samples;
    St->time = time;
    St->pending_site = pending;
    St->pending_dt = pending_dt;
    St->e_run = pending_R;
    St->step = step;
    St->next_k = next_k;
    St->frozen = frozen ? 1 : 0;
  }
}

void launch_nfold(const NfoldParams *P, ExactState *S, int8_t *lat_pool, int32_t *list_pool,
                  mcg_sample *series, int64_t series_cap, const uint8_t *active, int n_chains,
                  int64_t n_passes, int64_t sample_period, int sample_now, int64_t max_events,
                  double stop_time, int select_at_end, bool general, int lds_bytes, hipStream_t stream) {
  if (general || max_events >= 0)
    hipLaunchKernelGGL(nfold_kernel<true>, dim3(n_chains), dim3(64), lds_bytes, stream, P, S,
                       lat_pool, list_pool, series, series_cap, active, n_passes, sample_period,
                       sample_now, max_events, stop_time, select_at_end);
  else
    hipLaunchKernelGGL(nfold_kernel<false>, dim3(n_chains), dim3(64), lds_bytes, stream, P, S,
                       lat_pool, list_pool, series, series_cap, active, n_passes, sample_period,
                       sample_now, max_events, stop_time, select_at_end);
}

hipError_t nfold_set_max_lds(int bytes) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(nfold_kernel<true>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return e;
  return hipFuncSetAttribute(reinterpret_cast<const void *>(nfold_kernel<false>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

#undef MCG_INLINE

}  // namespace mcg
