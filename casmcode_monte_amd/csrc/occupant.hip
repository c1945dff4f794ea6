// occupant.hip -- OCCUPANT mode: the reference's generic occupant-event
// Metropolis chain over an OccLocation with several asymmetric units, for
// semi-grand canonical single-site events or canonical pair swaps, reproduced
// bit for bit by one walking wavefront per chain.  In occupant_kernel a second one
// twists the engine's next generation meanwhile (mt_producer, walk.hh);
// occupant_sgc_kernel has four more waves.
//
// Reference: the loop of occupation_metropolis.hh:87-153 with
// propose_semigrand_canonical_event (OccEventProposal.hh:261-352) or
// propose_canonical_event (:109-236) over an OccLocation (OccLocation.hh:
// 257-261 choose_mol; OccLocation.cc:39-118 initialize, 216-283 apply) and
// metropolis_acceptance (metropolis.hh:25-35).
//
// Per step the reference draws one word for the swap type (random_real over
// the summed counts of the swap types: n(cand_a) for semi-grand swaps,
// n(cand_a) n(cand_b) for canonical ones), one Lemire word for the slot in
// cand_a's list (and, canonical, one for cand_b's), and one more only when
// dE >= 0.  dE is a function of the swap type and the neighbour sums (Sa, and
// for pairs Sb of b after a changed), so the acceptance is a per-class word
// threshold as in the EXACT mode; the class tables come from the host.
//
// Device OccLocation: every asymmetric unit b with two occupants owns a
// segment [off_b, off_b + size_b) of the LDS list array that holds both of its
// candidate lists: occupant 0's from the front (slot j at off_b + j), occupant
// 1's from the back (slot j at off_b + size_b - 1 - j).  Removing slot i of a
// list moves its last entry into slot i (OccLocation.cc:262-266), and the
// position that frees is exactly where the other list's push_back lands, so a
// transform is two LDS writes.  Entries are site indices; the host converts
// them to and from Mol ids.  Sites of units with one occupant are in no list.
//
// Block walk: lane t evaluates stream position P+t as if a step started there,
// from the block-start state.  Rejected steps change nothing, so every step up
// to and including the first accepted one is exact; the block commits those
// and starts again after them.  (An accepted step changes the list sizes and
// with them every later step's swap choice and Lemire range, so nothing past
// it can be kept.)
//
// occupant_kernel takes every system.  The common one -- semi-grand events whose
// swap types are, unit by unit, occupant 0 -> 1 and then 1 -> 0 of at most three
// units (what make_semigrand_canonical_swaps builds) -- has its own kernel,
// occupant_sgc_kernel below.
#include <cstddef>

#include "internal.hh"
#include "walk.hh"

namespace mcg {

namespace {

// one swap type's lists at the block start: sizes, slot -> position maps
// (position = base + dir * slot) and units.  dir is +1 for a unit's occupant-0
// list (the front of its segment) and -1 for its occupant-1 list, so it is
// also the occupant change of a transformed site (0 -> 1 or 1 -> 0).
struct SwapTab {
  int32_t na, base_a, dir_a, ua;
  int32_t nb, base_b, dir_b, ub;
};

struct Nbrs {
  uint32_t up, dn, rt, lf;
};

__device__ __forceinline__ Nbrs nbrs_of(uint32_t l, int32_t rows, int32_t cols, uint64_t magic) {
  const uint32_t j = (uint32_t)(((uint64_t)l * magic) >> 40);
  const uint32_t i = l - j * (uint32_t)rows;
  const uint32_t iu = (i + 1 == (uint32_t)rows) ? 0u : i + 1;
  const uint32_t id = (i == 0) ? (uint32_t)rows - 1 : i - 1;
  const uint32_t ju = (j + 1 == (uint32_t)cols) ? 0u : j + 1;
  const uint32_t jd = (j == 0) ? (uint32_t)cols - 1 : j - 1;
  return {iu + (uint32_t)rows * j, id + (uint32_t)rows * j, i + (uint32_t)rows * ju,
          i + (uint32_t)rows * jd};
}

// A site's byte is its occupant + 2 (its neighbour slots at occupant 1): a proposal reads
// one byte a site, and an accepted event adds to five (exact modulo 2^32 in any order).
__device__ __forceinline__ void add_byte(uint8_t *lat, uint32_t l, uint32_t v) {
  atomicAdd(reinterpret_cast<uint32_t *>(lat) + (l >> 2), v << (8u * (l & 3u)));
}
__device__ __forceinline__ void flip_byte(uint8_t *lat, uint32_t l, const Nbrs &nb, int dir) {
  add_byte(lat, l, (uint32_t)dir);
  const uint32_t two = (uint32_t)(2 * dir);
  add_byte(lat, nb.up, two);
  add_byte(lat, nb.dn, two);
  add_byte(lat, nb.rt, two);
  add_byte(lat, nb.lf, two);
}
// sum of the neighbour slots' spins (a slot that is the site itself among them)
__device__ __forceinline__ int spin_sum(uint8_t v) { return 2 * (v >> 1) - 4; }

// One proposed event evaluated from a state: the swap type, the chosen sites
// with their list positions and the positions (and entries) of their lists'
// last slots, the class, and the bond-sum and spin-sum changes.
struct Proposal {
  SwapTab e;
  int32_t pa, pba, pb, pbb;
  uint32_t a, la, b, lb;
  int k, dS, dM;
};

// The neighbour sums, class and observable changes of a proposal whose sites
// are known (the site and list-entry reads done).
__device__ __forceinline__ void classify(Proposal &p, int si, int canonical, const uint8_t *lat,
                                         int32_t rows, int32_t cols, uint64_t magic) {
  const int sa_old = p.e.dir_a < 0 ? 1 : -1, sa_new = -sa_old;
  const int self_nb = 2 * (rows == 1) + 2 * (cols == 1);  // slots that are the site itself
  const int Sa = spin_sum(lat[p.a]);
  p.k = si * 25 + ((Sa + 4) >> 1) * 5;
  p.dS = (sa_new - sa_old) * (Sa - self_nb * sa_old);
  p.dM = sa_new - sa_old;
  if (canonical) {  // b after a has changed
    const int sb_old = p.e.dir_b < 0 ? 1 : -1, sb_new = -sb_old;
    const Nbrs nb = nbrs_of(p.b, rows, cols, magic);
    const int at_a = (nb.up == p.a) + (nb.dn == p.a) + (nb.rt == p.a) + (nb.lf == p.a);
    const int Sb = spin_sum(lat[p.b]) + at_a * (sa_new - sa_old);
    p.k += (Sb + 4) >> 1;
    p.dS += (sb_new - sb_old) * (Sb - self_nb * sb_old);
    p.dM += sb_new - sb_old;
  }
}

// OccLocation.cc:254-283 for a, then for b (the second transform sees the
// first's lists), by one lane: each removal moves its list's last entry into
// the freed slot, and the position the last entry leaves is where the other
// list of the unit appends.  With a and b on one unit, b's list has gained a
// at that position, so b's removal moves a into b's slot and b lands there.
__device__ __forceinline__ void apply_proposal(const Proposal &p, int canonical, uint8_t *lat,
                                               uint16_t *list, int32_t *cnt, int32_t rows,
                                               int32_t cols, uint64_t magic) {
  list[p.pa] = (uint16_t)p.la;
  list[p.pba] = (uint16_t)p.a;
  flip_byte(lat, p.a, nbrs_of(p.a, rows, cols, magic), p.e.dir_a);
  atomicAdd(&cnt[p.e.ua], -p.e.dir_a);
  if (canonical) {
    if (p.e.ub == p.e.ua) {
      list[p.pb] = (uint16_t)p.a;
      list[p.pba] = (uint16_t)p.b;
    } else {
      list[p.pb] = (uint16_t)p.lb;
      list[p.pbb] = (uint16_t)p.b;
    }
    flip_byte(lat, p.b, nbrs_of(p.b, rows, cols, magic), p.e.dir_b);
    atomicAdd(&cnt[p.e.ub], -p.e.dir_b);
  }
}

}  // namespace

// canonical: pair swaps; NS: swap types at most.  A block's time is its ~300 instructions,
// ~120 more for an accepted event, and the chain word -> type -> slot -> sites -> bytes ->
// class -> starts.  Measured on MI355X, one chain of 128x128 sites over two units, four pair
// swaps, 131072 steps: 10.4 ms at 500 K and 32.9 at 3000 K (14.6 and 43.4 with a byte that
// was the occupant alone; 26.1 and 62.8 with that, the starts taken an attempt at a time,
// 64-bit products and 15 compares for the type).
template <bool canonical, int NS>
__global__ __launch_bounds__(128) void occupant_kernel(
    const OccParams *__restrict__ Pp, const OccTables *__restrict__ Tp,
    ExactState *__restrict__ Sp, int8_t *__restrict__ lat_pool, int32_t *__restrict__ list_pool,
    mcg_sample *__restrict__ series, int64_t series_cap, const uint8_t *__restrict__ active,
    int64_t n_passes, int64_t n_steps, int64_t sample_period) {
  const int c = blockIdx.x;
  if (!active[c]) return;
  const int lane = threadIdx.x & 63;
  const bool producer = threadIdx.x >= 64;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ uint64_t raw[3][MT_N];
  __shared__ uint64_t ring[3][MT_N];
  __shared__ int done;
  __shared__ uint64_t thr_s[OCC_NCLASS];
  __shared__ double dq_s[OCC_NCLASS];
  __shared__ uint8_t flg_s[OCC_NCLASS];
  __shared__ SwapTab tab_s[OCC_MAX_SWAPS];
  __shared__ int32_t cnt_s[OCC_MAX_ASYM];

  const OccParams *P = Pp + c;
  const OccTables *T = Tp + c;
  ExactState *St = Sp + c;
  const int32_t rows = P->rows, cols = P->cols, n = P->n, n_mut = P->n_mut;
  const int n_swaps = P->n_swaps, W = P->window;
  const uint64_t magic = P->div_magic;
  int8_t *g_lat = lat_pool + P->lat_off;
  int32_t *g_list = list_pool + P->lat_off;
  uint8_t *lat = smem;
  uint16_t *list = reinterpret_cast<uint16_t *>(smem + ((n + 15) & ~15));

  if (!producer) {
    for (int i = lane; i < MT_N; i += 64) {
      raw[0][i] = St->mt[i];
      ring[0][i] = mt_temper(raw[0][i]);
    }
    for (int i = lane; i < OCC_NCLASS; i += 64) {
      thr_s[i] = T->thr[i];
      dq_s[i] = T->dq[i];
      flg_s[i] = T->flags[i];
    }
    if (lane < OCC_MAX_ASYM) cnt_s[lane] = St->occ_cnt0[lane];
    for (int i = lane; i < ((n + 15) & ~15); i += 64) lat[i] = i < n ? (uint8_t)(g_lat[i] & 1) : 0;
    asm volatile("" ::: "memory");  // (one wave: its LDS operations execute in issue order)
    for (int i = lane; i < n; i += 64) {
      if (!(g_lat[i] & 1)) continue;
      const Nbrs nb = nbrs_of((uint32_t)i, rows, cols, magic);
      add_byte(lat, nb.up, 2u);
      add_byte(lat, nb.dn, 2u);
      add_byte(lat, nb.rt, 2u);
      add_byte(lat, nb.lf, 2u);
    }
    for (int i = lane; i < n_mut; i += 64) list[i] = (uint16_t)g_list[i];
    if (lane == 0) done = 0;
  }
  __syncthreads();
  if (producer) {  // wave 1 twists the engine (walk.hh); wave 0 walks
    mt_producer(raw, ring, &done, lane);
    return;
  }

  // Lane j < n_swaps keeps swap type j's table entry (its two lists' sizes
  // change with every accepted event of their units) and writes it to tab_s
  // when it changes; the cumulative counts tsum[j+1] are exact integers, kept
  // uniform.
  SwapTab mine = {};
  if (lane < n_swaps) {
    const int ca = P->swap_a[lane], cb = P->swap_b[lane];
    const int ua = P->cand_asym[ca], oa = P->cand_occ[ca];
    const int ub = P->cand_asym[cb], ob = P->cand_occ[cb];
    const int32_t c0a = St->occ_cnt0[ua], c0b = St->occ_cnt0[ub];
    const int32_t za = P->asym_size[ua], zb = P->asym_size[ub];
    mine.na = oa ? za - c0a : c0a;
    mine.base_a = P->asym_off[ua] + (oa ? za - 1 : 0);
    mine.dir_a = oa ? -1 : 1;
    mine.ua = ua;
    mine.nb = ob ? zb - c0b : c0b;
    mine.base_b = P->asym_off[ub] + (ob ? zb - 1 : 0);
    mine.dir_b = ob ? -1 : 1;
    mine.ub = ub;
  }

  const int64_t pos0 = St->pos;
  int64_t pos = pos0;
  MtRing3 eng;
  int64_t n_pass = St->n_pass, n_acc = St->n_accept, n_rej = St->n_reject;
  int64_t S = St->S, M = St->M, n_samples = St->n_samples;
  double e_run = St->e_run;
  int64_t step = St->step;
  int64_t frozen = 0;

  auto ensure = [&](int64_t upto) { eng.ensure(upto); };
  const uint64_t *ringf = &ring[0][0];
  auto word = [&](int64_t q) -> uint64_t { return ringf[eng.index(q)]; };
  // libstdc++ uniform_int_distribution over [0, m-1] with the rejection loop
  auto lemire_scalar = [&](uint64_t m) -> uint32_t {
    ensure(pos + 1);
    uint64_t x = word(pos);
    ++pos;
    uint64_t lo = x * m, hi = __umul64hi(x, m);
    if (lo < m) {
      const uint64_t th = (0ULL - m) % m;
      while (lo < th) {
        ensure(pos + 1);
        x = word(pos);
        ++pos;
        lo = x * m;
        hi = __umul64hi(x, m);
      }
    }
    return (uint32_t)hi;
  };

  uint32_t ts[NS];  // the last types' beyond any draw
  double Ttot = 0.0;
  // OccEventProposal.hh:127-139 / 276-288: the cumulative counts from the
  // lanes' entries (n(cand_a), or n(cand_a) n(cand_b) for canonical swaps)
  auto publish = [&]() {
    uint32_t w = 0;
    if (lane < n_swaps) {
      tab_s[lane] = mine;
      w = canonical ? (uint32_t)mine.na * (uint32_t)mine.nb : (uint32_t)mine.na;
    }
    uint32_t run = 0;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      run += __builtin_amdgcn_readlane(w, j);
      ts[j] = j < n_swaps - 1 ? run : 0xFFFFFFFFu;
    }
    Ttot = (double)run;
    asm volatile("" ::: "memory");
  };
  // the swap type of a draw: the first j with rand < tsum[j+1]; for an integer
  // t, rand < t exactly when floor(rand) < t, so the comparisons are integer
  // ones: the number of tsum[j+1] <= floor(rand) (they do not decrease, and
  // rand < tsum[n_swaps])
  auto choose = [&](double rand) -> int {
    const uint32_t r = (uint32_t)rand;
    int i = 0;
#pragma unroll
    for (int j = 0; j < NS - 1; ++j) i += ts[j] <= r ? 1 : 0;
    return i;
  };
  // every lane's entry after an accepted event changed the occupant-0 counts
  // of units ua (by -dir_a) and, canonical, ub (by -dir_b)
  auto account = [&](int ua, int dir_a, int ub, int dir_b) {
    if (lane < n_swaps) {
      auto d = [&](int u) { return (u == ua ? -dir_a : 0) + (canonical && u == ub ? -dir_b : 0); };
      mine.na += d(mine.ua) * mine.dir_a;
      mine.nb += d(mine.ub) * mine.dir_b;
    }
  };

  // slot of a Lemire word among m, and whether the word may be rejected (low half < m)
  auto slot_of = [&](uint64_t x, uint32_t m, bool &may_reject) -> uint32_t {
    const uint64_t p0 = (uint64_t)(uint32_t)x * m;
    const uint64_t p1 = (uint64_t)(uint32_t)(x >> 32) * m + (p0 >> 32);
    may_reject |= (uint32_t)p1 == 0u && (uint32_t)p0 < m;
    return (uint32_t)(p1 >> 32);
  };
  constexpr int base_len = canonical ? 3 : 2;
  WindowStarts<base_len> starts;
  const uint64_t win = W >= 64 ? ~0ull : (1ull << W) - 1ull;
  const int64_t target = n_passes * (int64_t)n_mut + n_steps;
  int64_t done_steps = 0;
  bool dirty = true;
  while (done_steps < target) {
    if (dirty) {
      publish();
      dirty = false;
    }
    if (Ttot == 0.0) {  // OccEventProposal.hh:136-139 / 290-293: no events possible
      frozen = 1;
      break;
    }
    ensure(pos + W + 3);
    const bool inwin = lane < W;
    const int64_t q = inwin ? pos + lane : pos;
    // consecutive positions are consecutive words of the ring
    auto after = [](uint32_t i) { return min(i + 1u, i + 1u - 3u * MT_N); };
    const uint32_t i0 = (uint32_t)eng.index(q), i1 = after(i0), i2 = after(i1), i3 = after(i2);
    const uint64_t x0 = ringf[i0], x1 = ringf[i1], x2 = ringf[i2];
    const uint64_t x3 = canonical ? ringf[i3] : 0ULL;
    const double rand = __dmul_rn(canonical_from_word(x0), Ttot);  // random_real(tsum.back())
    const int si = choose(rand);
    Proposal p;
    p.e = tab_s[si];
    bool special = false;
    const uint32_t sa = slot_of(x1, (uint32_t)p.e.na, special);
    p.pa = p.e.base_a + p.e.dir_a * (int32_t)sa;
    p.pba = p.e.base_a + p.e.dir_a * (p.e.na - 1);
    p.a = list[p.pa];
    p.la = list[p.pba];
    uint64_t xm = x2;
    if (canonical) {
      const uint32_t sb = slot_of(x2, (uint32_t)p.e.nb, special);
      p.pb = p.e.base_b + p.e.dir_b * (int32_t)sb;
      p.pbb = p.e.base_b + p.e.dir_b * (p.e.nb - 1);
      p.b = list[p.pb];
      p.lb = list[p.pbb];
      xm = x3;
    }
    classify(p, si, canonical, lat, rows, cols, magic);
    const uint32_t fl = flg_s[p.k];
    const uint64_t thr = thr_s[p.k];
    const double dq = dq_s[p.k];
    const bool nd = !(fl & 1u);
    const bool acc = !nd || (fl & 2u) || (xm < thr);
    const uint64_t ND = __ballot(nd);
    const uint64_t AC = __ballot(acc);
    const uint64_t SP = __ballot(special);

    // step starts: 0, then +base_len or +base_len+1 (a uniform drawn), up to
    // the first accepted step or before the first special one
    uint64_t exec = starts(nd) & win;
    const uint64_t stop = exec & (AC | SP);
    if (stop) {
      const uint64_t f = stop & (0ull - stop);
      exec &= (f - 1ull) | (f & ~SP);
    }
    int steps = __popcll(exec);
    const int64_t to_pass_end = (int64_t)n_mut - step;
    const int64_t to_target = target - done_steps;
    const int64_t lim = to_pass_end < to_target ? to_pass_end : to_target;
    if (steps > lim) {
      uint64_t rest = exec;
      for (int r = 0; r < lim; ++r) rest &= rest - 1;
      exec ^= rest;
      steps = (int)lim;
    }
    int used = 0;
    if (exec) {
      const int last = 63 - __builtin_clzll(exec);
      used = last + base_len + (int)((ND >> last) & 1ull);
    }
    const uint64_t F = exec & AC;  // at most one step: the last one
    if (F) {
      const int f = __builtin_ctzll(F);
      if (lane == f) apply_proposal(p, canonical, lat, list, cnt_s, rows, cols, magic);
      asm volatile("" ::: "memory");
      e_run = __dadd_rn(e_run, readlane_f64(dq, f));
      S += __builtin_amdgcn_readlane(p.dS, f);
      M += __builtin_amdgcn_readlane(p.dM, f);
      const int ua = __builtin_amdgcn_readlane(p.e.ua, f), da = __builtin_amdgcn_readlane(p.e.dir_a, f);
      const int ub = __builtin_amdgcn_readlane(p.e.ub, f), db = __builtin_amdgcn_readlane(p.e.dir_b, f);
      ++n_acc;
      if (!canonical || ua != ub || da + db != 0) {  // else a unit's swap: no list's size changes
        account(ua, da, ub, db);
        dirty = true;
      }
    }
    n_rej += steps - (F ? 1 : 0);
    pos += used;
    step += steps;
    done_steps += steps;

    if ((SP & 1ull) && steps == 0 && done_steps < target) {
      // a step whose Lemire draw may reject, with the full rejection loops;
      // every lane computes it, lane 0 writes
      ensure(pos + 1);
      const double r1 = __dmul_rn(canonical_from_word(word(pos)), Ttot);
      ++pos;
      const int i1 = choose(r1);
      Proposal q1;
      q1.e = tab_s[i1];
      const uint32_t s1a = lemire_scalar((uint64_t)q1.e.na);
      q1.pa = q1.e.base_a + q1.e.dir_a * (int32_t)s1a;
      q1.pba = q1.e.base_a + q1.e.dir_a * (q1.e.na - 1);
      q1.a = list[q1.pa];
      q1.la = list[q1.pba];
      if (canonical) {
        const uint32_t s1b = lemire_scalar((uint64_t)q1.e.nb);
        q1.pb = q1.e.base_b + q1.e.dir_b * (int32_t)s1b;
        q1.pbb = q1.e.base_b + q1.e.dir_b * (q1.e.nb - 1);
        q1.b = list[q1.pb];
        q1.lb = list[q1.pbb];
      }
      classify(q1, i1, canonical, lat, rows, cols, magic);
      bool ok;
      if (flg_s[q1.k] & 1u) {
        ok = true;
      } else {
        ensure(pos + 1);
        const uint64_t xr = word(pos);
        ++pos;
        ok = (flg_s[q1.k] & 2u) || (xr < thr_s[q1.k]);
      }
      // one wavefront walks: its LDS operations execute in issue order and the
      // asm keeps the compiler from reordering them
      asm volatile("" ::: "memory");
      if (ok) {
        if (lane == 0) apply_proposal(q1, canonical, lat, list, cnt_s, rows, cols, magic);
        e_run = __dadd_rn(e_run, dq_s[q1.k]);
        S += q1.dS;
        M += q1.dM;
        account(q1.e.ua, q1.e.dir_a, q1.e.ub, q1.e.dir_b);
        ++n_acc;
        dirty = true;
      } else {
        ++n_rej;
      }
      asm volatile("" ::: "memory");
      ++step;
      ++done_steps;
    }

    if (step == n_mut) {
      step = 0;
      ++n_pass;
      if (n_pass % sample_period == 0) {
        if (lane == 0 && n_samples < series_cap) {
          mcg_sample rec = {};
          rec.pass = n_pass;
          rec.S1 = S;
          rec.M = M;
          rec.e_run = e_run;
          series[(int64_t)c * series_cap + n_samples] = rec;
        }
        ++n_samples;
      }
    }
  }

  // release the producer (it waits at the barrier this one matches)
  eng.finish(&done, lane);
  int64_t g_fin = 0, p_fin = pos0;
  if (pos != pos0) {
    g_fin = (pos - 1) / MT_N;
    p_fin = pos - (int64_t)MT_N * g_fin;
  }
  for (int i = lane; i < MT_N; i += 64) St->mt[i] = raw[g_fin % 3][i];
  for (int i = lane; i < n; i += 64) g_lat[i] = (int8_t)(lat[i] & 1);
  for (int i = lane; i < n_mut; i += 64) g_list[i] = (int32_t)list[i];
  if (lane < OCC_MAX_ASYM) St->occ_cnt0[lane] = cnt_s[lane];
  if (lane == 0) {
    St->pos = p_fin;
    St->n_pass = n_pass;
    St->n_accept = n_acc;
    St->n_reject = n_rej;
    St->S = S;
    St->M = M;
    St->e_run = e_run;
    St->n_samples = n_samples;
    St->step = step;
    St->frozen = frozen;
  }
}

// ---------------------------------------------------------------------------
// Semi-grand events over U units with their swap types in pairs (0 -> 1, 1 -> 0).
//
// Every mutating site is in exactly one swap type's list, so the summed counts
// never change, and a step's draw fixes its unit and its place r' within the
// unit's pair ahead of time; only the split of a pair (the number of its sites
// at occupant 0) moves.  As in the EXACT block walk (exact.hip) whatever does not
// depend on the state is done by other waves, since the latency of one dependent
// chain bounds the walk: waves 2-4 twist the engine and turn each word into a
// record (r', unit, and which of the 10 U classes the word accepts), wave 1 adds
// energies and writes samples.  The lattice holds each site's class in a byte,
// 5 (2 unit + occupant) + up neighbours, so a step reads one list entry and one
// byte, and an accepted one adds to five bytes (exact modulo 2^32 in any order).
// Blocks end at the first accepted step as in occupant_kernel: it changes the
// split and with it half of the later steps' slots.
//
// Measured on MI355X, 64 chains of 128x128 sites over two units, 131072 steps each:
// 74.7 ms by occupant_kernel, 23.5 ms here (1370 and 450 cycles a step at 2.4 GHz
// for the chain that accepts most, 45 for the coldest): a block per accepted step,
// its time the chain record -> list entry -> class byte -> starts -> next record.
// The starts come from one scan of the window, not an attempt at a time: 28.1 ms and
// 225 cycles a step cold without it.  Blocks that went on to a second accepted step
// (21 words three times, for the splits one step can leave) took 23.4 ms but 1.2 to
// 1.4 times as long below an acceptance of 0.2.
// ---------------------------------------------------------------------------
namespace {

constexpr int OCC_THREADS = 5 * 64;
constexpr int OCC_SGC_UNITS = 3;                    // at most: 30 acceptance bits a word
constexpr int OCC_SGC_NCLASS = 10 * OCC_SGC_UNITS;
// the class byte of a site in no list starts here (its value is never used)
constexpr uint32_t OCC_FIXED_CLASS = 200;

// fixed LDS parts at address 0; the lattice follows, then the lists
struct OccWalkLds {
  uint64_t x[REC_RING + REC_MIRROR];    // tempered words
  uint64_t rec[REC_RING + REC_MIRROR];  // low: r' | unit << 16, high: accepted classes
  uint64_t raw[3][MT_N];
  double dq[OCC_SGC_NCLASS + 2];
  int32_t dS[OCC_SGC_NCLASS + 2], dM[OCC_SGC_NCLASS + 2];
  uint8_t fifo[FIFO];
  uint32_t done, pub;
};
static_assert(sizeof(OccWalkLds) <= OCC_SGC_FIXED_LDS, "the lattice starts behind it");
static_assert(OCC_MAX_SITES_LDS <= 65535, "r' and the lists are 16-bit");

}  // namespace

template <int U>
__global__ __launch_bounds__(OCC_THREADS) void occupant_sgc_kernel(
    const OccParams *__restrict__ Pp, const OccTables *__restrict__ Tp,
    ExactState *__restrict__ Sp, int8_t *__restrict__ lat_pool, int32_t *__restrict__ list_pool,
    const int8_t *__restrict__ asym_pool, mcg_sample *__restrict__ series_pool,
    int64_t series_cap, const uint8_t *__restrict__ active, int64_t n_passes, int64_t n_steps,
    int64_t sample_period) {
  const int c = blockIdx.x;
  if (!active[c]) return;
  const int lane = threadIdx.x & 63;
  const int wave = rfl32(threadIdx.x >> 6);
  extern __shared__ __align__(16) unsigned char smem[];

  const OccParams *P = Pp + c;
  const OccTables *T = Tp + c;
  ExactState *St = Sp + c;
  mcg_sample *series = series_pool + (int64_t)c * series_cap;
  const int32_t rows = P->rows, cols = P->cols, n = P->n, n_mut = P->n_mut;
  int8_t *g_lat = lat_pool + P->lat_off;
  const int8_t *g_asym = asym_pool + P->lat_off;
  int32_t *g_list = list_pool + P->lat_off;
  OccWalkLds &L = *reinterpret_cast<OccWalkLds *>(smem);
  volatile lds_u32 *done = lds_at(offsetof(OccWalkLds, done));
  volatile lds_u32 *pub = lds_at(offsetof(OccWalkLds, pub));
  uint8_t *cls = smem + OCC_SGC_FIXED_LDS;
  const uint32_t list_base = OCC_SGC_FIXED_LDS + (((uint32_t)n + 15u) & ~15u);
  uint16_t *list = reinterpret_cast<uint16_t *>(smem + list_base);
  // pair u: asymmetric unit, segment, place of its first type's draws
  int unit[U], off[U], size[U], first_r[U];
#pragma unroll
  for (int u = 0, r = 0; u < U; ++u) {
    unit[u] = P->cand_asym[P->swap_a[2 * u]];
    off[u] = P->asym_off[unit[u]];
    size[u] = P->asym_size[unit[u]];
    first_r[u] = r;
    r += size[u];
  }
  // acceptance of each class: bit 5 type + up neighbours
  uint32_t nd_mask = 0, always = 0;
  uint64_t thr[10 * U];
#pragma unroll
  for (int k = 0; k < 10 * U; ++k) {
    const int t = 25 * (k / 5) + 5 * (k % 5);
    const uint32_t f = T->flags[t];
    nd_mask |= (f & 1u ? 0u : 1u) << k;
    always |= (f ? 1u : 0u) << k;
    thr[k] = f ? 0 : T->thr[t];
  }
  const double Ttot = (double)n_mut;
  auto record = [&](uint64_t x) -> uint64_t {
    // OccEventProposal.hh:276-288: the first type whose cumulative count exceeds
    // random_real(total); floor(rand) decides it (occupant_kernel's choose)
    const uint32_t r = (uint32_t)__dmul_rn(canonical_from_word(x), Ttot);
    uint32_t u = 0, base = 0;
#pragma unroll
    for (int k = 1; k < U; ++k) {
      const bool in = r >= (uint32_t)first_r[k];
      u = in ? (uint32_t)k : u;
      base = in ? (uint32_t)first_r[k] : base;
    }
    uint32_t acc = always;
#pragma unroll
    for (int k = 0; k < 10 * U; ++k) acc |= (x < thr[k] ? 1u : 0u) << k;
    return ((uint64_t)acc << 32) | (r - base) | (u << 16);
  };
  auto put = [&](int slot, int k, uint64_t raw_word, int = 0) {
    const uint64_t x = mt_temper(raw_word), r = record(x);
    L.x[slot * MT_N + k] = x;
    L.rec[slot * MT_N + k] = r;
    if (slot == 0) {
      L.x[REC_RING + k] = x;
      L.rec[REC_RING + k] = r;
    }
  };

  // classes without neighbours first, then every up site adds one to the four
  for (int i = threadIdx.x; i < ((n + 15) & ~15); i += OCC_THREADS) {
    uint32_t v = OCC_FIXED_CLASS;
    if (i < n) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (g_asym[i] == unit[u]) v = 5u * (2u * u + (uint32_t)(g_lat[i] & 1));
    }
    cls[i] = (uint8_t)v;
  }
  for (int i = threadIdx.x; i < n_mut; i += OCC_THREADS) list[i] = (uint16_t)g_list[i];
  for (int i = threadIdx.x; i < MT_N; i += OCC_THREADS) {
    L.raw[0][i] = St->mt[i];
    put(0, i, St->mt[i]);
  }
  if (threadIdx.x < 10 * U) {
    const int k = threadIdx.x, s = (k / 5) & 1 ? 1 : -1, m = 2 * (k % 5) - 4;
    const int self_nb = 2 * (rows == 1) + 2 * (cols == 1);
    L.dq[k] = T->dq[25 * (k / 5) + 5 * (k % 5)];
    L.dS[k] = -2 * s * (m - self_nb * s);  // a slot that is the site itself keeps its bond
    L.dM[k] = -2 * s;
  }
  if (threadIdx.x == 0) {
    *done = 0;
    *pub = 0;
  }
  // floor(l / rows) for l rows < 2^31
  const uint32_t magic = (uint32_t)(((1ull << 31) + (uint32_t)rows - 1) / (uint32_t)rows);
  auto add_byte = [&](uint32_t l, uint32_t v) {
    lds_add(OCC_SGC_FIXED_LDS + (l & ~3u), v << ((l & 3u) * 8u));
  };
  auto neighbours = [&](uint32_t l, uint32_t (&x)[4]) {
    const uint32_t j = (uint32_t)(((uint64_t)l * magic) >> 31);
    const uint32_t i = l - j * (uint32_t)rows;
    const uint32_t wrap = (uint32_t)rows * (uint32_t)cols;
    x[0] = l + 1u - (i + 1u == (uint32_t)rows ? (uint32_t)rows : 0u);
    x[1] = l - 1u + (i == 0u ? (uint32_t)rows : 0u);
    x[2] = l + (uint32_t)rows - (j + 1u == (uint32_t)cols ? wrap : 0u);
    x[3] = l - (uint32_t)rows + (j == 0u ? wrap : 0u);
  };
  const int64_t pos0 = St->pos;
  const int64_t total = n_passes * (int64_t)n_mut + n_steps;
  __syncthreads();
  for (int l = threadIdx.x; l < n; l += OCC_THREADS) {
    if (!(g_lat[l] & 1)) continue;
    uint32_t x[4];
    neighbours((uint32_t)l, x);
    for (int e = 0; e < 4; ++e) add_byte(x[e], 1u);
  }
  __syncthreads();
  if (wave >= 2) {
    walk_producer(L.raw, done, wave - 2, lane, put);
    return;
  }
  if (wave == 1) {
    walk_energy(St, series, series_cap, sample_period, total, false, L.fifo, L.dq, L.dS, L.dM, pub,
                done, lane);
    return;
  }

  int n0[U];  // sites of pair u at occupant 0
#pragma unroll
  for (int u = 0; u < U; ++u) n0[u] = St->occ_cnt0[unit[u]];
  WalkRing ring{(int)pos0};
  uint32_t pushed = 0;
  int64_t remaining = total, step = St->step;
  int seg = 0, left = 0;
  auto ensure = [&](int upto) { ring.ensure(upto, pushed, pub, lane); };
  auto segment_end = [&]() -> bool {
    step += seg;
    remaining -= seg;
    if (step == n_mut) {
      step = 0;
      if (lane == 0) lds_byte(offsetof(OccWalkLds, fifo) + (pushed & (FIFO - 1)), FIFO_PASS_END);
      ++pushed;
    }
    seg = left = (int)(remaining < (int64_t)n_mut - step ? remaining : (int64_t)n_mut - step);
    return remaining > 0;
  };
  // an accepted step of class k at site a (list entry at position pa, last entry la
  // at position pba), by the calling lane
  auto apply = [&](uint32_t a, const uint32_t (&x)[4], uint32_t la, uint32_t pa, uint32_t pba,
                   bool to_one) {
    list[pa] = (uint16_t)la;
    list[pba] = (uint16_t)a;
    add_byte(a, to_one ? 5u : 0u - 5u);
    for (int e = 0; e < 4; ++e) add_byte(x[e], to_one ? 1u : 0xFFFFFFFFu);
  };
  // one step with the full Lemire rejection loop, every lane alike
  auto special_step = [&]() {
    auto next_word = [&]() -> uint64_t {
      ensure(1);
      const uint64_t x = ring.word(L.raw);
      ++ring.rp;
      return x;
    };
    const uint64_t r = record(next_word());
    const uint32_t u1 = (uint32_t)rfl32((int32_t)((uint32_t)r >> 16));
    uint32_t n0u = 0, offu = 0, sizeu = 0;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u1 == (uint32_t)u) {
        n0u = (uint32_t)n0[u];
        offu = (uint32_t)off[u];
        sizeu = (uint32_t)size[u];
      }
    const bool zero = rfl32((int32_t)((uint32_t)r & 0xFFFFu)) < (int32_t)n0u;
    const uint64_t m = zero ? n0u : sizeu - n0u;
    uint64_t xs = next_word();
    const uint64_t th = (0ULL - m) % m;
    while (xs * m < th) xs = next_word();
    const uint32_t slot = (uint32_t)__umul64hi(xs, m);
    const uint32_t pa = zero ? offu + slot : offu + sizeu - 1 - slot;
    const uint32_t pba = offu + n0u - (zero ? 1u : 0u);
    const uint32_t a = list[pa], la = list[pba];
    const uint32_t k = (uint32_t)rfl32((int32_t)cls[a]);
    bool ok = true;
    if ((nd_mask >> k) & 1u) ok = ((uint32_t)rfl32((int32_t)(record(next_word()) >> 32)) >> k) & 1u;
    asm volatile("" ::: "memory");
    if (ok) {
      uint32_t x[4];
      neighbours(a, x);
      if (lane == 0) {
        apply(a, x, la, pa, pba, zero);
        lds_byte(offsetof(OccWalkLds, fifo) + (pushed & (FIFO - 1)), k);
      }
      ++pushed;
#pragma unroll
      for (int u = 0; u < U; ++u) n0[u] += u1 == (uint32_t)u ? (zero ? -1 : 1) : 0;
    }
    asm volatile("" ::: "memory");
    --left;
  };

  WindowStarts<2> starts;
  uint64_t r0 = 0, x1 = 0;
  uint32_t acc2 = 0;
  auto fetch = [&]() {
    const uint32_t at = 8u * (uint32_t)(ring.rp + lane);
    r0 = L.rec[ring.rp + lane];
    x1 = L.x[ring.rp + lane + 1];
    acc2 = *lds_at(at + offsetof(OccWalkLds, rec) + 20);  // the high half two records on
  };
  while (left > 0 || segment_end()) {
    ensure(66);
    fetch();
    for (;;) {
      // the list, its size and the slot under the block-start split
      const uint32_t uu = (uint32_t)r0 >> 16, rr = (uint32_t)r0 & 0xFFFFu;
      uint32_t n0u = (uint32_t)n0[0], offu = (uint32_t)off[0], sizeu = (uint32_t)size[0];
#pragma unroll
      for (int u = 1; u < U; ++u) {
        n0u = uu == (uint32_t)u ? (uint32_t)n0[u] : n0u;
        offu = uu == (uint32_t)u ? (uint32_t)off[u] : offu;
        sizeu = uu == (uint32_t)u ? (uint32_t)size[u] : sizeu;
      }
      const bool zero = rr < n0u;
      const uint32_t m = zero ? n0u : sizeu - n0u;
      const uint64_t p0 = (uint64_t)(uint32_t)x1 * m;
      const uint64_t p1 = (uint64_t)(uint32_t)(x1 >> 32) * m + (p0 >> 32);
      const uint32_t slot = (uint32_t)(p1 >> 32);
      const uint32_t pa = zero ? offu + slot : offu + sizeu - 1u - slot;
      const uint32_t pba = offu + n0u - (zero ? 1u : 0u);
      const uint32_t a = list[pa];
      uint32_t la = list[pba];
      // the low word may be below m: the rejection test (special_step)
      const uint64_t SP = __ballot((uint32_t)p1 == 0u);
      const uint64_t ZERO = __ballot(zero);
      const uint32_t k = cls[a];
      __builtin_amdgcn_sched_barrier(0);
      uint32_t x[4];
      neighbours(a, x);
      asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(la));
      const uint64_t AC = __ballot((acc2 >> k) & 1u);
      const bool nd = (nd_mask >> k) & 1u;
      if (__builtin_expect(SP & 1ull, 0)) {
        special_step();
        break;
      }
      // step starts up to the first accepted one or before the first special one
      uint64_t exec = starts(nd);
      const uint64_t stop = exec & (AC | SP);
      if (stop) {
        const uint64_t f = stop & (0ull - stop);
        exec &= (f - 1ull) | (f & ~SP);
      }
      int steps = __popcll(exec);
      if (__builtin_expect(steps > left, 0)) {
        uint64_t rest = exec;
        for (int r = 0; r < left; ++r) rest &= rest - 1;
        exec ^= rest;
        steps = left;
      }
      const int last = 63 - __builtin_clzll(exec);
      ring.rp += last + 2 + (int)((__ballot(nd) >> last) & 1ull);
      left -= steps;
      const bool more = ((ring.end - 66 - ring.rp) | (left - 1)) >= 0;
      const uint64_t F = (1ull << last) & AC;  // only the last step can be accepted
      uint32_t uf = 0;
      if (U > 1) uf = (uint32_t)__builtin_amdgcn_readlane((int)uu, last);
      if (more) fetch();
      asm volatile("" ::: "memory");
      if (F) {
        if (__builtin_amdgcn_inverse_ballot_w64(F)) {
          apply(a, x, la, pa, pba, zero);
          lds_byte(offsetof(OccWalkLds, fifo) + (pushed & (FIFO - 1)), k);
        }
        ++pushed;
        const int dn = (ZERO >> last) & 1ull ? -1 : 1;
#pragma unroll
        for (int u = 0; u < U; ++u) n0[u] += uf == (uint32_t)u ? dn : 0;
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
  for (int i = lane; i < n; i += 64)
    if (cls[i] < OCC_FIXED_CLASS) g_lat[i] = (int8_t)((cls[i] / 5) & 1);
  for (int i = lane; i < n_mut; i += 64) g_list[i] = (int32_t)list[i];
  if (lane == 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) St->occ_cnt0[unit[u]] = n0[u];
    St->pos = p_fin;
    St->step = step;
    St->frozen = 0;
  }
}

void launch_occupant(const OccParams *P, const OccTables *T, ExactState *S, int8_t *lat_pool,
                     int32_t *list_pool, const int8_t *asym_pool, mcg_sample *series,
                     int64_t series_cap, const uint8_t *active, int n_chains, int64_t n_passes,
                     int64_t n_steps, int64_t sample_period, bool canonical, int n_swaps,
                     int sgc_units, int lds_bytes, hipStream_t stream) {
#define MCG_OCC_ANY(CANONICAL, NS)                                                                  \
  hipLaunchKernelGGL((occupant_kernel<CANONICAL, NS>), dim3(n_chains), dim3(128), lds_bytes, stream, \
                     P, T, S, lat_pool, list_pool, series, series_cap, active, n_passes, n_steps,   \
                     sample_period)
#define MCG_OCC_SGC(U)                                                                            \
  hipLaunchKernelGGL(occupant_sgc_kernel<U>, dim3(n_chains), dim3(OCC_THREADS), lds_bytes, stream, \
                     P, T, S, lat_pool, list_pool, asym_pool, series, series_cap, active, n_passes, \
                     n_steps, sample_period)
  if (sgc_units == 1)
    MCG_OCC_SGC(1);
  else if (sgc_units == 2)
    MCG_OCC_SGC(2);
  else if (sgc_units == 3)
    MCG_OCC_SGC(3);
  else if (canonical && n_swaps <= 4)
    MCG_OCC_ANY(true, 4);
  else if (canonical)
    MCG_OCC_ANY(true, OCC_MAX_SWAPS);
  else if (n_swaps <= 4)
    MCG_OCC_ANY(false, 4);
  else
    MCG_OCC_ANY(false, OCC_MAX_SWAPS);
#undef MCG_OCC_ANY
#undef MCG_OCC_SGC
}

hipError_t occupant_set_max_lds(int general_bytes, int sgc_bytes) {
  const void *any[] = {reinterpret_cast<const void *>(occupant_kernel<true, 4>),
                       reinterpret_cast<const void *>(occupant_kernel<true, OCC_MAX_SWAPS>),
                       reinterpret_cast<const void *>(occupant_kernel<false, 4>),
                       reinterpret_cast<const void *>(occupant_kernel<false, OCC_MAX_SWAPS>)};
  hipError_t e = hipSuccess;
  for (const void *f : any)
    if (e == hipSuccess)
      e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, general_bytes);
  const void *sgc[] = {reinterpret_cast<const void *>(occupant_sgc_kernel<1>),
                       reinterpret_cast<const void *>(occupant_sgc_kernel<2>),
                       reinterpret_cast<const void *>(occupant_sgc_kernel<3>)};
  for (const void *f : sgc)
    if (e == hipSuccess) e = set_dynamic_lds(f, sgc_bytes, true);
  return e;
}

}  // namespace mcg
