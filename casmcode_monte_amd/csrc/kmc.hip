// kmc.hip -- KMC mode: kinetic Monte Carlo with atom tracking for a square
// lattice gas, bit for bit the loop of kinetic_monte_carlo.hh:136-229 under a
// rejection event selector, by one walking wavefront per chain.  In kmc_kernel a
// second one twists the engine's next generation meanwhile (mt_producer, walk.hh);
// kmc_walk_kernel has four more waves.
//
// Model: occupant 0 = vacancy, 1 = atom, E = -J sum over nearest-neighbour
// bonds of n_i n_j.  Selector: attempts follow one another at 1/R, R = 4 *
// (number of atoms); an attempt chooses an atom uniformly from the
// OccLocation list of atoms (one Lemire word, OccLocation.hh:257-261) and a
// direction (random_int(3): one word, its top two bits), is rejected when the
// target holds an atom, and otherwise is accepted without a draw when
// dE = J (a - b) <= 0 (a, b: atoms next to the origin other than at the
// target, next to the target other than at the origin), else when one more
// canonical word falls below exp(-beta dE) (a per-class word threshold from
// the host).  The accepted attempt is the selected event, with time increment
// fl(k / R) for the k attempts it took; the loop's time is the running FP64
// sum of the increments in event order.
//
// Device OccLocation with atom tracking (OccLocation.cc:39-118, 216-330): one
// 16-bit list array holds the vacancy list from the front and the atom list
// from the back (slot j at n - 1 - j); each site has its position in that
// array and the id of its atom (0xFFFF for none); each atom its displacement
// since the start and its jump count.  An event's two transforms (origin
// 1 -> 0, then target 0 -> 1) and the atom's move are six LDS writes.
//
// Block walk: lane t evaluates stream position P+t as if an attempt started
// there, from the block-start state.  Rejected attempts change nothing but the
// clock, and an accepted hop changes only what a later attempt reads at its
// own slots and sites, so the block commits every attempt up to the first one
// an earlier accepted hop changes and starts again after them.
#include <cstddef>

#include "internal.hh"
#include "walk.hh"

namespace mcg {

namespace {

constexpr uint16_t NO_ATOM = 0xFFFFu;

__device__ __forceinline__ uint32_t kmc_nbr(uint32_t l, int d, int32_t rows, int32_t cols,
                                            uint64_t magic) {
  const uint32_t j = (uint32_t)(((uint64_t)l * magic) >> 40);
  const uint32_t i = l - j * (uint32_t)rows;
  switch (d) {
    case 0: return ((i + 1 == (uint32_t)rows) ? 0u : i + 1) + (uint32_t)rows * j;
    case 1: return ((i == 0) ? (uint32_t)rows - 1 : i - 1) + (uint32_t)rows * j;
    case 2: return i + (uint32_t)rows * ((j + 1 == (uint32_t)cols) ? 0u : j + 1);
    default: return i + (uint32_t)rows * ((j == 0) ? (uint32_t)cols - 1 : j - 1);
  }
}

// One attempt evaluated from a state: the atom's list slot and position, the
// origin and target, whether the target is free, the class a - b + 3, the
// atom and its displacement.
struct Attempt {
  int32_t pa;        // list position of the atom's slot
  uint32_t from, to;
  int dir;
  bool free;         // the target is a vacancy
  int cls;           // a - b + 3
  uint32_t atom;
  int32_t dx, dy;
};

__device__ __forceinline__ void kmc_eval(Attempt &at, uint32_t slot, int dir, int32_t n,
                                         const uint16_t *list, const uint16_t *site_atom,
                                         const int32_t *adx, const int32_t *ady, int32_t rows,
                                         int32_t cols, uint64_t magic) {
  at.pa = n - 1 - (int32_t)slot;
  at.from = list[at.pa];
  at.dir = dir;
  at.to = kmc_nbr(at.from, dir, rows, cols, magic);
  at.atom = site_atom[at.from];
  at.free = site_atom[at.to] == NO_ATOM;
  int a = 0, b = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t x = kmc_nbr(at.from, e, rows, cols, magic);
    const uint32_t y = kmc_nbr(at.to, e, rows, cols, magic);
    a += (x != at.to && site_atom[x] != NO_ATOM) ? 1 : 0;
    b += (y != at.from && site_atom[y] != NO_ATOM) ? 1 : 0;
  }
  at.cls = a - b + 3;
  at.dx = adx[at.atom];
  at.dy = ady[at.atom];
}

// OccLocation::apply for the two transforms (origin 1 -> 0, target 0 -> 1)
// and the atom's move, by one lane.  The atom list's last entry moves into the
// origin's slot, the origin takes the vacancy list's new last place, the
// vacancy list's last entry (now the origin) moves into the target's slot, and
// the target takes the atom list's new last place: the same position pba.
__device__ __forceinline__ void kmc_apply(const Attempt &at, int32_t pba, uint16_t *list,
                                          uint16_t *pos, uint16_t *site_atom, int32_t *adx,
                                          int32_t *ady, int32_t *ajump) {
  const int32_t pt = pos[at.to];
  const uint16_t back = list[pba];
  list[at.pa] = back;
  pos[back] = (uint16_t)at.pa;
  list[pt] = (uint16_t)at.from;
  pos[at.from] = (uint16_t)pt;
  list[pba] = (uint16_t)at.to;
  pos[at.to] = (uint16_t)pba;
  site_atom[at.from] = NO_ATOM;
  site_atom[at.to] = (uint16_t)at.atom;
  adx[at.atom] = at.dx + (at.dir == 0 ? 1 : at.dir == 1 ? -1 : 0);
  ady[at.atom] = at.dy + (at.dir == 2 ? 1 : at.dir == 3 ? -1 : 0);
  ajump[at.atom] += 1;
}

}  // namespace

__global__ __launch_bounds__(128) void kmc_kernel(const KmcParams *__restrict__ Pp,
                                                 ExactState *__restrict__ Sp,
                                                 int8_t *__restrict__ lat_pool,
                                                 int32_t *__restrict__ list_pool,
                                                 int32_t *__restrict__ atom_pool,
                                                 KmcHop *__restrict__ hop_pool,
                                                 int32_t *__restrict__ hop_count_pool,
                                                 mcg_sample *__restrict__ series,
                                                 int64_t series_cap,
                                                 const uint8_t *__restrict__ active,
                                                 int64_t n_passes, int64_t n_steps,
                                                 int64_t sample_period, double stop_time,
                                                 int select_at_end) {
  const int c = blockIdx.x;
  if (!active[c]) return;
  const int lane = threadIdx.x & 63;
  const bool producer = threadIdx.x >= 64;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ uint64_t raw[3][MT_N];
  __shared__ uint64_t ring[3][MT_N];
  __shared__ int done;
  __shared__ uint64_t thr_s[KMC_NCLASS];

  const KmcParams *P = Pp + c;
  ExactState *St = Sp + c;
  const int32_t rows = P->rows, cols = P->cols, n = P->n, n_atoms = P->n_atoms;
  const int W = P->window;
  const uint64_t magic = P->div_magic;
  const double R = P->attempt_rate, period = P->time_period;
  int8_t *g_lat = lat_pool + P->lat_off;
  int32_t *g_list = list_pool + P->lat_off;
  int32_t *g_atoms = atom_pool + 4 * P->lat_off;  // per atom: site, dx, dy, jumps
  const int a_al = (n + 7) & ~7;
  uint16_t *list = reinterpret_cast<uint16_t *>(smem);
  uint16_t *pos = list + a_al;
  uint16_t *site_atom = pos + a_al;
  int32_t *adx = reinterpret_cast<int32_t *>(site_atom + a_al);
  int32_t *ady = adx + a_al;
  int32_t *ajump = ady + a_al;

  if (!producer) {
    for (int i = lane; i < MT_N; i += 64) {
      raw[0][i] = St->mt[i];
      ring[0][i] = mt_temper(raw[0][i]);
    }
    if (lane < KMC_NCLASS) thr_s[lane] = P->thr[lane];
    for (int i = lane; i < n; i += 64) {
      const uint16_t l = (uint16_t)g_list[i];
      list[i] = l;
      pos[l] = (uint16_t)i;
      site_atom[i] = NO_ATOM;
    }
    for (int i = lane; i < n_atoms; i += 64) {
      adx[i] = g_atoms[4 * i + 1];
      ady[i] = g_atoms[4 * i + 2];
      ajump[i] = g_atoms[4 * i + 3];
    }
    if (lane == 0) done = 0;
  }
  __syncthreads();
  if (!producer)
    for (int i = lane; i < n_atoms; i += 64) site_atom[g_atoms[4 * i]] = (uint16_t)i;
  __syncthreads();
  if (producer) {  // wave 1 twists the engine (walk.hh); wave 0 walks
    mt_producer(raw, ring, &done, lane);
    return;
  }

  const int64_t pos0 = St->pos;
  int64_t ps = pos0;
  MtRing3 eng;
  int64_t n_pass = St->n_pass, n_acc = St->n_accept, n_rej = St->n_reject;
  int64_t S = St->S, n_samples = St->n_samples;
  int64_t sum_sq = St->kmc_sum_sq, sum_dx = St->kmc_sum_dx, sum_dy = St->kmc_sum_dy;
  int64_t k_run = St->kmc_k;  // attempts since the last event
  double time = St->time;
  int64_t next_k = St->next_k;
  int64_t step = St->step;
  int64_t frozen = 0;
  const uint32_t draw_mask = P->draw_mask, full_mask = P->full_mask;
  const int64_t spin_limit = P->spin_limit;
  const int32_t pba = n - n_atoms;  // the atom list's last position (fixed: hops keep the count)
  const int64_t target = n_passes * (int64_t)n + n_steps;
  int64_t done_ev = 0;
  int64_t pending_site = St->pending_site, pending_dir = St->kmc_pdir, pending_k = St->kmc_pk;
  double pending_time = St->pending_dt;

  auto ensure = [&](int64_t upto) { eng.ensure(upto); };
  const uint64_t *ringf = &ring[0][0];
  auto word = [&](int64_t q) -> uint64_t { return ringf[eng.index(q)]; };
  auto lemire_scalar = [&](uint64_t m) -> uint32_t {
    ensure(ps + 1);
    uint64_t x = word(ps);
    ++ps;
    uint64_t lo = x * m, hi = __umul64hi(x, m);
    if (lo < m) {
      const uint64_t th = (0ULL - m) % m;
      while (lo < th) {
        ensure(ps + 1);
        x = word(ps);
        ++ps;
        lo = x * m;
        hi = __umul64hi(x, m);
      }
    }
    return (uint32_t)hi;
  };
  auto record = [&](int64_t pass_field, double t) {
    if (lane == 0 && n_samples < series_cap) {
      mcg_sample rec = {};
      rec.pass = pass_field;
      rec.S1 = S;
      rec.M = n_atoms;
      rec.S2 = sum_sq;
      rec.S3 = sum_dx;
      rec.T3 = sum_dy;
      rec.time = t;
      series[(int64_t)c * series_cap + n_samples] = rec;
    }
    ++n_samples;
  };
  // the executed event's bookkeeping (all lanes, uniform): time-grid samples
  // it reaches (before it applies), its time, bond and displacement sums
  auto account = [&](int64_t k_ev, int cls, int dir, int32_t dx, int32_t dy) {
    const double event_time = __dadd_rn(time, __ddiv_rn((double)k_ev, R));
    if (period > 0.0)
      while (event_time >= __dmul_rn((double)next_k, period)) {
        record(n_pass * (int64_t)n + step, __dmul_rn((double)next_k, period));
        ++next_k;
      }
    time = event_time;
    S += 3 - cls;  // b - a
    const int ddx = dir == 0 ? 1 : dir == 1 ? -1 : 0, ddy = dir == 2 ? 1 : dir == 3 ? -1 : 0;
    sum_dx += ddx;
    sum_dy += ddy;
    sum_sq += 2 * (int64_t)dx * ddx + 2 * (int64_t)dy * ddy + 1;
  };

  // hop correlations: after an atom's hop (by the lane that applied it, time
  // already the event's, step and pass still the event's own), its
  // displacement when its jump count is a multiple of hop_every
  const int32_t hop_every = P->hop_every, hop_max = P->hop_max;
  auto hop_record = [&](int32_t atom) {
    if (hop_every <= 0 || ajump[atom] % hop_every != 0) return;
    int32_t *cnt = hop_count_pool + P->lat_off;
    const int32_t k = cnt[atom];
    if (k >= hop_max) return;
    KmcHop r;
    r.dx = adx[atom];
    r.dy = ady[atom];
    r.step = step;
    r.pass = n_pass;
    r.time = time;
    hop_pool[P->hop_off + (int64_t)k * n + atom] = r;
    cnt[atom] = k + 1;
  };

  // a selected event: left pending (its site, direction, attempts and time
  // kept for the next launch) or applied
  bool stopped = false;
  auto pend = [&](uint32_t from, int dir, int64_t k, double event_time) {
    pending_site = from;
    pending_dir = dir;
    pending_k = k;
    pending_time = event_time;
    stopped = true;
  };
  auto bump = [&]() {
    ++n_acc;
    ++step;
    ++done_ev;
    if (step == n) {
      step = 0;
      ++n_pass;
      if (period <= 0.0 && n_pass % sample_period == 0) record(n_pass, time);
    }
  };

  // the event selected at the end of the previous launch comes first
  if (pending_site >= 0 && n_atoms > 0) {
    if (pending_time >= stop_time) {
      stopped = true;
    } else {
      Attempt a0;
      const uint32_t from = (uint32_t)pending_site;
      kmc_eval(a0, (uint32_t)(n - 1 - (int32_t)pos[from]), pending_dir, n, list, site_atom, adx,
               ady, rows, cols, magic);
      account(pending_k, a0.cls, a0.dir, a0.dx, a0.dy);
      if (lane == 0) {
        kmc_apply(a0, pba, list, pos, site_atom, adx, ady, ajump);
        hop_record(a0.atom);
      }
      asm volatile("" ::: "memory");
      pending_site = -1;
      bump();
    }
  }

  while (!stopped && n_atoms > 0) {
    // past the target: select one more event and leave it pending, if asked
    const bool select_only = done_ev >= target;
    if (select_only && !select_at_end) break;
    ensure(ps + W + 2);
    const bool inwin = lane < W;
    const int64_t q = inwin ? ps + lane : ps;
    const uint64_t x1 = word(q), x2 = word(q + 1), x3 = word(q + 2);
    const uint64_t na = (uint64_t)n_atoms;
    const uint32_t slot = (uint32_t)__umul64hi(x1, na);
    const bool special = inwin && (x1 * na) < na;
    Attempt at;
    kmc_eval(at, slot, (int)(x2 >> 62), n, list, site_atom, adx, ady, rows, cols, magic);
    // dE > 0 draws a word (draw_mask); all words may accept (full_mask)
    const bool nd = at.free && ((draw_mask >> at.cls) & 1u);
    const bool acc =
        at.free && (!((draw_mask >> at.cls) & 1u) || ((full_mask >> at.cls) & 1u) || x3 < thr_s[at.cls]);
    const bool valid = inwin && !special;
    const uint64_t ND = __ballot(valid && nd);
    const uint64_t AC = __ballot(valid && acc);
    const uint64_t SP = __ballot(special);

    // attempt starts over the window: 0, then +2 or +3 (a uniform drawn), up
    // to the first special one
    const uint64_t A = window_starts2(ND, SP, 0ull, W);
    // An attempt evaluated from the block-start state stays exact until an
    // earlier accepted hop changes what it reads: the hop rewrites its own
    // list slot and the atom list's last slot, and changes its origin and
    // target sites.  So an attempt is hit when its slot is one of those two,
    // or its origin, target or their neighbours include the hop's origin or
    // target (its class, its free target and its atom are read there).  The
    // block runs up to the first hit attempt; hits found from accepted lanes
    // past it change nothing.  A window without an accepted attempt skips all
    // of this.
    const uint64_t AA = A & AC;
    uint64_t exec = A;
    if (AA & (AA - 1ull) ? true : (AA && (A >> __builtin_ctzll(AA)) > 1ull)) {
      uint32_t nf[4], ntg[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        nf[e] = kmc_nbr(at.from, e, rows, cols, magic);
        ntg[e] = kmc_nbr(at.to, e, rows, cols, magic);
      }
      const bool is_att = (A >> lane) & 1ull;
      bool hit = false;
      uint64_t HIT = 0;
      for (uint64_t rem = AA; rem; rem &= rem - 1) {
        const int e = __builtin_ctzll(rem);
        if (HIT & ((1ull << e) - 1)) break;  // past the first hit attempt
        const int32_t pa_e = __builtin_amdgcn_readlane(at.pa, e);
        const uint32_t fe = (uint32_t)__builtin_amdgcn_readlane((int)at.from, e);
        const uint32_t te = (uint32_t)__builtin_amdgcn_readlane((int)at.to, e);
        bool h = at.pa == pa_e || at.pa == pba || at.from == fe || at.from == te ||
                 at.to == fe || at.to == te;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          h = h || nf[k] == fe || nf[k] == te || ntg[k] == fe || ntg[k] == te;
        hit = hit || (lane > e && h);
        HIT = __ballot(is_att && hit);
      }
      if (HIT) exec = A & ((1ull << __builtin_ctzll(HIT)) - 1);
    }

    // the attempts in order: rejected ones (counted in bulk between events)
    // add to the next event's increment; accepted ones are the events,
    // applied in order by their lanes (their slots and sites are disjoint from
    // every later attempt run here)
    int64_t kk = k_run;
    int last = -1;
    int attempts = 0;
    uint64_t consumed = 0;
    bool cut = false;
    for (uint64_t ev = exec & AC; ev; ev &= ev - 1) {
      const int t = __builtin_ctzll(ev);
      const uint64_t upto = t == 63 ? ~0ull : ((2ull << t) - 1ull);
      const uint64_t span = exec & upto & ~consumed;  // attempts since the last event, with t
      const int cnt = __popcll(span);
      consumed |= span;
      kk += cnt;
      attempts += cnt;
      n_rej += cnt - 1;
      last = t;
      const int cls = __builtin_amdgcn_readlane(at.cls, t);
      const int dir = __builtin_amdgcn_readlane(at.dir, t);
      const int32_t dx = __builtin_amdgcn_readlane(at.dx, t), dy = __builtin_amdgcn_readlane(at.dy, t);
      const uint32_t from = __builtin_amdgcn_readlane((int)at.from, t);
      const double event_time = __dadd_rn(time, __ddiv_rn((double)kk, R));
      if (done_ev >= target || event_time >= stop_time) {
        pend(from, dir, kk, event_time);
        kk = 0;
        cut = true;
        break;
      }
      account(kk, cls, dir, dx, dy);
      if (lane == t) {
        kmc_apply(at, pba, list, pos, site_atom, adx, ady, ajump);
        hop_record(at.atom);
      }
      asm volatile("" ::: "memory");
      bump();
      kk = 0;
      if (done_ev >= target && !select_at_end) {  // the launch's events are done
        cut = true;
        break;
      }
    }
    if (!cut) {  // rejected attempts after the last event
      const uint64_t rest = exec & ~consumed;
      const int cnt = __popcll(rest);
      kk += cnt;
      attempts += cnt;
      n_rej += cnt;
      if (rest) last = 63 - __builtin_clzll(rest);
    }
    k_run = kk;
    if (last >= 0) ps += last + 2 + (int)((ND >> last) & 1ull);

    if (!stopped && (SP & 1ull) && attempts == 0) {
      // an attempt whose Lemire draw may reject, with the full rejection loop;
      // every lane computes it, lane 0 writes
      const uint32_t s1 = lemire_scalar(na);
      ensure(ps + 1);
      const int d1 = (int)(word(ps) >> 62);
      ++ps;
      Attempt a1;
      kmc_eval(a1, s1, d1, n, list, site_atom, adx, ady, rows, cols, magic);
      bool ok = a1.free;
      if (a1.free && ((draw_mask >> a1.cls) & 1u)) {
        ensure(ps + 1);
        const uint64_t xr = word(ps);
        ++ps;
        ok = ((full_mask >> a1.cls) & 1u) || xr < thr_s[a1.cls];
      }
      ++k_run;
      // one wavefront walks: its LDS operations execute in issue order
      asm volatile("" ::: "memory");
      if (ok) {
        const double event_time = __dadd_rn(time, __ddiv_rn((double)k_run, R));
        if (select_only || event_time >= stop_time) {
          pend(a1.from, a1.dir, k_run, event_time);
        } else {
          account(k_run, a1.cls, a1.dir, a1.dx, a1.dy);
          if (lane == 0) {
            kmc_apply(a1, pba, list, pos, site_atom, adx, ady, ajump);
            hop_record(a1.atom);
          }
          asm volatile("" ::: "memory");
          bump();
        }
        k_run = 0;
      } else {
        ++n_rej;
      }
    }
    // no event in spin_limit attempts (every move of the state has a
    // vanishing probability): stop instead of spinning
    if (k_run > spin_limit) {
      frozen = 1;
      break;
    }
  }

  // release the producer (it waits at the barrier this one matches)
  eng.finish(&done, lane);
  int64_t g_fin = 0, p_fin = pos0;
  if (ps != pos0) {
    g_fin = (ps - 1) / MT_N;
    p_fin = ps - (int64_t)MT_N * g_fin;
  }
  for (int i = lane; i < MT_N; i += 64) St->mt[i] = raw[g_fin % 3][i];
  for (int i = lane; i < n; i += 64) {
    g_list[i] = (int32_t)list[i];
    g_lat[i] = site_atom[i] == NO_ATOM ? (int8_t)0 : (int8_t)1;
    const uint16_t a = site_atom[i];
    if (a != NO_ATOM) {
      g_atoms[4 * a + 0] = (int32_t)i;
      g_atoms[4 * a + 1] = adx[a];
      g_atoms[4 * a + 2] = ady[a];
      g_atoms[4 * a + 3] = ajump[a];
    }
  }
  if (lane == 0) {
    St->pos = p_fin;
    St->n_pass = n_pass;
    St->n_accept = n_acc;
    St->n_reject = n_rej;
    St->S = S;
    St->M = n_atoms;
    St->n_samples = n_samples;
    St->step = step;
    St->time = time;
    St->next_k = next_k;
    St->kmc_k = k_run;
    St->kmc_sum_sq = sum_sq;
    St->kmc_sum_dx = sum_dx;
    St->kmc_sum_dy = sum_dy;
    St->frozen = frozen;
    St->pending_site = pending_site;
    St->pending_dt = pending_time;
    St->kmc_pdir = pending_dir;
    St->kmc_pk = pending_k;
  }
}

// ---------------------------------------------------------------------------
// Runs of whole counts of events (no stop time, nothing pending, no hop
// correlations): the same chain with the state-independent work on other waves,
// as in the EXACT block walk (exact.hip).
//
// The number of atoms is fixed, so waves 2-4 turn each engine word into a record:
// the list entry it chooses as an atom, its direction, and which of the seven
// classes it accepts.  A site is one word -- atom id, place in the list, occupant,
// atoms next to it -- so an attempt reads one list entry and two words, its class
// is a difference of two counts, and a hop is nine adds to words (they commute, and
// no field leaves its range) and three list entries; all hops of a block apply at
// once.  Wave 1 takes the events in order: their times (FP64, in order), the
// atoms' displacements, the sums and the records.
//
// Conflicts: positions that would hop mark the eight sites whose words they
// change (beside each word; 64 * epoch + lane as in exact.hip); an attempt whose
// origin or target holds a lower lane of this block stops it.  The atom list's
// last entry changes with every hop.
//
// Measured on MI355X, 64 chains of 64x64 sites at 8 T x 8 densities, 40960 events
// each: 50.9 ms by kmc_kernel, 9.5 ms here (the slowest chain, 440000 attempts: 51
// cycles an attempt at 2.4 GHz; at 1.2 attempts an event 107 cycles an event; ~235
// instructions a block of ~27 attempts, which one wave issues in ~5 cycles each).
// 1024 such chains 3 passes: 54.3 and 8.8 ms; one 12x12 chain: 24.0 and 4.0 ms per
// 100 passes; 600 chains of 80x80: 41.7 and 6.6 ms.
// ---------------------------------------------------------------------------
namespace {

constexpr int KMC_WALK_THREADS = 5 * 64;
constexpr int KMC_FIFO = 1024;  // events and pass ends; walk_energy's bound, per two words
constexpr uint32_t KMC_PASS_END = 1u << 31;
constexpr uint32_t KMC_NO_MARK = 0xFFFFFFFFu;
constexpr uint32_t KMC_FIRST_EPOCH = KMC_NO_MARK / 64u - 1u;
// fields of a site's word
constexpr int KMC_POS = 13, KMC_CNT = 26, KMC_OCC = 29;

// A direction's constants, sites being byte addresses (8 l), coordinates in units of
// 8 along i and of 1 along j: the step and the wrapped one, the coordinate at which
// it wraps, the one whose target is there, and the one at the line's other end;
// across it, the step up, the wrapped one and the last coordinate
struct KmcDir {
  uint32_t step, wrap, edge, next;
  uint32_t far, up, up_wrap, up_edge;
};

// fixed LDS parts at address 0; the sites (word, mark), the list and the atoms follow
struct KmcWalkLds {
  // bits 0-16 list entry's address, 17-18 direction, 19-25 accepted classes, 31
  // the Lemire draw may reject
  uint32_t rec[REC_RING + REC_MIRROR];
  uint64_t raw[3][MT_N];
  uint32_t cum[KMC_FIFO];   // attempts of the launch up to the event, modulo 2^32
  uint32_t what[KMC_FIFO];  // atom | direction << 13 | class << 15, or KMC_PASS_END
  uint32_t tos[64];         // a block's targets, in order
  KmcDir dir[4];            // along i: 0 +, 1 -; along j: 2 +, 3 -
  uint32_t done, pub;
  uint32_t tail;            // attempts after the launch's last event
};
static_assert(sizeof(KmcWalkLds) <= KMC_WALK_FIXED_LDS, "the words start behind it");

// Wave 1: see above.  x, y, jumps: the atoms'.
__device__ inline void kmc_account(const KmcParams *P, ExactState *St, int32_t *g_atoms,
                                   mcg_sample *__restrict__ series, int64_t series_cap,
                                   int64_t sample_period, const KmcWalkLds &L, int32_t *x,
                                   int32_t *y, int32_t *jumps, const volatile lds_u32 *pub,
                                   const volatile lds_u32 *done, int lane) {
  const double R = P->attempt_rate, period = P->time_period;
  const bool grid = period > 0.0;
  double time = St->time;
  int64_t next_k = St->next_k, n_pass = St->n_pass, n_samples = St->n_samples;
  int64_t S = St->S, sq = St->kmc_sum_sq, sx = St->kmc_sum_dx, sy = St->kmc_sum_dy;
  int64_t aS = 0, asq = 0, ax = 0, ay = 0;  // this lane's share since the last reduction
  const int64_t ev0 = n_pass * (int64_t)P->n + St->step;
  int64_t n_ev = 0, carry = St->kmc_k;  // attempts before the launch, since the last event
  int64_t attempts = 0;                 // this lane's share, of the launch
  uint32_t head = 0;
  int nbar = 0;
  auto record = [&](int64_t pass_field, double t) {
    S += walk_sum(aS);
    sq += walk_sum(asq);
    sx += walk_sum(ax);
    sy += walk_sum(ay);
    aS = asq = ax = ay = 0;
    if (lane == 0 && n_samples < series_cap) {
      mcg_sample rec = {};
      rec.pass = pass_field;
      rec.S1 = S;
      rec.M = P->n_atoms;
      rec.S2 = sq;
      rec.S3 = sx;
      rec.T3 = sy;
      rec.time = t;
      series[n_samples] = rec;
    }
    ++n_samples;
  };
  for (bool last = false; !last;) {
    __syncthreads();
    last = rfl32((int32_t)*done) == ++nbar;
    const uint32_t end = (uint32_t)rfl32((int32_t)*pub);
    asm volatile("" ::: "memory");  // the entries are read after the count
    while (end != head) {
      const uint32_t left = end - head;
      if (left < 64u && !last) break;
      const int m = left < 64u ? (int)left : 64;
      const uint32_t at = (head + (uint32_t)lane) & (KMC_FIFO - 1);
      const uint32_t v = L.what[at];
      const bool event = lane < m && !(v & KMC_PASS_END);
      int64_t k = (int64_t)(uint32_t)(L.cum[at] - L.cum[(at - 1u) & (KMC_FIFO - 1)]);
      attempts += event ? k : 0;
      if (lane == 0) k += carry;  // (a launch's first entry is an event)
      carry = 0;
      const double q = event ? __ddiv_rn((double)k, R) : 0.0;  // (a time plus 0 is itself)
      const uint64_t EV = __ballot(event);
      const uint64_t ENDS = __ballot(lane < m && !event);
      // lanes [from, to) of the events: sums and displacements.  An atom that hops
      // twice: whatever order the two adds take, the sum of squares telescopes
      auto add = [&](int from, int to) {
        if (event && lane >= from && lane < to) {
          const uint32_t atom = v & 0x1FFFu, dir = (v >> KMC_POS) & 3u;
          const int d = dir & 1u ? -1 : 1;
          const int32_t was = atomicAdd((dir < 2u ? x : y) + atom, d);
          atomicAdd(jumps + atom, 1);
          aS += 3 - (int)((v >> 15) & 7u);
          asq += 2 * (int64_t)was * d + 1;
          ax += dir < 2u ? d : 0;
          ay += dir < 2u ? 0 : d;
        }
      };
      double t = time;
#pragma unroll
      for (int j = 0; j < 64; ++j) t = __dadd_rn(t, readlane_f64(q, j));
      int from = 0;
      if (grid ? t >= __dmul_rn((double)next_k, period) : ENDS != 0) {
        // every event's own time
        double mine = time, u = time;
        for (int j = 0; j < m; ++j) {
          u = __dadd_rn(u, readlane_f64(q, j));
          mine = lane >= j ? u : mine;
        }
        if (grid) {
          // a grid time is recorded before the first event that reaches it
          for (;;) {
            const uint64_t G = __ballot(event && mine >= __dmul_rn((double)next_k, period));
            if (!G) break;
            const int e = __builtin_ctzll(G);
            add(from, e);
            from = e;
            record(ev0 + n_ev + __popcll(EV & ((1ull << e) - 1ull)),
                   __dmul_rn((double)next_k, period));
            ++next_k;
          }
        } else {
          for (uint64_t rem = ENDS; rem; rem &= rem - 1) {
            if ((n_pass + 1 + __popcll(ENDS & ((rem & -rem) - 1))) % sample_period) continue;
            const int e = __builtin_ctzll(rem);
            add(from, e);
            from = e;
            record(n_pass + 1 + __popcll(ENDS & ((1ull << e) - 1ull)), readlane_f64(mine, e));
          }
        }
      }
      add(from, 64);
      time = t;
      n_pass += __popcll(ENDS);
      n_ev += __popcll(EV);
      head += (uint32_t)m;
    }
  }
  S += walk_sum(aS);
  sq += walk_sum(asq);
  sx += walk_sum(ax);
  sy += walk_sum(ay);
  attempts = walk_sum(attempts) + L.tail;
  for (int a = lane; a < P->n_atoms; a += 64) {
    g_atoms[4 * a + 1] = x[a];
    g_atoms[4 * a + 2] = y[a];
    g_atoms[4 * a + 3] = jumps[a];
  }
  if (lane == 0) {
    St->n_pass = n_pass;
    St->n_accept += n_ev;
    St->n_reject += attempts - n_ev;
    St->S = S;
    St->M = P->n_atoms;
    St->n_samples = n_samples;
    St->time = time;
    St->next_k = next_k;
    St->kmc_sum_sq = sq;
    St->kmc_sum_dx = sx;
    St->kmc_sum_dy = sy;
  }
}

}  // namespace

__global__ __launch_bounds__(KMC_WALK_THREADS) void kmc_walk_kernel(
    const KmcParams *__restrict__ Pp, ExactState *__restrict__ Sp, int8_t *__restrict__ lat_pool,
    int32_t *__restrict__ list_pool, int32_t *__restrict__ atom_pool,
    mcg_sample *__restrict__ series, int64_t series_cap, const uint8_t *__restrict__ active,
    int64_t n_passes, int64_t n_steps, int64_t sample_period) {
  const int c = blockIdx.x;
  if (!active[c]) return;
  const int lane = threadIdx.x & 63;
  const int wave = rfl32(threadIdx.x >> 6);
  extern __shared__ __align__(16) unsigned char smem[];

  const KmcParams *P = Pp + c;
  ExactState *St = Sp + c;
  const uint32_t rows = (uint32_t)P->rows, cols = (uint32_t)P->cols, n = (uint32_t)P->n;
  const uint32_t n_atoms = (uint32_t)P->n_atoms;
  int8_t *g_lat = lat_pool + P->lat_off;
  int32_t *g_list = list_pool + P->lat_off;
  int32_t *g_atoms = atom_pool + 4 * P->lat_off;  // per atom: site, dx, dy, jumps
  KmcWalkLds &L = *reinterpret_cast<KmcWalkLds *>(smem);
  volatile lds_u32 *done = lds_at(offsetof(KmcWalkLds, done));
  volatile lds_u32 *pub = lds_at(offsetof(KmcWalkLds, pub));
  const uint32_t n8 = (n + 7u) & ~7u;
  const uint32_t list_base = KMC_WALK_FIXED_LDS + 8u * n8;
  uint32_t *site = reinterpret_cast<uint32_t *>(smem + KMC_WALK_FIXED_LDS);  // word, mark
  uint16_t *list = reinterpret_cast<uint16_t *>(smem + list_base);  // 8 site, as an address
  int32_t *ax = reinterpret_cast<int32_t *>(smem + list_base + 2u * n8);
  int32_t *ay = ax + n8, *ajump = ay + n8;

  const uint32_t draw_mask = P->draw_mask, always = ~draw_mask | P->full_mask;
  uint64_t thr[KMC_NCLASS];
#pragma unroll
  for (int k = 0; k < KMC_NCLASS; ++k) thr[k] = P->thr[k];
  auto record = [&](uint64_t x) -> uint32_t {
    const uint32_t slot = (uint32_t)__umul64hi(x, (uint64_t)n_atoms);
    uint32_t acc = always;
#pragma unroll
    for (int k = 0; k < KMC_NCLASS; ++k) acc |= (x < thr[k] ? 1u : 0u) << k;
    return (list_base + 2u * (n - 1u - slot)) | ((uint32_t)(x >> 62) << 17) |
           ((acc & ((1u << KMC_NCLASS) - 1u)) << 19) | (x * n_atoms < n_atoms ? 1u << 31 : 0u);
  };
  auto put = [&](int slot, int k, uint64_t raw_word, int = 0) {
    const uint32_t r = record(mt_temper(raw_word));
    L.rec[slot * MT_N + k] = r;
    if (slot == 0) L.rec[REC_RING + k] = r;
  };
  // coordinates (8 i and j) of the site at byte address 8 l: exact while
  // 8 l * 8 rows < 2^32
  const uint32_t col8 = 8u * rows;  // a step in j
  const uint32_t magic = (uint32_t)(((1ull << 32) + col8 - 1u) / col8);
  auto split = [&](uint32_t a, uint32_t &i8, uint32_t &j) __attribute__((always_inline)) {
    j = __umulhi(a, magic);
    i8 = a - j * col8;
  };

  for (uint32_t i = threadIdx.x; i < MT_N; i += KMC_WALK_THREADS) {
    L.raw[0][i] = St->mt[i];
    put(0, (int)i, St->mt[i]);
  }
  for (uint32_t i = threadIdx.x; i < n; i += KMC_WALK_THREADS) {
    const uint32_t l = (uint32_t)g_list[i];
    list[i] = (uint16_t)(8u * l);
    site[2 * l] = (i << KMC_POS) | (i >= n - n_atoms ? 1u << KMC_OCC : 0u);
    site[2 * l + 1] = KMC_NO_MARK;
  }
  if (threadIdx.x < 4) {
    const bool along_i = threadIdx.x < 2, plus = !(threadIdx.x & 1);
    const uint32_t s = along_i ? 8u : col8, w = along_i ? col8 - 8u : 8u * n - col8;
    const uint32_t top = along_i ? col8 - 8u : cols - 1u, unit = along_i ? 8u : 1u;
    KmcDir &D = L.dir[threadIdx.x];
    D.step = plus ? s : 0u - s;
    D.wrap = plus ? 0u - w : w;
    D.edge = plus ? top : 0u;
    D.next = plus ? top - unit : unit;
    D.far = plus ? 0u : top;
    D.up = along_i ? col8 : 8u;
    D.up_wrap = along_i ? col8 - 8u * n : 8u - col8;
    D.up_edge = along_i ? cols - 1u : col8 - 8u;
  }
  if (threadIdx.x == 0) {
    *done = 0;
    *pub = 0;
    L.cum[KMC_FIFO - 1] = 0;
  }
  __syncthreads();
  for (uint32_t a = threadIdx.x; a < n_atoms; a += KMC_WALK_THREADS) {
    const uint32_t l = (uint32_t)g_atoms[4 * a];
    ax[a] = g_atoms[4 * a + 1];
    ay[a] = g_atoms[4 * a + 2];
    ajump[a] = g_atoms[4 * a + 3];
    uint32_t i8, j;
    split(8u * l, i8, j);
    lds_add(KMC_WALK_FIXED_LDS + 8u * l, a);
    for (int d = 0; d < 4; ++d)
      lds_add(KMC_WALK_FIXED_LDS + 8u * l +
                  ((d < 2 ? i8 : j) == L.dir[d].edge ? L.dir[d].wrap : L.dir[d].step),
              1u << KMC_CNT);
  }
  __syncthreads();
  if (wave >= 2) {
    walk_producer(L.raw, done, wave - 2, lane, put);
    return;
  }
  if (wave == 1) {
    kmc_account(P, St, g_atoms, series + (int64_t)c * series_cap, series_cap, sample_period, L, ax,
                ay, ajump, pub, done, lane);
    return;
  }

  const int64_t pos0 = St->pos;
  WalkRing ring{(int)pos0};
  uint32_t pushed = 0;
  // attempts of this launch, and at its last event, modulo 2^32
  uint32_t cum = 0, cum_ev = 0u - (uint32_t)(St->kmc_k < (1ll << 31) ? St->kmc_k : 1ll << 31);
  bool any_event = false;
  const uint32_t spin_limit = (uint32_t)P->spin_limit;
  int64_t remaining = n_passes * (int64_t)n + n_steps, step = St->step;
  int seg = 0, left = 0;  // events up to the end of the pass or launch, and those to go
  bool frozen = false;
  const uint32_t pba_adr = list_base + 2u * (n - n_atoms);  // the atom list's last entry
  const uint32_t pba_f = (n - n_atoms) << KMC_POS;
  uint32_t back0 = (uint32_t)rfl32((int32_t)list[n - n_atoms]);
  uint32_t my_mark = KMC_FIRST_EPOCH * 64u + (uint32_t)lane;
  auto ensure = [&](int upto) { ring.ensure(upto, pushed, pub, lane); };
  auto push = [&](uint32_t rank, uint32_t k, uint32_t what) __attribute__((always_inline)) {
    const uint32_t at = 4u * ((pushed + rank) & (KMC_FIFO - 1));
    *lds_at(offsetof(KmcWalkLds, cum) + at) = k;
    *lds_at(offsetof(KmcWalkLds, what) + at) = what;
  };
  auto segment_end = [&]() -> bool {
    step += seg;
    remaining -= seg;
    any_event = any_event || seg > 0;
    if (step == (int64_t)n) {
      step = 0;
      if (lane == 0) push(0, cum, KMC_PASS_END);
      ++pushed;
    }
    seg = left = (int)(remaining < (int64_t)n - step ? remaining : (int64_t)n - step);
    // a block takes an epoch only if it has an event
    if ((my_mark >> 6) <= (uint32_t)left) {
      for (uint32_t i = lane; i < n; i += 64) site[2 * i + 1] = KMC_NO_MARK;
      my_mark = KMC_FIRST_EPOCH * 64u + (uint32_t)lane;
    }
    return remaining > 0;
  };
  // an attempt's sites (byte addresses): origin and target, their other neighbours.
  // Its class a - b + 3 from the words' upper bits, for an occupied origin and a free
  // target: (8 + a) - (b + 1) - 4, edges being at least 3 sites.  With an occupied
  // target that is -7 to -1: as a shift's amount 25 to 31, where no mask has a bit
  struct Hop {
    uint32_t a, to, behind, beyond, f0, f1, t0, t1;
  };
  auto direction = [&](uint32_t d) __attribute__((always_inline)) { return L.dir[d]; };
  auto target = [&](const KmcDir &D, bool along_i, Hop &h, uint32_t &u, uint32_t &v)
      __attribute__((always_inline)) {
    uint32_t i8, j;
    split(h.a, i8, j);
    u = along_i ? i8 : j;
    v = along_i ? j : i8;
    h.to = h.a + (u == D.edge ? D.wrap : D.step);
  };
  auto others = [&](const KmcDir &D, Hop &h, uint32_t u, uint32_t v)
      __attribute__((always_inline)) {
    h.behind = h.a - (u == D.far ? D.wrap : D.step);
    h.beyond = h.to + (u == D.next ? D.wrap : D.step);
    const uint32_t up = v == D.up_edge ? D.up_wrap : D.up;
    const uint32_t down = v == 0u ? D.up_wrap : D.up;
    h.f0 = h.a + up;
    h.f1 = h.a - down;
    h.t0 = h.to + up;
    h.t1 = h.to - down;
  };
  constexpr uint32_t CNT1 = 1u << KMC_CNT, OCC1 = 1u << KMC_OCC;
  auto put_list = [&](uint32_t at, uint32_t a) __attribute__((always_inline)) {
    *(volatile __attribute__((address_space(3))) uint16_t *)(uintptr_t)at = (uint16_t)a;
  };
  // a hop by the calling lane: list entry pa (its address; as a field of a word) and
  // the two words, all but what depends on the atom list's last site ...
  auto apply = [&](const Hop &h, uint32_t pa_f, uint32_t wf, uint32_t wt)
      __attribute__((always_inline)) {
    const uint32_t pt_f = wt & (0x1FFFu << KMC_POS), atom = wf & 0x1FFFu;
    lds_add(KMC_WALK_FIXED_LDS + h.behind, 0u - CNT1);
    lds_add(KMC_WALK_FIXED_LDS + h.f0, 0u - CNT1);
    lds_add(KMC_WALK_FIXED_LDS + h.f1, 0u - CNT1);
    lds_add(KMC_WALK_FIXED_LDS + h.beyond, CNT1);
    lds_add(KMC_WALK_FIXED_LDS + h.t0, CNT1);
    lds_add(KMC_WALK_FIXED_LDS + h.t1, CNT1);
    lds_add(KMC_WALK_FIXED_LDS + h.a, pt_f - pa_f - atom - OCC1 + CNT1);
    lds_add(KMC_WALK_FIXED_LDS + h.to, pba_f - pt_f + atom + OCC1 - CNT1);
    put_list(list_base + (pt_f >> (KMC_POS - 1)), h.a);
  };
  // ... and that
  auto apply_back = [&](uint32_t pa, uint32_t pa_f, uint32_t back)
      __attribute__((always_inline)) {
    put_list(pa, back);
    lds_add(KMC_WALK_FIXED_LDS + back, pa_f - pba_f);
  };
  auto pos_field = [&](uint32_t pa) __attribute__((always_inline)) {
    return (pa - list_base) << (KMC_POS - 1);
  };
  auto word_at = [&](uint32_t a) __attribute__((always_inline)) {
    return *lds_at(KMC_WALK_FIXED_LDS + a);
  };
  // one attempt with the full Lemire rejection loop, every lane alike
  auto special_attempt = [&]() {
    auto next_word = [&]() -> uint64_t {
      ensure(1);
      const uint64_t x = ring.word(L.raw);
      ++ring.rp;
      return x;
    };
    const uint64_t m = n_atoms, th = (0ULL - m) % m;
    uint64_t x = next_word();
    while (x * m < th) x = next_word();
    const uint32_t pa = list_base + 2u * (n - 1u - (uint32_t)__umul64hi(x, m));
    const uint32_t dir = (uint32_t)(next_word() >> 62);
    const KmcDir D = direction(dir);
    Hop h;
    uint32_t u, v;
    h.a = list[(pa - list_base) >> 1];
    target(D, dir < 2u, h, u, v);
    others(D, h, u, v);
    const uint32_t wf = word_at(h.a), wt = word_at(h.to);
    const int k = rfl32((int)(wf >> KMC_CNT) - (int)(wt >> KMC_CNT) - 4);
    bool ok = k >= 0;
    if (ok && ((draw_mask >> k) & 1u))
      ok = next_word() < P->thr[k] || ((P->full_mask >> k) & 1u);
    ok = rfl32(ok) != 0;
    asm volatile("" ::: "memory");
    ++cum;
    if (ok) {
      if (lane == 0) {
        apply(h, pos_field(pa), wf, wt);
        apply_back(pa, pos_field(pa), back0);
        put_list(pba_adr, h.to);
        push(0, cum, (wf & 0x1FFFu) | (dir << KMC_POS) | ((uint32_t)k << 15));
      }
      ++pushed;
      --left;
      back0 = (uint32_t)rfl32((int32_t)h.to);
      cum_ev = cum;
    }
    asm volatile("" ::: "memory");
  };
  auto bits_below = [&](uint64_t m, uint32_t plus) __attribute__((always_inline)) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, plus));
  };

  WindowStarts<2> starts;
  uint32_t r0 = 0, r1 = 0, r2 = 0;
  auto fetch = [&]() __attribute__((always_inline)) {
    r0 = L.rec[ring.rp + lane];
    r1 = L.rec[ring.rp + lane + 1];
    r2 = L.rec[ring.rp + lane + 2];
  };
  while (!frozen && (left > 0 || segment_end())) {
    ensure(66);
    fetch();
    for (;;) {
      const uint32_t pa = r0 & 0x1FFFFu, dir = (r1 >> 17) & 3u, acc = r2 >> 19;
      Hop h;
      h.a = *(const __attribute__((address_space(3))) uint16_t *)(uintptr_t)pa;
      const KmcDir D = direction(dir);
      const uint64_t SP = __ballot((int32_t)r0 < 0);
      uint32_t u, v;
      target(D, dir < 2u, h, u, v);
      const uint32_t wf = word_at(h.a), wt = word_at(h.to);
      __builtin_amdgcn_sched_barrier(0);
      others(D, h, u, v);
      asm volatile(""
                   : "+v"(h.behind), "+v"(h.beyond), "+v"(h.f0), "+v"(h.f1), "+v"(h.t0), "+v"(h.t1));
      const uint32_t k = (wf >> KMC_CNT) - (wt >> KMC_CNT) - 4u;
      const uint32_t kbit = 1u << (k & 31u);
      const uint64_t AC = __ballot((acc & kbit) != 0u);
      uint64_t ND = __ballot((draw_mask & kbit) != 0u);
      uint64_t exec = starts(__builtin_amdgcn_inverse_ballot_w64(ND));
      if (__builtin_expect(SP != 0, 0)) {  // attempt starts up to the first special one
        exec &= SP & exec ? ((SP & exec) & (0ull - (SP & exec))) - 1ull : ~0ull;
        if (!exec) {
          special_attempt();
          frozen = cum - cum_ev > spin_limit;
          break;
        }
      }
      uint64_t EV = exec & AC;
      if (EV) {
        if (__builtin_amdgcn_inverse_ballot_w64(EV)) {
          constexpr uint32_t MARK = KMC_WALK_FIXED_LDS + 4u;
          lds_min(MARK + h.a, my_mark);
          lds_min(MARK + h.to, my_mark);
          lds_min(MARK + h.behind, my_mark);
          lds_min(MARK + h.beyond, my_mark);
          lds_min(MARK + h.f0, my_mark);
          lds_min(MARK + h.f1, my_mark);
          lds_min(MARK + h.t0, my_mark);
          lds_min(MARK + h.t1, my_mark);
          // for the attempts of the list's last entry (an address that the compiler
          // does not know to be one: it would reduce the values first)
          uint32_t b0 = back0;
          asm("" : "+v"(b0));
          lds_min(MARK + b0, my_mark);
        }
        asm volatile("" ::: "memory");
        const uint32_t m0 = word_at(h.a + 4u), m1 = word_at(h.to + 4u);
        asm volatile("" ::: "memory");
        const uint64_t HIT = exec & __ballot((m0 < m1 ? m0 : m1) < my_mark);
        if (HIT) {
          exec &= (HIT & (0ull - HIT)) - 1ull;
          EV &= exec;
        }
        my_mark -= 64u;
      }
      int n_ev = __popcll(EV);
      if (__builtin_expect(n_ev >= left, 0)) {  // up to the segment's last event
        uint64_t rest = EV;
        for (int r = 1; r < left; ++r) rest &= rest - 1;
        const uint64_t upto = ((rest & (0ull - rest)) << 1) - 1ull;
        exec &= upto;
        EV &= upto;
        n_ev = left;
      }
      const int last = 63 - __builtin_clzll(exec);
      ring.rp += last + 2 + (int)((ND >> last) & 1ull);
      left -= n_ev;
      const bool more = ((ring.end - 66 - ring.rp) | (left - 1)) >= 0;
      if (more) fetch();
      asm volatile("" ::: "memory");
      const uint32_t cum0 = cum;
      cum += (uint32_t)__popcll(exec);
      if (EV) {
        const int lev = 63 - __builtin_clzll(EV);
        if (__builtin_amdgcn_inverse_ballot_w64(EV)) {
          const uint32_t rank = bits_below(EV, 0u);
          constexpr uint32_t TOS = offsetof(KmcWalkLds, tos);
          *(volatile lds_u32 *)lds_at(TOS + 4u * rank) = h.to;
          uint32_t back = *(volatile lds_u32 *)lds_at(TOS + 4u * (rank ? rank - 1u : 0u));
          push(rank, bits_below(exec, cum0 + 1u),
               (wf & 0x1FFFu) | (dir << KMC_POS) | (k << 15));
          const uint32_t pa_f = pos_field(pa);
          apply(h, pa_f, wf, wt);
          back = rank ? back : back0;
          apply_back(pa, pa_f, back);
          if (lane == lev) put_list(pba_adr, h.to);
        }
        back0 = (uint32_t)__builtin_amdgcn_readlane((int)h.to, lev);
        pushed += (uint32_t)n_ev;
        cum_ev = cum - (uint32_t)__popcll((exec >> lev) >> 1);
      } else if (__builtin_expect(cum - cum_ev > spin_limit, 0)) {
        frozen = true;
        break;
      }
      asm volatile("" ::: "memory");
      if (!more) break;
    }
  }
  if (frozen) {  // the events made so far
    step += seg - left;
    any_event = any_event || seg > left;
    if (step == (int64_t)n) {
      step = 0;
      if (lane == 0) push(0, cum, KMC_PASS_END);
      ++pushed;
    }
  }

  // release the other waves
  const int64_t k_run = any_event ? (int64_t)(cum - cum_ev) : St->kmc_k + cum;
  if (lane == 0) {
    L.tail = any_event ? cum - cum_ev : cum;
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
    const uint32_t w = site[2 * i];
    g_list[i] = (int32_t)(list[i] >> 3);
    g_lat[i] = (int8_t)(w >> KMC_OCC);
    if (w >> KMC_OCC) g_atoms[4 * (w & 0x1FFFu)] = (int32_t)i;
  }
  if (lane == 0) {
    St->pos = p_fin;
    St->step = step;
    St->kmc_k = k_run;
    St->frozen = frozen;
  }
}

void launch_kmc(const KmcParams *P, ExactState *S, int8_t *lat_pool, int32_t *list_pool,
                int32_t *atom_pool, KmcHop *hop_pool, int32_t *hop_count_pool,
                mcg_sample *series, int64_t series_cap, const uint8_t *active, int n_chains,
                int64_t n_passes, int64_t n_steps, int64_t sample_period, double stop_time,
                int select_at_end, bool walk, int lds_bytes, hipStream_t stream) {
  if (walk)
    hipLaunchKernelGGL(kmc_walk_kernel, dim3(n_chains), dim3(KMC_WALK_THREADS), lds_bytes, stream,
                       P, S, lat_pool, list_pool, atom_pool, series, series_cap, active, n_passes,
                       n_steps, sample_period);
  else
    hipLaunchKernelGGL(kmc_kernel, dim3(n_chains), dim3(128), lds_bytes, stream, P, S, lat_pool,
                       list_pool, atom_pool, hop_pool, hop_count_pool, series, series_cap, active,
                       n_passes, n_steps, sample_period, stop_time, select_at_end);
}

hipError_t kmc_set_max_lds(int general_bytes, int walk_bytes) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kmc_kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           general_bytes);
  return e != hipSuccess ? e
                         : set_dynamic_lds(reinterpret_cast<const void *>(kmc_walk_kernel),
                                           walk_bytes, true);
}

}  // namespace mcg
