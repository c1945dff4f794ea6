// checker_bits.hip -- CHECKERBOARD HBM path of large even lattices on bit-packed
// copies: 2D in bands of lines streamed through registers, 3D J1+J2 a plane at a
// time in LDS, 3D J1 a word a thread.  Trajectories are those of the colour-by-colour sweep (checker.hip):
// same colours in the same order on the same neighbour values with the same random
// words.
//
// A run packs the lattices it updates (one byte a site in HBM) into words of 32
// sites, makes its passes on those -- 1/8 of the bytes, so two 4096x4096 lattices
// live in the caches -- and unpacks them at its end.
#include "checker_bits.hh"

#include <algorithm>

namespace mcg {

namespace {

// words of a half line
__host__ __device__ inline int bit_hw(int L0) { return (L0 / 2 + 31) / 32; }

// parts of 8 oct sites of a half line
__host__ __device__ inline int bit_parts(int L0, int oct) {
  return (L0 / 2 + 8 * oct - 1) / (8 * oct);
}

struct BitLattice {
  int L0, L1, half, hw, lw;  // lw: words per line
};

__device__ __forceinline__ BitLattice bit_lattice(const CheckerParams &P) {
  BitLattice G;
  G.L0 = P.L0;
  G.L1 = P.L1;
  G.half = P.L0 >> 1;
  G.hw = bit_hw(P.L0);
  G.lw = 2 * G.hw;
  return G;
}

// Word wi of chain P's lattice (line-major: line, half, word): its first site's
// byte, and whether it has 32 sites or 16.
__device__ __forceinline__ int64_t word_byte(const BitLattice &G, int64_t wi, bool &full) {
  const int64_t line = wi / G.lw;
  const int r = (int)(wi - line * G.lw), a = r >= G.hw ? 1 : 0, w = r - a * G.hw;
  full = 32 * w + 32 <= G.half;
  return line * G.L0 + a * G.half + 32 * w;
}

}  // namespace

// items: (chain, offset) of every chain; a 2D chain's words go to the buffer of its
// pass's parity, a 3D one's to its only buffer.
__global__ __launch_bounds__(256) void bit_pack_kernel(const CheckerParams *__restrict__ Pp,
                                                      const CheckerState *__restrict__ Sp,
                                                      const int8_t *__restrict__ lat_pool,
                                                      uint32_t *__restrict__ bits,
                                                      const BitItem *__restrict__ items) {
  const BitItem it = items[blockIdx.y];
  const CheckerParams P = Pp[it.chain];
  const BitLattice G = bit_lattice(P);
  const int64_t words = (int64_t)P.L1 * P.L2 * G.lw;
  const int64_t wi = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (wi >= words) return;
  uint32_t *to = bits + it.off + (P.ndim == 2 ? (Sp[it.chain].n_pass & 1) * words : 0);
  bool full;
  const uint4 *src =
      reinterpret_cast<const uint4 *>(lat_pool + P.lat_off + word_byte(G, wi, full));
  uint32_t x = pack16(src[0]);
  if (full) x |= pack16(src[1]) << 16;
  to[wi] = x;
}

__global__ __launch_bounds__(256) void bit_unpack_kernel(const CheckerParams *__restrict__ Pp,
                                                        const CheckerState *__restrict__ Sp,
                                                        int8_t *__restrict__ lat_pool,
                                                        const uint32_t *__restrict__ bits,
                                                        const BitItem *__restrict__ items) {
  const BitItem it = items[blockIdx.y];
  const CheckerParams P = Pp[it.chain];
  const BitLattice G = bit_lattice(P);
  const int64_t words = (int64_t)P.L1 * P.L2 * G.lw;
  const int64_t wi = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (wi >= words) return;
  const uint32_t x = bits[it.off + (P.ndim == 2 ? (Sp[it.chain].n_pass & 1) * words : 0) + wi];
  bool full;
  uint4 *dst = reinterpret_cast<uint4 *>(lat_pool + P.lat_off + word_byte(G, wi, full));
  dst[0] = unpack16(x);
  if (full) dst[1] = unpack16(x >> 16);
}

// ---------------------------------------------------------------------------
// 2D: a band of H lines [j0, j0 + H) by the hw lanes of a group, lane w holding word
// w (or part w of the words) of both halves of the lines it works on; a wavefront takes as many groups (bands)
// as fit its 64 lanes.  Lines stream through registers; the word's neighbours in the
// line come from the group's lanes by ds_bpermute, so nothing waits at a barrier.
//
// 4 colours (A: 0 then 1 on the even lines, B: 2 then 3 on the odd ones): A(j) reads
// the odd lines j-1, j+1 before the pass, B(j) the even lines j-1, j+1 after A.  With
// A(j) done B(j-1) follows.  The band's last odd line needs A on the next band's
// first line: it is made here too and not kept.  2 colours (A: colour 0 of every
// line, B: colour 1): the same with A on the lines before and behind the band.  A
// pass reads one buffer and writes the other, so bands do not wait for each other.
//
// A lane's words are whole ones, or halves or bytes of them where whole ones would leave
// SIMDs without a wave (word_cost, api.hip).
//
// Measured on MI355X, us a pass, against the two launches of checker_band_kernel and
// checker_seam_kernel: two lattices of 4096x4096 J1+J2 25 and 48, J1 24 and 44; 16 of
// them 120 and 241, J1 103; two of 1504x1000 9.8 and 28; one of 512x512 7.2 and 30.  Few waves
// (two a SIMD on two 4096x4096 lattices): latency and the launches bound those,
// instruction issue the 16.
// ---------------------------------------------------------------------------
namespace {

struct StreamLane {
  int left, right;      // lanes of the neighbouring words, times 4
  uint32_t top, ltop;   // place of the own word's last site, of the left word's
  uint32_t valid;       // the word's sites
  __device__ __forceinline__ uint32_t from(int lane4, uint32_t x) const {
    return (uint32_t)__builtin_amdgcn_ds_bpermute(lane4, (int)x);
  }
  // index h - 1 of the half (west of an even site), index h + 1 (east of an odd one)
  __device__ __forceinline__ uint32_t west(uint32_t x) const {
    return ((x << 1) & valid) | ((from(left, x) >> ltop) & 1u);
  }
  __device__ __forceinline__ uint32_t east(uint32_t x) const {
    return (x >> 1) | ((from(right, x) & 1u) << top);
  }
};

// sum of four bit vectors
__device__ __forceinline__ void sum4(uint32_t a, uint32_t b, uint32_t c, uint32_t d,
                                     uint32_t (&s)[3]) {
  uint32_t t, k;
  csa(a, b, c, t, k);
  s[0] = t ^ d;
  const uint32_t u = t & d;
  s[1] = k ^ u;
  s[2] = k & u;
}

}  // namespace

constexpr int STREAM_BLOCK = 256;

// a lane's part of a word
template <int OCT>
struct BitPart {
  using type = uint32_t;
};
template <>
struct BitPart<1> {
  using type = uint8_t;
};
template <>
struct BitPart<2> {
  using type = uint16_t;
};

// OCT: a lane holds 8 OCT sites of each half (w: that part of the line)
template <bool FOUR, int OCT>
__global__ __launch_bounds__(STREAM_BLOCK) void checker_stream_kernel(
    const CheckerParams *__restrict__ Pp, const CheckerState *__restrict__ Sp,
    uint32_t *__restrict__ bits, const uint32_t *__restrict__ tables,
    const BitItem *__restrict__ items, int, int ahead) {
  __shared__ uint32_t thi[FOUR ? 64 : 256];  // thresholds' high halves (two sites': pairs)
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = blockIdx.x * (STREAM_BLOCK / 64) + wave;
  const BitItem it = items[wi];  // (a workgroup's are one chain's; the last may be empty)
  const CheckerParams P = checker_ahead(Pp, it.chain, ahead);
  const int64_t pass = Sp[it.chain].n_pass + ahead;
  const uint32_t *tab = tables + P.tab_off;
  if (FOUR)
    bit_load_thresholds<false>(reinterpret_cast<uint16_t *>(thi), tab, threadIdx.x, STREAM_BLOCK);
  else
    pair_load_thresholds(thi, tab, threadIdx.x, STREAM_BLOCK);
  __syncthreads();
  if (it.n_groups == 0) return;
  const BitLattice G = bit_lattice(P);
  using Part = typename BitPart<OCT>::type;
  constexpr int PER = 4 / OCT;  // parts a word
  const int hw = bit_parts(G.L0, OCT), L1 = P.L1, H = it.H;
  int g = lane / hw;
  const int w = lane - g * hw;
  const bool live = g < it.n_groups;
  g = live ? g : 0;
  StreamLane S;
  S.left = 4 * (w == 0 ? lane + hw - 1 : lane - 1);
  S.right = 4 * (w == hw - 1 ? lane - w : lane + 1);
  const bool odd16 = OCT == 4 && (G.half & 31) != 0;
  S.top = odd16 && w == hw - 1 ? 15u : 8u * OCT - 1u;
  S.ltop = odd16 && (w == 0 || hw == 1) ? 15u : 8u * OCT - 1u;
  S.valid = odd16 && w == hw - 1 ? 0xFFFFu : 0xFFFFFFFFu >> (32 - 8 * OCT);
  const int64_t words = (int64_t)L1 * G.lw;
  const uint32_t *src = bits + it.off + (pass & 1) * words;
  uint32_t *dst = bits + it.off + (~pass & 1) * words;
  const int j0 = it.j0 + g * H;
  const int opl = (G.half + 7) >> 3;
  auto wrap = [&](int j) __attribute__((always_inline)) {
    return j < 0 ? j + L1 : (j >= L1 ? j - L1 : j);
  };
  auto load = [&](int j, uint32_t &h0, uint32_t &h1) __attribute__((always_inline)) {
    const Part *p = reinterpret_cast<const Part *>(src + (int64_t)wrap(j) * G.lw) + w;
    h0 = p[0];
    h1 = p[PER * G.hw];
  };
  auto store = [&](int j, uint32_t h0, uint32_t h1) __attribute__((always_inline)) {
    if (!live) return;
    Part *p = reinterpret_cast<Part *>(dst + (int64_t)j * G.lw) + w;
    p[0] = (Part)h0;
    p[PER * G.hw] = (Part)h1;
  };
  BitRng rng{(uint32_t)pass, (uint32_t)(pass >> 32), 0u, P.key0, P.key1};
  BitDelta d;
  // one colour of one line: class line ln, neighbours n (nearest) and m (next nearest)
  auto update = [&](uint32_t own, uint32_t color, int ln, uint32_t n1, uint32_t n2, uint32_t n3,
                    uint32_t n4, uint32_t m1, uint32_t m2, uint32_t m3, uint32_t m4,
                    bool count) __attribute__((always_inline)) {
    uint32_t c1[3], c2[3] = {0u, 0u, 0u};
    sum4(n1, n2, n3, n4, c1);
    if (FOUR) sum4(m1, m2, m3, m4, c2);
    uint32_t x[8] = {0u, c2[0], c2[1], c2[2], c1[0], c1[1], c1[2], own};
    rng.color = color;
    const uint32_t first = (uint32_t)(ln * opl + OCT * w);
    const uint32_t site0 = (uint32_t)(ln * G.half + 8 * OCT * w);
    const uint32_t flip =
        S.valid & (FOUR ? bit_flips<false, OCT>(x, rng, first, site0,
                                                reinterpret_cast<const uint16_t *>(thi), tab)
                        : pair_flips<OCT>(c1, own, rng, first, site0, thi, tab));
    if (count) d.add(own, flip, c1, c2);
    return own ^ flip;
  };

  if (FOUR) {
    uint32_t o0, o1, e0, e1, n0, n1;  // lines j-1 (old), j, j+1
    load(j0 - 1, o0, o1);
    load(j0, e0, e1);
    load(j0 + 1, n0, n1);
    uint32_t ow = S.west(o1), oe = S.east(o0);
    uint32_t p0 = 0, p1 = 0, pw = 0, pe = 0;  // line j-2 after A
    for (int i = 0; i <= H / 2; ++i) {
      const int j = j0 + 2 * i;
      uint32_t a0 = 0, a1 = 0, b0 = 0, b1 = 0;
      if (i < H / 2) {
        load(j + 2, a0, a1);
        load(j + 3, b0, b1);
      }
      const uint32_t nw = S.west(n1), ne = S.east(n0);
      const int ln = wrap(j) >> 1;
      e0 = update(e0, 0, ln, e1, S.west(e1), o0, n0, o1, ow, n1, nw, i < H / 2);
      const uint32_t ee = S.east(e0);
      e1 = update(e1, 1, ln, e0, ee, o1, n1, o0, oe, n0, ne, i < H / 2);
      const uint32_t ew = S.west(e1);
      if (i < H / 2) store(j, e0, e1);
      if (i > 0) {
        const int lo = (j - 1) >> 1;
        o0 = update(o0, 2, lo, o1, ow, p0, e0, p1, pw, e1, ew, true);
        o1 = update(o1, 3, lo, o0, S.east(o0), p1, e1, p0, pe, e0, ee, true);
        store(j - 1, o0, o1);
      }
      p0 = e0;
      p1 = e1;
      pw = ew;
      pe = ee;
      o0 = n0;
      o1 = n1;
      ow = nw;
      oe = ne;
      e0 = a0;
      e1 = a1;
      n0 = b0;
      n1 = b1;
    }
  } else {
    // lines j-2 (after A), j-1 (after A), j, j+1; the band from j = j0 - 1 (odd)
    uint32_t q0 = 0, q1 = 0, p0, p1, c0, c1, n0, n1;
    load(j0 - 2, p0, p1);
    load(j0 - 1, c0, c1);
    load(j0, n0, n1);
    auto shift = [&](int a, uint32_t x) __attribute__((always_inline)) {
      return a ? S.east(x) : S.west(x);
    };
    // A on line j, whose own half is a (the parity of j), then B on line j-1
    auto step = [&](int j, int a) __attribute__((always_inline)) {
      uint32_t f0 = 0, f1 = 0;
      if (j < j0 + H) load(j + 2, f0, f1);
      uint32_t &own = a ? c1 : c0;
      const uint32_t oth = a ? c0 : c1;
      own = update(own, 0, wrap(j), oth, shift(a, oth), a ? p1 : p0, a ? n1 : n0, 0, 0, 0, 0,
                   j >= j0 && j < j0 + H);
      if (j > j0) {
        uint32_t &bown = a ? p1 : p0;
        const uint32_t both = a ? p0 : p1;
        bown = update(bown, 1, j - 1, both, shift(a, both), a ? q1 : q0, own, 0, 0, 0, 0, true);
        store(j - 1, p0, p1);
      }
      q0 = p0;
      q1 = p1;
      p0 = c0;
      p1 = c1;
      c0 = n0;
      c1 = n1;
      n0 = f0;
      n1 = f1;
    };
    for (int j = j0 - 1; j <= j0 + H; j += 2) {
      step(j, 1);
      step(j + 1, 0);
    }
  }
  int s[4] = {0, 0, 0, 0};
  if (live) d.sums(P.z1, P.z2, s);
  bit_add_deltas(P, wi, s, lane);
}

// ---------------------------------------------------------------------------
// 3D J1+J2 (8 colours (i&1) + 2(j&1) + 4(k&1)).  A plane holds one k parity, so the
// even planes carry colours 0-3 and the odd ones 4-7, and a site's neighbours lie in
// its own plane and the planes k+-1: one launch updates the even planes, the next the
// odd ones, in place, a plane per workgroup.  The three planes are read into LDS once
// (rows padded to an odd word count); between the four colours is a barrier.  A
// thread updates 8 OCT sites of one colour in a word, their 6 and 12 neighbour bits from
// 18 words.
//
// Measured on MI355X, us a pass, against slabs streamed through an LDS ring from bytes
// with their edge planes in a second launch: two lattices of 256^3 34.9 and 63.7, 16
// of them 162 and 297, one of 192^3 28.8 and 52, one of 64x100x80 16.2 and 33.6.
// ---------------------------------------------------------------------------
namespace {

struct PlaneGeom {
  int hw, rs, L1;  // words per half row, per padded row; rows
};

// 8 OCT sites (part `part` of word w) of a colour (half a of row j) of the plane in
// `own`, planes k-1 and k+1 in km and kp.
template <int OCT>
__device__ __forceinline__ void plane_word(const PlaneGeom &G, uint32_t *own, const uint32_t *km,
                                           const uint32_t *kp, int j, int a, int w, int part,
                                           const BitRng &rng, uint32_t first, uint32_t site0,
                                           const uint16_t *thi, const uint32_t *tab,
                                           BitDelta &d) {
  const int o = a ^ 1;
  const int jp = j + 1 == G.L1 ? 0 : j + 1, jm = j == 0 ? G.L1 - 1 : j - 1;
  // the word that supplies the bit shifted in: a = 0 takes index h-1 (word
  // w-1, its top bit), a = 1 index h+1 (word w+1, its bottom bit)
  const int wn = a ? (w + 1 == G.hw ? 0 : w + 1) : (w == 0 ? G.hw - 1 : w - 1);
  const int rj = j * G.rs, rjp = jp * G.rs, rjm = jm * G.rs;
  const int sa = a * G.hw + w, so = o * G.hw + w, sn = o * G.hw + wn;
  auto sh = [&](uint32_t x, uint32_t xn) -> uint32_t {
    return a ? ((x >> 1) | (xn << 31)) : ((x << 1) | (xn >> 31));
  };
  uint32_t b = own[rj + sa];
  // nearest neighbours: in-line (other half, indices h and h-1+2a), rows j+-1,
  // planes k+-1
  const uint32_t oo = own[rj + so], oon = own[rj + sn];
  const uint32_t n1 = oo, n2 = sh(oo, oon);
  const uint32_t n3 = own[rjp + sa], n4 = own[rjm + sa];
  const uint32_t n5 = kp[rj + sa], n6 = km[rj + sa];
  // next-nearest: in-plane diagonals (rows j+-1, other half), (i+-1, k+-1)
  // (planes k+-1, row j, other half), (j+-1, k+-1) (planes k+-1, rows j+-1)
  const uint32_t pj = own[rjp + so], pjn = own[rjp + sn];
  const uint32_t mj = own[rjm + so], mjn = own[rjm + sn];
  const uint32_t pk = kp[rj + so], pkn = kp[rj + sn];
  const uint32_t mk = km[rj + so], mkn = km[rj + sn];
  const uint32_t m1 = pj, m2 = sh(pj, pjn), m3 = mj, m4 = sh(mj, mjn);
  const uint32_t m5 = pk, m6 = sh(pk, pkn), m7 = mk, m8 = sh(mk, mkn);
  const uint32_t m9 = kp[rjp + sa], m10 = kp[rjm + sa], m11 = km[rjp + sa], m12 = km[rjm + sa];
  // c1 = n1 + ... + n6
  uint32_t sa1, ca1, sb1, cb1, c1[3];
  csa(n1, n2, n3, sa1, ca1);
  csa(n4, n5, n6, sb1, cb1);
  c1[0] = sa1 ^ sb1;
  csa(ca1, cb1, sa1 & sb1, c1[1], c1[2]);
  // c2 = m1 + ... + m12
  uint32_t s1, k1, s2, k2, s3, k3, s4, k4, u1, v1, c2[4];
  csa(m1, m2, m3, s1, k1);
  csa(m4, m5, m6, s2, k2);
  csa(m7, m8, m9, s3, k3);
  csa(m10, m11, m12, s4, k4);
  csa(s1, s2, s3, u1, v1);
  c2[0] = u1 ^ s4;
  const uint32_t w1 = u1 & s4;
  uint32_t x1, y1, x2, y2;
  csa(k1, k2, k3, x1, y1);
  csa(k4, v1, w1, x2, y2);
  c2[1] = x1 ^ x2;
  csa(y1, y2, x1 & x2, c2[2], c2[3]);
  if (OCT < 4) {
    const int s = 8 * OCT * part;
    b >>= s;
#pragma unroll
    for (int p = 0; p < 3; ++p) c1[p] >>= s;
#pragma unroll
    for (int p = 0; p < 4; ++p) c2[p] >>= s;
  }
  uint32_t x[8] = {c2[0], c2[1], c2[2], c2[3], c1[0], c1[1], c1[2], b};
  const uint32_t flip = bit_flips<true, OCT>(x, rng, first + OCT * part, site0 + 8 * OCT * part,
                                             thi, tab);
  if (OCT == 4)
    own[rj + sa] = b ^ flip;
  else if (OCT == 2)
    reinterpret_cast<uint16_t *>(own + rj + sa)[part] = (uint16_t)(b ^ flip);
  else
    reinterpret_cast<uint8_t *>(own + rj + sa)[part] = (uint8_t)(b ^ flip);
  d.add(b, flip, c1, c2);
}

}  // namespace

// items: (chain, first of the plane pair, offset)
template <int OCT>
__global__ __launch_bounds__(512) void checker_plane_kernel(
    const CheckerParams *__restrict__ Pp, const CheckerState *__restrict__ Sp,
    uint32_t *__restrict__ bits, const uint32_t *__restrict__ tables,
    const BitItem *__restrict__ items, int parity, int ahead) {
  extern __shared__ __align__(16) uint32_t planes[];
  __shared__ uint16_t thi[CHECKER_NTAB];
  const BitItem it = items[blockIdx.x];
  const CheckerParams P = checker_ahead(Pp, it.chain, ahead);
  const int64_t pass = Sp[it.chain].n_pass + ahead;
  const uint32_t *tab = tables + P.tab_off;
  const int t = threadIdx.x, nt = blockDim.x;
  bit_load_thresholds<true>(thi, tab, t, nt);
  const BitLattice B = bit_lattice(P);
  const PlaneGeom G{B.hw, B.lw + 1, P.L1};
  const int k = it.j0 + parity, pw = P.L1 * B.lw, ps = P.L1 * G.rs;
  uint32_t *lat = bits + it.off;
  uint32_t *own = planes, *km = planes + ps, *kp = planes + 2 * ps;
  const int kd = k == 0 ? P.L2 - 1 : k - 1, ku = k + 1 == P.L2 ? 0 : k + 1;
  // floor(i / hw) for i hw < 2^32
  const uint32_t magic = 0xFFFFFFFFu / (uint32_t)B.hw + 1u;
  auto row_of = [&](int i) __attribute__((always_inline)) {
    return B.hw == 1 ? i : (int)__umulhi((uint32_t)i, magic);
  };
  // two words at a time, a thread's loads of the three planes before its LDS writes;
  // rows are one word longer in LDS
  uint2 *src = reinterpret_cast<uint2 *>(lat);
  const int ph = pw >> 1;
  for (int i0 = t; i0 < ph; i0 += 2 * nt) {
    uint2 v[2][3];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int i = min(i0 + e * nt, ph - 1);
      v[e][0] = src[(int64_t)k * ph + i];
      v[e][1] = src[(int64_t)kd * ph + i];
      v[e][2] = src[(int64_t)ku * ph + i];
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int i = min(i0 + e * nt, ph - 1), at = 2 * i + row_of(i);
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        planes[p * ps + at] = v[e][p].x;
        planes[p * ps + at + 1] = v[e][p].y;
      }
    }
  }
  __syncthreads();
  constexpr int PER = 4 / OCT;  // threads a word
  const int h1 = P.L1 >> 1, opl = B.half >> 3, words = h1 * B.hw;
  BitDelta d;
  BitRng rng{(uint32_t)pass, (uint32_t)(pass >> 32), 0u, P.key0, P.key1};
  for (int cc = 0; cc < 4; ++cc) {
    rng.color = (uint32_t)(4 * parity + cc);
    for (int u = t; u < PER * words; u += nt) {
      const int i = u / PER, r = row_of(i), w = i - r * B.hw, ln = r + h1 * (k >> 1);
      plane_word<OCT>(G, own, km, kp, (cc >> 1) + 2 * r, cc & 1, w, u % PER, rng,
                 (uint32_t)(ln * opl + 4 * w), (uint32_t)(ln * B.half + 32 * w), thi, tab, d);
    }
    __syncthreads();
  }
  for (int i = t; i < ph; i += nt) {
    const int at = 2 * i + row_of(i);
    src[(int64_t)k * ph + i] = make_uint2(own[at], own[at + 1]);
  }
  int s[4];
  d.sums(P.z1, P.z2, s);
  bit_add_deltas(P, (int)blockIdx.x + 32 * (t >> 6), s, t & 63);
}

// ---------------------------------------------------------------------------
// 3D J1 (2 colours (i + j + k) & 1).  A colour's sites have no neighbours of it, so a
// launch per colour updates it in place with no order among its words: a thread takes
// 8 OCT sites of one from the seven words around it, which come from the caches.
//
// Measured on MI355X, us a pass, against a launch per colour on bytes: one 64x100x80
// lattice 8.2 and 23.6, one of 192^3 12.9 and 46, two of 256^3 27 and 66.
// ---------------------------------------------------------------------------
// items: (chain, block of CUBE_BLOCK threads, offset)
constexpr int CUBE_BLOCK = 256;
template <int OCT>
__global__ __launch_bounds__(CUBE_BLOCK) void checker_cube_kernel(
    const CheckerParams *__restrict__ Pp, const CheckerState *__restrict__ Sp,
    uint32_t *__restrict__ bits, const uint32_t *__restrict__ tables,
    const BitItem *__restrict__ items, int color, int ahead) {
  // a workgroup of small parts makes few lookups: the smaller table (192^3, us a pass:
  // 12.9, 13.3 with pairs)
  constexpr bool PAIRS = OCT == 4;
  __shared__ uint32_t thi[PAIRS ? 256 : 64];
  const BitItem it = items[blockIdx.x];
  const CheckerParams P = checker_ahead(Pp, it.chain, ahead);
  const int64_t pass = Sp[it.chain].n_pass + ahead;
  const uint32_t *tab = tables + P.tab_off;
  const int t = threadIdx.x;
  if (PAIRS)
    pair_load_thresholds(thi, tab, t, CUBE_BLOCK);
  else
    bit_load_thresholds<false>(reinterpret_cast<uint16_t *>(thi), tab, t, CUBE_BLOCK);
  __syncthreads();
  const BitLattice G = bit_lattice(P);
  constexpr int PER = 4 / OCT;  // threads a word
  const uint32_t at = (uint32_t)it.j0 * CUBE_BLOCK + t;
  const uint32_t wd = at / PER, part = at % PER;
  const uint32_t ln = wd / (uint32_t)G.hw, w = wd - ln * (uint32_t)G.hw;
  int s[4] = {0, 0, 0, 0};
  if (ln < (uint32_t)(P.L1 * P.L2)) {
    const int k = (int)(ln / (uint32_t)P.L1), j = (int)ln - k * P.L1, a = (color + j + k) & 1;
    const uint32_t wn = a ? (w + 1 == (uint32_t)G.hw ? 0u : w + 1) : (w == 0 ? G.hw - 1u : w - 1);
    uint32_t *lat = bits + it.off;
    uint32_t *own = lat + (int64_t)ln * G.lw;
    const int64_t row = G.lw, plane = (int64_t)P.L1 * G.lw;
    const uint32_t *jp = own + (j + 1 == P.L1 ? row - plane : row);
    const uint32_t *jm = own - (j == 0 ? row - plane : row);
    const int64_t all = P.L2 * plane;
    const uint32_t *kp = own + (k + 1 == P.L2 ? plane - all : plane);
    const uint32_t *km = own - (k == 0 ? plane - all : plane);
    const uint32_t sa = a * G.hw + w, so = (a ^ 1) * G.hw + w, sn = (a ^ 1) * G.hw + wn;
    uint32_t b = own[sa];
    const uint32_t n1 = own[so], nn = own[sn];
    const uint32_t n3 = jp[sa], n4 = jm[sa], n5 = kp[sa], n6 = km[sa];
    const uint32_t n2 = a ? ((n1 >> 1) | (nn << 31)) : ((n1 << 1) | (nn >> 31));
    uint32_t s1, k1, s2, k2, c1[3];
    csa(n1, n2, n3, s1, k1);
    csa(n4, n5, n6, s2, k2);
    c1[0] = s1 ^ s2;
    csa(k1, k2, s1 & s2, c1[1], c1[2]);
    const uint32_t sh = 8 * OCT * part;
    b >>= sh;
#pragma unroll
    for (int p = 0; p < 3; ++p) c1[p] >>= sh;
    const BitRng rng{(uint32_t)pass, (uint32_t)(pass >> 32), (uint32_t)color, P.key0, P.key1};
    const uint32_t first = ln * (uint32_t)(G.half >> 3) + 4 * w + OCT * part;
    const uint32_t site0 = ln * (uint32_t)G.half + 32 * w + 8 * OCT * part;
    uint32_t x[8] = {0u, 0u, 0u, 0u, c1[0], c1[1], c1[2], b};
    const uint32_t flip = PAIRS ? pair_flips<OCT>(c1, b, rng, first, site0, thi, tab)
                                : bit_flips<false, OCT>(x, rng, first, site0,
                                                        reinterpret_cast<const uint16_t *>(thi), tab);
    if (OCT == 4)
      own[sa] = b ^ flip;
    else if (OCT == 2)
      reinterpret_cast<uint16_t *>(own + sa)[part] = (uint16_t)(b ^ flip);
    else
      reinterpret_cast<uint8_t *>(own + sa)[part] = (uint8_t)(b ^ flip);
    BitDelta d;
    const uint32_t none[1] = {0u};
    d.add(b, flip, c1, none);
    d.sums(P.z1, P.z2, s);
  }
  bit_add_deltas(P, (int)(blockIdx.x * (CUBE_BLOCK / 64)) + (t >> 6), s, t & 63);
}

// ---------------------------------------------------------------------------
// 2D lattices that fit a workgroup: all passes of a run by one workgroup a chain, the
// lattice as bits in LDS, a word of 8 OCT sites of one class a thread.  Even edges:
// parity colourings; an odd edge (RING): the nine ring classes of checker_ring.hip,
// whose seam sites -- the last of an odd line -- are a class of their own, a site a
// thread.
//
// A line has its even-i sites, then its odd-i ones, hw words each, lines padded to an
// odd word count.  Between classes is one barrier and no other: each wave leaves its
// sums of a pass in LDS, double-buffered by pass, and thread 0 adds them up and writes
// the record while the others go on.
//
// Measured on MI355X, us a pass, against the workgroups on bytes (checker_lds_kernel,
// checker_ring_lds_kernel): 64 chains of 128x128 2.6 and 6.6, one of 32x32 1.5 and 3.8,
// 64 of 250x250 6.4 and 101 (lines that are no multiple of 32 took 4 sites a thread
// and byte loads), 64 of 181x253 12 and 64, 64 of 31x45 6 and 12.  A step of the
// smallest is the latency of one word's chain and a barrier, ~1 us.
// ---------------------------------------------------------------------------
template <bool RING, bool NNN, int OCT>
__global__ __launch_bounds__(1024) void checker_words_kernel(
    const CheckerParams *__restrict__ Pp, CheckerState *__restrict__ Sp,
    int8_t *__restrict__ lat_pool, const uint32_t *__restrict__ tables,
    mcg_sample *__restrict__ series, int64_t series_cap, const uint8_t *__restrict__ active,
    int64_t n_passes, int64_t sample_period) {
  constexpr int W = 8 * OCT;
  constexpr uint32_t FULL = OCT == 4 ? 0xFFFFFFFFu : (1u << (W & 31)) - 1u;
  const int c = blockIdx.x;
  if (!active[c]) return;
  extern __shared__ __align__(16) uint32_t words[];
  __shared__ uint32_t ltab[RING ? 128 : NNN ? 64 : 256];  // RING: thresholds; else high halves
  __shared__ int red[2][16][4];
  const CheckerParams P = Pp[c];
  CheckerState *St = Sp + c;
  int8_t *lat = lat_pool + P.lat_off;
  const uint32_t *tab = tables + P.tab_off;
  const int t = threadIdx.x, nt = blockDim.x, lane = t & 63, wid = t >> 6;
  const int L0 = P.L0, L1 = P.L1;
  const bool odd = RING && (L0 & 1);
  const int n_even = (L0 + 1) >> 1, n_odd = L0 >> 1;
  const int hw = (n_even + W - 1) / W, rs = 2 * hw + 1;
  // the place in its word of the site that a line's first has to its west (a choice between
  // variables inside the lambda below would put them and the sums into scratch memory: 1024
  // chains of 31x31, eight passes 156 us, so 105)
  const int wrap_place = (n_odd + (odd ? 1 : 0) - 1) % W;
  if (RING) {
    for (int i = t; i < 128; i += nt) ltab[i] = tab[((i & 0x78) << 1) | (i & 7)];
  } else if (NNN) {
    bit_load_thresholds<false>(reinterpret_cast<uint16_t *>(ltab), tab, t, nt);
  } else {
    pair_load_thresholds(ltab, tab, t, nt);
  }
  const uint16_t *thi = reinterpret_cast<const uint16_t *>(ltab);
  // site h of half a of line j, in the chain's layout
  auto byte_at = [&](int j, int a, int h) {
    return (int64_t)j * L0 + (RING ? 2 * h + a : a * n_odd + h);
  };
  // Parity chains: eight sites of a half line (a byte of a word) at a time, so that a wave's
  // accesses lie side by side.  With a word a thread a byte at a time, each access of a wave
  // touched 64 lines: 1024 chains of 128x128, one pass 94 us, so 39; one of 250x250 57 and 36.
  const int half8 = OCT * hw, line8 = 2 * half8, n8 = L1 * line8;
  const bool wide = (n_odd & 7) == 0;  // eight sites are eight aligned bytes
  const uint32_t inv = 0xFFFFFFFFu / (uint32_t)line8 + 1u;  // (i * line8 < 2^32)
  // the i-th of them: the first byte, the sites (at most 8 count); the place in LDS
  auto eight = [&](int i, int8_t *&p, int &m) __attribute__((always_inline)) {
    const int j = (int)__umulhi((uint32_t)i, inv), r = i - j * line8, a = r >= half8 ? 1 : 0;
    const int o = r - a * half8;
    p = lat + byte_at(j, a, 8 * o);
    m = n_odd - 8 * o;
    return reinterpret_cast<uint8_t *>(words + j * rs + a * hw + o / OCT) + o % OCT;
  };
  if (RING) {
    for (int i = t; i < L1 * 2 * hw; i += nt) {
      const int j = i / (2 * hw), r = i - j * 2 * hw, a = r >= hw ? 1 : 0, w = r - a * hw;
      const int m = (a ? n_odd : n_even) - W * w;
      uint32_t x = 0u;
  #pragma unroll
      for (int e = 0; e < W; ++e)
        if (e < m) x |= (lat[byte_at(j, a, W * w + e)] ? 1u : 0u) << e;
      words[j * rs + r] = x;
    }
  } else {
    if (OCT < 4) {  // the bits above a word's sites are zero
      for (int i = t; i < L1 * rs; i += nt) words[i] = 0u;
      __syncthreads();
    }
#pragma unroll 4
    for (int i = t; i < n8; i += nt) {
      int8_t *p;
      int m;
      uint8_t *to = eight(i, p, m);
      uint32_t x = 0u;
      if (wide) {
        if (m > 0) {
          const uint2 v = *reinterpret_cast<const uint2 *>(p);
          x = pack4(v.x) | (pack4(v.y) << 4);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (e < m) x |= (p[e] ? 1u : 0u) << e;
      }
      *to = (uint8_t)x;
    }
  }
  __syncthreads();

  int64_t pass = St->n_pass, n_samples = St->n_samples;
  int64_t S1 = St->S1, S2 = St->S2, M = St->M, n_accept = St->n_accept;
  BitRng rng{0u, 0u, 0u, P.key0, P.key1};
  BitDelta d;
  // one word: half a of line j, class line ln of `calls` Philox calls, its `count`
  // first sites
  auto update = [&](int j, int a, int w, int ln, int calls, int count) __attribute__((always_inline)) {
    const int jp = j + 1 == L1 ? 0 : j + 1, jm = j == 0 ? L1 - 1 : j - 1;
    // the word and place that the bit shifted in comes from: west (a = 0) index h - 1 of
    // the odd half, before its first site the line's last; east (a = 1) index h + 1 of
    // the even half, behind its last the line's first
    const bool last = w == hw - 1;
    const int wrap_at = odd ? hw - 1 : 2 * hw - 1;
    const int from = a ? (last ? 0 : w + 1) : (w ? hw + w - 1 : wrap_at);
    const int place = a ? (last ? (n_odd - 1) % W : W - 1) : (w ? W - 1 : wrap_place);
    const uint32_t enter = a && last && odd ? 0u : 1u;
    auto shifted = [&](const uint32_t *line) __attribute__((always_inline)) {
      const uint32_t x = line[(a ? 0 : hw) + w], y = line[from];
      return a ? (x >> 1) | ((y & enter) << place) : (x << 1) | ((y >> place) & 1u);
    };
    uint32_t *own = words + j * rs;
    const uint32_t *up = words + jp * rs, *dn = words + jm * rs;
    const int sa = a * hw + w, so = (1 - a) * hw + w;
    const uint32_t b = own[sa];
    uint32_t c1[3], c2[3] = {0u, 0u, 0u};
    sum4(own[so], shifted(own), up[sa], dn[sa], c1);
    if (NNN) sum4(up[so], shifted(up), dn[so], shifted(dn), c2);
    uint32_t x[8] = {0u, c2[0], c2[1], c2[2], c1[0], c1[1], c1[2], b};
    uint32_t flip;
    if (RING)
      flip = ring_flips<OCT>(x, rng, (uint32_t)(ln * calls + 2 * OCT * w), ltab);
    else if (NNN)
      flip = bit_flips<false, OCT>(x, rng, (uint32_t)(ln * calls + OCT * w),
                                   (uint32_t)(ln * n_odd + W * w), thi, tab);
    else
      flip = pair_flips<OCT>(c1, b, rng, (uint32_t)(ln * calls + OCT * w),
                             (uint32_t)(ln * n_odd + W * w), ltab, tab);
    const int m = count - W * w;
    flip &= m >= W ? FULL : (1u << (m > 0 ? m : 0)) - 1u;
    own[sa] = b ^ flip;
    if (NNN)
      d.add(b, flip, c1, c2);
    else
      d.add(b, flip, c1, (const uint32_t(&)[1])c2);
  };
  // the last site of odd line j (RING), class line ln
  auto seam = [&](int j, int ln) {
    const int jp = j + 1 == L1 ? 0 : j + 1, jm = j == 0 ? L1 - 1 : j - 1;
    const int le = n_even - 1, lo = n_odd - 1;
    auto bit = [&](int row, int a, int h) -> int {
      return (words[row * rs + a * hw + h / W] >> (h % W)) & 1u;
    };
    const int b = bit(j, 0, le);
    const int c1 = bit(j, 1, lo) + bit(j, 0, 0) + bit(jp, 0, le) + bit(jm, 0, le);
    const int c2 = NNN ? bit(jp, 1, lo) + bit(jp, 0, 0) + bit(jm, 1, lo) + bit(jm, 0, 0) : 0;
    if (bit_philox((uint32_t)ln, rng).v[0] > ltab[(b << 6) | (c1 << 3) | c2]) return;
    words[j * rs + le / W] ^= 1u << (le % W);
    (b ? d.n1 : d.n0) += 1;
    (b ? d.c1_1 : d.c1_0) += c1;
    (b ? d.c2_1 : d.c2_0) += c2;
  };
  // this thread's first task as (line, word), and its step
  const int l_first = t / hw, w_first = t - l_first * hw;
  const int l_step = nt / hw, w_step = nt - l_step * hw;
  auto finish = [&](int64_t p) {  // the sums of pass p (thread 0)
    const int nw = (nt + 63) >> 6;
    int s[4] = {0, 0, 0, 0};
    for (int w = 0; w < nw; ++w)
      for (int q = 0; q < 4; ++q) s[q] += red[p & 1][w][q];
    S1 += s[0];
    S2 += s[1];
    M += s[2];
    n_accept += s[3];
    if (p % sample_period != 0) return;
    if (n_samples < series_cap) {
      mcg_sample rec = {};
      rec.pass = p;
      rec.S1 = S1;
      rec.S2 = S2;
      rec.M = M;
      series[(int64_t)c * series_cap + n_samples] = rec;
    }
    ++n_samples;
  };
  for (int64_t k = 0; k < n_passes; ++k) {
    rng.pass_lo = (uint32_t)pass;
    rng.pass_hi = (uint32_t)(pass >> 32);
    const int classes = RING ? 9 : (NNN ? 4 : 2);
    for (int col = 0; col < classes; ++col) {
      // lines j = j_first + j_step * line; RING: class (c0, c1) = (col % 3, col / 3)
      int n_lines, j_first, j_step, count;
      if (RING) {
        const int c0 = col % 3, r1 = col / 3;
        n_lines = r1 == 2 ? (L1 & 1) : (L1 & 1 ? (L1 - 1) >> 1 : L1 >> 1);
        j_first = r1 == 2 ? L1 - 1 : r1;
        j_step = 2;
        count = c0 == 2 ? (L0 & 1) : n_odd;
        if (n_lines == 0 || count == 0) continue;
        rng.color = (uint32_t)col | 0x40000000u;
        if (c0 == 2) {
          for (int line = t; line < n_lines; line += nt) seam(j_first + 2 * line, line);
          __syncthreads();
          continue;
        }
      } else {
        n_lines = NNN ? L1 >> 1 : L1;
        j_first = NNN ? col >> 1 : 0;
        j_step = NNN ? 2 : 1;
        count = n_odd;
        rng.color = (uint32_t)col;
      }
      for (int line = l_first, w = w_first; line < n_lines;) {
        const int j = j_first + j_step * line;
        const int a = RING ? col % 3 : (NNN ? col & 1 : (col + j) & 1);
        update(j, a, w, line, RING ? (n_odd + 3) >> 2 : (n_odd + 7) >> 3, count);
        line += l_step;
        w += w_step;
        if (w >= hw) {
          w -= hw;
          ++line;
        }
      }
      if (col + 1 < classes) __syncthreads();
    }
    ++pass;
    int s[4];
    d.sums(P.z1, P.z2, s);
    d = BitDelta();
#pragma unroll
    for (int q = 0; q < 4; ++q) s[q] = wave_sum_dpp(s[q]);
    if (lane == 63)
      for (int q = 0; q < 4; ++q) red[pass & 1][wid][q] = s[q];
    __syncthreads();
    if (t == 0) finish(pass);
  }
  if (RING) {
    for (int i = t; i < L1 * 2 * hw; i += nt) {
      const int j = i / (2 * hw), r = i - j * 2 * hw, a = r >= hw ? 1 : 0, w = r - a * hw;
      const int m = (a ? n_odd : n_even) - W * w;
      const uint32_t x = words[j * rs + r];
  #pragma unroll
      for (int e = 0; e < W; ++e)
        if (e < m) lat[byte_at(j, a, W * w + e)] = (int8_t)((x >> e) & 1u);
    }
  } else {
#pragma unroll 4
    for (int i = t; i < n8; i += nt) {
      int8_t *p;
      int m;
      const uint32_t x = *eight(i, p, m);
      if (wide) {
        if (m > 0) *reinterpret_cast<uint2 *>(p) = make_uint2(unpack4(x & 15u), unpack4(x >> 4));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (e < m) p[e] = (int8_t)((x >> e) & 1u);
      }
    }
  }
  if (t == 0) {
    St->n_pass = pass;
    St->S1 = S1;
    St->S2 = S2;
    St->M = M;
    St->n_accept = n_accept;
    St->n_samples = n_samples;
  }
}

int word_lds(int L0, int L1, int oct) {
  const int hw = ((L0 + 1) / 2 + 8 * oct - 1) / (8 * oct);
  return 4 * L1 * (2 * hw + 1);
}

int word_tasks(int L0, int L1, bool ring, bool nnn, int oct) {
  const int hw = ((L0 + 1) / 2 + 8 * oct - 1) / (8 * oct);
  return hw * (ring || nnn ? (L1 + 1) / 2 : L1);
}

namespace {

using WordsFn = void (*)(const CheckerParams *, CheckerState *, int8_t *, const uint32_t *,
                         mcg_sample *, int64_t, const uint8_t *, int64_t, int64_t);

template <bool RING, bool NNN>
WordsFn words_fn(int oct) {
  return oct == 1   ? checker_words_kernel<RING, NNN, 1>
         : oct == 2 ? checker_words_kernel<RING, NNN, 2>
         : oct == 3 ? checker_words_kernel<RING, NNN, 3>
                    : checker_words_kernel<RING, NNN, 4>;
}

WordsFn words_fn(bool ring, bool nnn, int oct) {
  return ring ? (nnn ? words_fn<true, true>(oct) : words_fn<true, false>(oct))
              : (nnn ? words_fn<false, true>(oct) : words_fn<false, false>(oct));
}

}  // namespace

void launch_checker_words(const CheckerParams *P, CheckerState *St, int8_t *lat_pool,
                          const uint32_t *tables, mcg_sample *series, int64_t series_cap,
                          const uint8_t *active, int n_chains, int64_t n_passes,
                          int64_t sample_period, bool ring, bool nnn, const WordPlan &w,
                          hipStream_t stream) {
  hipLaunchKernelGGL(words_fn(ring, nnn, w.oct), dim3(n_chains), dim3(w.block), w.lds, stream, P,
                     St, lat_pool, tables, series, series_cap, active, n_passes, sample_period);
}

hipError_t words_set_max_lds() {
  for (int oct = 1; oct <= 4; ++oct)
    for (int k = 0; k < 4; ++k) {
      const hipError_t e = hipFuncSetAttribute(
          reinterpret_cast<const void *>(words_fn(k & 1, k & 2, oct)),
          hipFuncAttributeMaxDynamicSharedMemorySize, WORDS_MAX_LDS);
      if (e != hipSuccess) return e;
    }
  return hipSuccess;
}

int64_t bit_words(const CheckerParams &P) {
  const int64_t w = (int64_t)P.L1 * P.L2 * 2 * bit_hw(P.L0);
  return P.ndim == 2 ? 2 * w : w;
}

int bit_groups(const CheckerParams &P, int oct) { return 64 / bit_parts(P.L0, oct); }

int bit_waves() { return STREAM_BLOCK / 64; }

bool bit_fits(const CheckerParams &P) {
  if (P.quad_only || P.L0 % 32 != 0) return false;
  if (P.ndim == 2) return bit_hw(P.L0) <= 64;
  if (P.L0 % 64 != 0) return false;
  return P.ncolor == 2 || bit_plane_lds(P) <= CHECKER_PLANE_MAX_LDS;
}

int64_t bit_cube_blocks(const CheckerParams &P, int oct) {
  return ((int64_t)P.L1 * P.L2 * bit_hw(P.L0) * (4 / oct) + CUBE_BLOCK - 1) / CUBE_BLOCK;
}

int bit_plane_lds(const CheckerParams &P) { return 3 * 4 * P.L1 * (2 * bit_hw(P.L0) + 1); }

int bit_plane_block(const CheckerParams &P, int oct) {
  const int words = (P.L1 / 2) * bit_hw(P.L0) * (4 / oct);
  return words >= 512 ? 512 : (words + 63) / 64 * 64;
}

// (a grid's second dimension ends at 65535)
template <typename Launch>
static void bit_copy(int64_t max_words, int n_chains, Launch launch) {
  for (int first = 0; first < n_chains; first += 65535)
    launch(dim3((unsigned)((max_words + 255) / 256), (unsigned)std::min(65535, n_chains - first)),
           first);
}

void launch_bit_pack(const CheckerParams *P, const CheckerState *St, const int8_t *lat_pool,
                     uint32_t *bits, const BitItem *chains, int n_chains, int64_t max_words,
                     hipStream_t stream) {
  bit_copy(max_words, n_chains, [&](dim3 grid, int first) {
    hipLaunchKernelGGL(bit_pack_kernel, grid, dim3(256), 0, stream, P, St, lat_pool, bits,
                       chains + first);
  });
}

void launch_bit_unpack(const CheckerParams *P, const CheckerState *St, int8_t *lat_pool,
                       const uint32_t *bits, const BitItem *chains, int n_chains,
                       int64_t max_words, hipStream_t stream) {
  bit_copy(max_words, n_chains, [&](dim3 grid, int first) {
    hipLaunchKernelGGL(bit_unpack_kernel, grid, dim3(256), 0, stream, P, St, lat_pool, bits,
                       chains + first);
  });
}

int bit_pass_launches(const BitPass &b, BitLaunch (&L)[2]) {
  if (b.cube) {
    void *fn = b.oct == 1   ? reinterpret_cast<void *>(&checker_cube_kernel<1>)
               : b.oct == 2 ? reinterpret_cast<void *>(&checker_cube_kernel<2>)
                            : reinterpret_cast<void *>(&checker_cube_kernel<4>);
    for (int color = 0; color < 2; ++color)
      L[color] = {fn, (unsigned)b.n_items, (unsigned)CUBE_BLOCK, 0u, color};
    return 2;
  }
  if (b.plane_lds > 0) {
    void *fn = b.oct == 1   ? reinterpret_cast<void *>(&checker_plane_kernel<1>)
               : b.oct == 2 ? reinterpret_cast<void *>(&checker_plane_kernel<2>)
                            : reinterpret_cast<void *>(&checker_plane_kernel<4>);
    for (int par = 0; par < 2; ++par)
      L[par] = {fn, (unsigned)b.n_items, (unsigned)b.plane_block, (unsigned)b.plane_lds, par};
    return 2;
  }
  void *four = b.oct == 1   ? reinterpret_cast<void *>(&checker_stream_kernel<true, 1>)
               : b.oct == 2 ? reinterpret_cast<void *>(&checker_stream_kernel<true, 2>)
                            : reinterpret_cast<void *>(&checker_stream_kernel<true, 4>);
  void *two = b.oct == 1   ? reinterpret_cast<void *>(&checker_stream_kernel<false, 1>)
              : b.oct == 2 ? reinterpret_cast<void *>(&checker_stream_kernel<false, 2>)
                           : reinterpret_cast<void *>(&checker_stream_kernel<false, 4>);
  L[0] = {b.four ? four : two, (unsigned)(b.n_items / (STREAM_BLOCK / 64)), (unsigned)STREAM_BLOCK, 0u, 0};
  return 1;
}

void launch_bit_pass(const CheckerParams *P, const CheckerState *St, const uint32_t *tables,
                     const BitPass &b, int ahead, hipStream_t stream) {
  BitLaunch L[2];
  const int n = bit_pass_launches(b, L);
  for (int i = 0; i < n; ++i) {
    void *args[] = {(void *)&P,       (void *)&St,         (void *)&b.bits, (void *)&tables,
                    (void *)&b.items, (void *)&L[i].last, (void *)&ahead};
    (void)hipLaunchKernel(L[i].fn, dim3(L[i].grid), dim3(L[i].block), args, L[i].lds, stream);
  }
}

hipError_t bit_set_max_lds() {
  const void *fns[] = {reinterpret_cast<const void *>(&checker_plane_kernel<1>),
                       reinterpret_cast<const void *>(&checker_plane_kernel<2>),
                       reinterpret_cast<const void *>(&checker_plane_kernel<4>)};
  for (const void *fn : fns) {
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             CHECKER_PLANE_MAX_LDS);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace mcg
