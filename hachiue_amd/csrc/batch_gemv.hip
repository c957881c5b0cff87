// The lm_head of several hidden states on gfx950's matrix cores: logits of M
// activation rows from one pass over the weights.
//
// One activation row at a time (lmhead_kernels.hip) reads the whole weight
// tensor again for every row: M rows cost M times one.  Here every 16-row
// tile of the weights is read and taken apart once per slice of 4 to 32
// activation rows.
//
// ---- Q4_K and Q6_K: integers on v_mfma_i32_16x16x64_i8
//
// A weight of a super-block (256 positions) is d * w with w = sc * (q - 32)
// (Q6_K, |w| <= 4096) or w = sc * q (Q4_K, at most 945, the minima apart): an
// integer of 14 bits, held as two int8, w = 256 hi + lo.  x is held as four
// int8 limbs per super-block: with 2^E above the block's largest |x|, x is
// rounded to n 2^(E - 31) and the limbs are n's balanced base-256 digits a_t,
// x = sum_t a_t 2^(E - 7 - 8t) to 2^(E - 32).  An A tile (16 x 64) holds four
// limbs of four activation rows, A row 4 h + t limb t of row h; B (64 x 16)
// one of the two bytes of 16 weight rows.  Eight MFMAs per super-block and A
// tile (four steps of 64 positions, hi and lo) leave in lane (j, h) of the
// result the four exact limb sums of (weight row j, activation row h), in
// magnitude at most 2^27: one product per lane, so the running binary32 sum
// of a tile takes one register per A tile.
// (One row on the same instruction fills a quarter of an A tile with zeros
// around its four limbs; four rows fill it.)
//
// The one-row kernels hold x to 2^(E_g - 28) with an exponent E_g for every
// 16 positions (Q4_0 and Q4_1 hold it in binary32, and round at 2^-25 of a
// block of 32).  Where a super-block's largest |x| is so far above a group's
// that its limbs are coarser than that (E_g < E - 4; for Q4_0 and Q4_1 a
// block's E_b < E - 7), the remainders of such groups become a second set of
// four limbs with an exponent of its own, which a wave adds in a branch for
// the super-blocks and A tiles that have one (outlier channels of 20 times
// the rest and more).  The two sets are no coarser than one row's limbs
// unless the small groups themselves lie more than 2^35 apart.
//
// The limbs are made by a kernel of their own (limbs_kernel) into the
// context's workspace, laid out as the A operands are read; a workgroup
// stages one super-block's A operands at a time in LDS (two buffers, one
// barrier per super-block), each of its waves streams the weights of its own
// tiles through a ring in LDS, as the one-row kernels do.
//
// What bounds it: up to 8 rows the weights' reads (151936 x 2048 Q6_K, 2
// rows: 67 us a call, of which 3 us are limbs_kernel; one row at a time 94
// us; 7 rows 69 and 276 us; Q4_K at K 4096, 7 rows 116 and 448 us), beyond
// that the instructions of a tile: about 250 vector instructions to take it
// apart, 13 per A tile to add its results up, 8 MFMAs per A tile (counters
// at 64 rows: vector units busy 45 % of the cycles, matrix cores 31 %, hardly
// overlapping).  16 rows 82 us (607 one at a time), 64 rows 219 us (2391).
// With four outlier channels of 1000 times the rest, so that half the
// super-blocks have a second set: 7 rows 76 us, 64 rows 276; Q4_K 7 rows 121.
#include "sampler_internal.h"
#include "kq_gemv.h"

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

namespace hs {

namespace bg {
typedef int v4i __attribute__((ext_vector_type(4)));
typedef short v2s __attribute__((ext_vector_type(2)));

// Raw bytes of one super-block of 16 weight rows, and its decode.
template <int FMT> struct Slab;

template <> struct Slab<kW_Q6_K> {
  static constexpr int kBytes = 210;                     // of a row's super-block
  static constexpr int kChunks = q6m::kRowChunks;        // its 16-byte aligned cover
  // bytes of an activation row's record: 2^(E - 7), the second set's or 0
  static constexpr int kRec = 16;
};
template <> struct Slab<kW_Q4_K> {
  static constexpr int kBytes = 144;
  static constexpr int kChunks = q4m::kRowChunks;
  static constexpr int kRec = 48;                        // and from byte 16 eight sums of x
};
template <> struct Slab<kW_Q4_0> {                        // eight blocks
  static constexpr int kBytes = 144;
  static constexpr int kChunks = 9;
  static constexpr int kRec = 16;
};
template <> struct Slab<kW_Q4_1> {
  static constexpr int kBytes = 160;
  static constexpr int kChunks = 10;
  static constexpr int kRec = 48;                        // as Q4_K's
};
template <int FMT> constexpr int slab_bytes() { return 256 * Slab<FMT>::kChunks; }
template <int FMT> constexpr int slab_loads() { return (16 * Slab<FMT>::kChunks + 63) / 64; }

// The A operands of one super-block of HT tiles (four activation rows each):
// [HT][4 steps][64 lanes][16 bytes], then the rows' records.
template <int FMT> constexpr int a_bytes(int ht) { return ht * (4096 + 4 * Slab<FMT>::kRec); }

template <int K>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(K) : "memory");
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// at most `n` slabs of L loads each, and A more loads, in flight
template <int L, int A>
__device__ __forceinline__ void wait_slabs(int n) {
  if (n >= 3) wait_vm<3 * L + A>();
  else if (n == 2) wait_vm<2 * L + A>();
  else if (n == 1) wait_vm<L + A>();
  else wait_vm<A>();
}
// 16 bytes a lane from the resource at `off` to LDS at dst + 16 lane (a
// wave-uniform LDS address), without the compiler's waits (see q6k_gemv.h)
__device__ __forceinline__ void to_lds(v4i rs, uint32_t off, uint32_t dst) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(dst);
  uint32_t keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\t"
      "buffer_load_dwordx4 %2, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
      : "=&s"(keep)
      : "s"(m0), "v"(off), "s"(rs)
      : "memory");
}
// 4 bytes a lane
__device__ __forceinline__ void to_lds4(v4i rs, uint32_t off, uint32_t dst) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(dst);
  uint32_t keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\t"
      "buffer_load_dword %2, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
      : "=&s"(keep)
      : "s"(m0), "v"(off), "s"(rs)
      : "memory");
}
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
  return (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint8_t *)p);
}
__device__ __forceinline__ v4i rsrc(const void *p, uint32_t bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(p);
  return v4i{(int)(uint32_t)b, (int)(uint32_t)(b >> 32), (int)bytes, 0x00020000};
}

// Bytes 0 and 2 (e) and 1 and 3 (o) of four weights as 16-bit pairs, times the
// factor pair, plus the addend pair (which holds 128 more than the value's
// own): the values' high bytes in hi, their low bytes in lo, value = 256 hi +
// lo with both signed.
__device__ __forceinline__ void split4(uint32_t e, uint32_t o, v2s mul, v2s add, int &hi, int &lo) {
  const uint32_t ve = __builtin_bit_cast(uint32_t, (v2s)(__builtin_bit_cast(v2s, e) * mul + add));
  const uint32_t vo = __builtin_bit_cast(uint32_t, (v2s)(__builtin_bit_cast(v2s, o) * mul + add));
  lo = (int)(__builtin_amdgcn_perm(vo, ve, 0x06020400u) ^ 0x80808080u);
  hi = (int)__builtin_amdgcn_perm(vo, ve, 0x07030501u);
}

// The B operands of one super-block of 16 rows from its slab at `rowb` (lane
// (j, G): row j's bytes): high and low bytes of the integer weights of four
// steps, the row's d and, for Q4_K, its dmin and eight minima.
struct BOps {
  v4i hi[4], lo[4];
  float d, dmin, mf[8];
};
// Q6_K: `o` = where the super-block starts in its 16-byte aligned cover
template <int FMT>
__device__ __forceinline__ void decode(const uint8_t *rowb, uint32_t o, int G, BOps &B) {
  if constexpr (FMT == kW_Q6_K) {
    const int nn = G >> 1, h2 = G & 1;
    const q6m::LSrc src{reinterpret_cast<const uint32_t *>(rowb), 0u};
    const uint32_t oa = o + 64u * nn + 16u * h2, ob = oa + 32u, oh = o + 128u + 32u * nn + 16u * h2;
    const uint32_t os = o + 192u + 8u * nn, od = o + 208u;
    q6m::Span<4> qa, qb, qh;
    q6m::Span<2> sc;
    qa.load(src, oa, oa + 15u);
    qb.load(src, ob, ob + 15u);
    qh.load(src, oh, oh + 15u);
    sc.load(src, os, os + 7u);
    B.d = q6m::h2f(src.dw(od & ~3u) >> (8u * (od & 3u)));
    v2s mul[4], add[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t scw = sc.at(k >> 1) >> (8u * (uint32_t)(h2 + 2 * (k & 1)));
      const short f = (short)(int8_t)(scw & 0xFFu);
      const short c0 = (short)(128 - 32 * f);
      mul[k] = v2s{f, f};
      add[k] = v2s{c0, c0};
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t a = qa.at(w), b = qb.at(w), hv = qh.at(w);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        // low nibble from the quarter's ql byte, two bits above it from qh;
        // what lies above bit 5 goes with the 16-bit masks
        const uint32_t lw = k == 0 ? a : k == 1 ? b : k == 2 ? a >> 4 : b >> 4;
        const uint32_t hw = k == 0 ? hv << 4 : k == 1 ? hv << 2 : k == 2 ? hv : hv >> 2;
        const uint32_t u = (lw & 0x0F0F0F0Fu) | (hw & ~0x0F0F0F0Fu);
        int x1, x0;
        split4(u & 0x003F003Fu, (u >> 8) & 0x003F003Fu, mul[k], add[k], x1, x0);
        B.hi[k][w] = x1;
        B.lo[k][w] = x0;
      }
    }
  } else {
    const uint4 hd = *reinterpret_cast<const uint4 *>(rowb);   // d, dmin, the scales
    B.d = q4m::h2f(hd.x);
    B.dmin = q4m::h2f(hd.x >> 16);
    const uint32_t sh = 4u * (uint32_t)(G >> 1), sh8 = sh + 8u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint4 qv = *reinterpret_cast<const uint4 *>(rowb + 16 + 16 * (G & 1) + 32 * k);
      uint32_t s0, m0, s1, m1;
      q4m::scale_min(hd.y, hd.z, hd.w, 2 * k, s0, m0);
      q4m::scale_min(hd.y, hd.z, hd.w, 2 * k + 1, s1, m1);
      B.mf[2 * k] = (float)m0;
      B.mf[2 * k + 1] = (float)m1;
      const short f = (short)(G >> 1 ? s1 : s0);
      const v2s mul = v2s{f, f}, add = v2s{128, 128};
      const uint32_t qd[4] = {qv.x, qv.y, qv.z, qv.w};
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        int x1, x0;
        split4((qd[w] >> sh) & 0x000F000Fu, (qd[w] >> sh8) & 0x000F000Fu, mul, add, x1, x0);
        B.hi[k][w] = x1;
        B.lo[k][w] = x0;
      }
    }
  }
}
}  // namespace bg

namespace bg {
// x to a multiple of 2^(E - 31), 2^E above the |x| of the wave's block: the
// four balanced base-256 digits as bytes, most significant first from byte 3
// down, and what is left of x (both exact)
__device__ __forceinline__ uint32_t digits(float x, int E, float &rest) {
  const float n = rintf(ldexpf(x, 31 - E));
  rest = x - ldexpf(n, E - 31);
  return ((uint32_t)(int)n + 0x80808080u) ^ 0x80808080u;
}
// E with |x| < 2^E for a largest |x| of mx, one more where the digits' largest
// number, 0x7F7F7F7F, would be passed
__device__ __forceinline__ int digits_exp(float mx) {
  int E = 0;
  (void)frexpf(mx, &E);
  return E + (ldexpf(mx, 31 - E) >= 0x7F7F7F80p0f ? 1 : 0);
}
// limb t of four positions from their digits
__device__ __forceinline__ uint32_t limb4(const uint32_t (&u)[4], int t) {
  const uint32_t sel = (uint32_t)(3 - t) | (uint32_t)(7 - t) << 8;   // one byte of each of two
  const uint32_t lo = __builtin_amdgcn_perm(u[1], u[0], sel), hi = __builtin_amdgcn_perm(u[3], u[2], sel);
  return (lo & 0xFFFFu) | hi << 16;
}
}  // namespace bg

// The A operands of activation rows 0..M-1: one wave per (super-block, row),
// four positions a lane.  tab: [ceil(M / 4 ht)][K / 256][a_bytes(ht)], the
// second sets' limbs in the same places from kBatchTabBytes on (written where
// the record says that there is one).  A block with a non-finite element gets
// a NaN scale, which makes every result of its row NaN.
template <int FMT>
__global__ __launch_bounds__(64) void limbs_kernel(const float *x, int64_t ldx, int NS, int ht,
                                                   uint8_t *tab) {
  constexpr bool k32 = FMT == kW_Q4_0 || FMT == kW_Q4_1;
  const int s = (int)blockIdx.x, m = (int)blockIdx.y, lane = (int)threadIdx.x;
  const float *xp = x + (int64_t)m * ldx + 256 * s + 4 * lane;
  float v[4], mx = 0.f;
  bool fin = true;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    v[b] = xp[b];
    mx = fmaxf(mx, fabsf(v[b]));
    fin = fin && __builtin_isfinite(v[b]);
  }
  double sum = ((double)v[0] + (double)v[1]) + ((double)v[2] + (double)v[3]);
#pragma unroll
  for (int o = 4; o > 0; o >>= 1) sum += __shfl_xor(sum, o);   // of the 32 positions of 8 lanes
  fin = __all(fin);
  // the largest of the group that one row's limbs share an exponent in (16
  // positions, 4 lanes; Q4_0 and Q4_1: of the block of 32), then of all
  constexpr int GL = k32 ? 8 : 4;
#pragma unroll
  for (int o = 1; o < GL; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  int Eg = 0;
  (void)frexpf(fin ? mx : 1.f, &Eg);
#pragma unroll
  for (int o = GL; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  const int E = bg::digits_exp(fin ? mx : 1.f);
  const bool coarse = Eg < E - (k32 ? 7 : 4);
  uint32_t u[4];
  float rest[4], mr = 0.f;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    u[b] = bg::digits(fin ? v[b] : 0.f, E, rest[b]);
    if (!coarse) rest[b] = 0.f;
    mr = fmaxf(mr, fabsf(rest[b]));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mr = fmaxf(mr, __shfl_xor(mr, o));
  // where the weights of position p sit in B: step and lane group (Q6_K:
  // p = 128 n + 32 step + 16 h + b in group 2 n + h, the quarters of a half
  // share their bytes; Q4_K: in order; Q4_0 and Q4_1, steps of 32: group G
  // has the low, then the high nibbles of bytes 4 G .. 4 G + 3)
  constexpr int W = k32 ? 8 : 16;   // bytes of a lane's A operand
  const int p = 4 * lane;
  const int step = k32 ? p >> 5 : FMT == kW_Q6_K ? (p >> 5) & 3 : p >> 6;
  const int G = k32 ? (p >> 2) & 3 : FMT == kW_Q6_K ? 2 * (p >> 7) + ((p >> 4) & 1) : (p >> 4) & 3;
  const int at = k32 ? 4 * ((p >> 4) & 1) : p & 15;
  const int hid = m % (4 * ht);
  uint8_t *a = tab + ((int64_t)(m / (4 * ht)) * NS + s) * bg::a_bytes<FMT>(ht);
  uint8_t *d = a + (hid >> 2) * 4096 + step * 64 * W + (16 * G + 4 * (hid & 3)) * W + at;
#pragma unroll
  for (int t = 0; t < 4; ++t) *reinterpret_cast<uint32_t *>(d + W * t) = bg::limb4(u, t);
  float scale2 = 0.f;
  if (mr > 0.f) {   // (uniform)
    const int E2 = bg::digits_exp(mr);
    scale2 = ldexpf(1.f, E2 - 7);
    float lost;
#pragma unroll
    for (int b = 0; b < 4; ++b) u[b] = bg::digits(rest[b], E2, lost);
    d += kBatchTabBytes;
#pragma unroll
    for (int t = 0; t < 4; ++t) *reinterpret_cast<uint32_t *>(d + W * t) = bg::limb4(u, t);
  }
  float *rec = reinterpret_cast<float *>(a + ht * 4096 + hid * bg::Slab<FMT>::kRec);
  if (lane == 0) {
    rec[0] = fin ? ldexpf(1.f, E - 7) : __builtin_nanf("");
    rec[1] = scale2;
  }
  if (bg::Slab<FMT>::kRec > 16 && (lane & 7) == 0)   // (Q4_1: in units of the first limb's)
    rec[4 + (lane >> 3)] = (float)(FMT == kW_Q4_1 ? ldexp(sum, 7 - E) : sum);
}

// Measured at 151936 x 2048, us a call, against one row at a time: Q1_0 4
// rows 20 (54), 64 rows 118 (828); PQ2_0 4 rows 23 (63), 16 rows 41 (226);
// PTQ1_0 4 rows 40 (79), 8 rows 44 (155); Q4_0, K 1024, 4 rows 29 (86), 64
// rows 125 (1220); Q4_1 4 rows 52 (137), 16 rows 81 (484); F32, K 1024, 4 rows
// 149 (432), 64 rows 220 (6871).  Errors against binary64, K 2048, rms over
// the logits' rms, and one row's: Q6_K 5.9e-8 (8.5e-8), Q4_K 6.9e-8 (9.0e-8),
// Q4_0 8.2e-8 (2.3e-7), Q4_1 1.1e-7 (1.3e-7), F32 1.1e-7 (1.2e-7).

// ---- the stream, shared by the formats
//
// A grid of groups x slices workgroups of NW waves.  A wave's tiles (16 weight
// rows each) are gw, gw + nwx, ... (at any time the waves read neighbouring
// tiles, and the tiles of a last, partial round spread over all workgroups),
// taken in passes of at most RT; a pass goes through the row's NS slabs in
// order, each over the pass's tiles.  The items (pass, slab, tile) stream
// through the wave's ring of NB slabs in LDS; a step (pass, slab) has its A
// operands in LDS for the whole workgroup, those of the next step on their
// way into a second buffer.
//
// Body (per format) has kLoads and kSlab (loads and LDS bytes of a slab),
// kA (A bytes of a step), and
//   at(s), go(tile, dst)  the loads of slab s of a tile into LDS at dst
//   zero(t)               a pass begins for its tile t
//   step(ab)              a step's A operands are at ab
//   take(t, tile, s, cur) the tile's slab s is at cur
//   put(t, tile)          the pass's tile t is complete
template <class Body, int RT, int NW, int NB>
__device__ __forceinline__ void batch_stream(Body &body, const uint8_t *atab, int NS, int N, int slices,
                                             int groups, uint8_t *lds) {
  using namespace bg;
  constexpr int L = Body::kLoads, SB = Body::kSlab, AB = Body::kA;
  // A loads of a wave (1 KiB each; past the last piece a wave reads that one
  // again, so that every wave has the same count in flight)
  constexpr int AP = (AB + 1023) / 1024, AL = (AP + NW - 1) / NW;
  static_assert(NB >= 2 && NB <= 4 && 3 * L + AL < 64, "wait_slabs counts");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint8_t *ring = lds + 2 * AB + wave * NB * SB;
  const uint32_t abuf_a = lds_addr(lds), ring_a = lds_addr(ring);
  // Workgroups b, b + 8, ... of one XCD: the slices of one group of tiles are
  // neighbours there and share the weights in its L2
  const int b = (int)blockIdx.x, xg = ((b >> 3) / slices) * 8 + (b & 7);
  const int ntiles = (N + 15) >> 4;
  const int nwx = groups * NW, gw = wave * groups + xg;
  const int cnt = gw < ntiles ? (ntiles - 1 - gw) / nwx + 1 : 0;
  const int maxcnt = (ntiles - 1) / nwx + 1;
  const int np = (maxcnt + RT - 1) / RT;
  auto plo = [&](int p) {   // first tile of pass p
    const int i = p * maxcnt / np;
    return i < cnt ? i : cnt;
  };
  const int total = cnt * NS;
  const v4i ra = rsrc(atab, (uint32_t)(NS * AB));

  // next slab to issue: its tile, slab and ring slot
  int iz = 0, is = 0, ip = 0, ilo = 0, ihi = plo(1), ii = 0, islot = 0;
  body.at(0);
  auto issue = [&]() {
    body.go(gw + ii * nwx, ring_a + islot * SB);
    ++iz;
    islot = islot + 1 == NB ? 0 : islot + 1;
    if (++ii == ihi) {
      ii = ilo;
      if (++is == NS) {
        is = 0;
        ++ip;
        ilo = ihi;
        ihi = plo(ip + 1);
        ii = ilo;
      }
      body.at(is);
    }
  };
  auto issue_a = [&](int s, uint32_t dst) {
#pragma unroll
    for (int c = 0; c < AL; ++c) {
      const int i = c * NW + wave < AP ? c * NW + wave : AP - 1;
      const uint32_t o = (uint32_t)(i * 1024 + 16 * lane);
      if (AB % 1024 == 0 || o < (uint32_t)AB) to_lds(ra, (uint32_t)(s * AB) + o, dst + i * 1024);
    }
  };

  issue_a(0, abuf_a);
#pragma unroll
  for (int k = 0; k < NB - 1; ++k)
    if (iz < total) issue();
  int z = 0, slot = 0;
  int iza = 0;   // slabs issued before the latest A loads
  for (int p = 0; p < np; ++p) {
    const int lo = plo(p), n = plo(p + 1) - lo;
#pragma unroll
    for (int t = 0; t < RT; ++t) body.zero(t);
    for (int s = 0; s < NS; ++s) {
      const int q = p * NS + s;
      // this wave's share of A has arrived (the slabs issued after it may
      // still be in flight), its reads of the other buffer are done
      wait_slabs<L, 0>(iz - iza < iz - z ? iz - iza : iz - z);
      wait_lds();
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const bool more = q + 1 < np * NS;
      if (more) {
        issue_a(s + 1 == NS ? 0 : s + 1, abuf_a + ((q + 1) & 1) * AB);
        iza = iz;
      }
      body.step(lds + (q & 1) * AB);
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        if (t < n) {
          wait_lds();   // the previous slab's reads are done: its slot is free
          if (iz < total) issue();
          // slab z has arrived: the later slabs may be in flight, and the A
          // loads where they were issued after it
          if (z < iza && more) wait_slabs<L, AL>(iz - z - 1);
          else wait_slabs<L, 0>(iz - z - 1);
          const uint8_t *cur = ring + slot * SB;
          slot = slot + 1 == NB ? 0 : slot + 1;
          ++z;
          body.take(t, gw + (lo + t) * nwx, s, cur);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t)
      if (t < n) body.put(t, gw + (lo + t) * nwx);
  }
}
// the slice of activation rows of this workgroup (see batch_stream)
__device__ __forceinline__ int batch_slice(int slices) { return ((int)blockIdx.x >> 3) % slices; }

// ---- Q4_K and Q6_K

namespace bg {
// the four limb sums of a product, in units of the first limb's
__device__ __forceinline__ float limb_sum(v4i d) {
  float val = fmaf((float)d[3], 0x1p-8f, (float)d[2]);
  val = fmaf(val, 0x1p-8f, (float)d[1]);
  return fmaf(val, 0x1p-8f, (float)d[0]);
}
// bit r: row r of the slice (`rows` of them exist) has a second set of limbs
// in the step whose records are at rec
template <int FMT, int HT>
__device__ __forceinline__ uint32_t second_rows(const uint8_t *rec, int lane, int rows) {
  static_assert(4 * HT <= 32, "a bit a row");
  float s = 0.f;
  if (lane < 4 * HT && lane < rows) s = *reinterpret_cast<const float *>(rec + lane * Slab<FMT>::kRec + 4);
  return (uint32_t)__builtin_amdgcn_ballot_w64(s > 0.f);
}
}  // namespace bg

template <int FMT, int HT, int RT, bool HOLD>
struct KqBatch {
  using S = bg::Slab<FMT>;
  using v4i = bg::v4i;
  static constexpr int kLoads = bg::slab_loads<FMT>(), kSlab = bg::slab_bytes<FMT>();
  static constexpr int kA = bg::a_bytes<FMT>(HT);
  const GemvArgs &g;
  const int slice, lane, j, G;
  const v4i rw;
  uint32_t vo[kLoads];   // a lane's byte offset in a tile, per load
  const uint8_t *ab, *rec;
  const uint8_t *second;   // the slice's second sets
  uint32_t more;           // rows of the slice that have one in this step
  v4i A[HOLD ? HT : 1][4];
  float xs[HT];
  float acc[RT][HT];

  __device__ __forceinline__ KqBatch(const GemvArgs &args, const uint8_t *tab, int sl)
      : g(args), slice(sl), lane(threadIdx.x & 63), j(lane & 15), G(lane >> 4),
        rw(bg::rsrc(args.w, (args.w_bytes + 15u) & ~15u)), second(tab + kBatchTabBytes) {}
  // (rows at and past N lie past the resource, or wrap to its start: unused)
  __device__ __forceinline__ void at(int s) {
#pragma unroll
    for (int c = 0; c < kLoads; ++c) {
      const int q = c * 64 + lane, rj = q / S::kChunks, cc = q % S::kChunks;
      vo[c] = (((uint32_t)rj * g.row_bytes + (uint32_t)S::kBytes * (uint32_t)s) & ~15u) + 16u * (uint32_t)cc;
    }
  }
  __device__ __forceinline__ void go(int tile, uint32_t dst) {
    const uint32_t base = (uint32_t)tile * 16u * g.row_bytes;   // a multiple of 16
#pragma unroll
    for (int c = 0; c < kLoads; ++c)
      if (c + 1 < kLoads || 16 * S::kChunks % 64 == 0 || lane < 16 * S::kChunks % 64)
        bg::to_lds(rw, base + vo[c], dst + c * 1024);
  }
  __device__ __forceinline__ void zero(int t) {
#pragma unroll
    for (int h = 0; h < HT; ++h) acc[t][h] = 0.f;
  }
  __device__ __forceinline__ v4i a_op(int h, int k) const {
    return *reinterpret_cast<const v4i *>(ab + h * 4096 + k * 1024 + lane * 16);
  }
  __device__ __forceinline__ void step(const uint8_t *a) {
    ab = a;
    rec = a + HT * 4096;
    more = bg::second_rows<FMT, HT>(rec, lane, g.M - slice * 4 * HT);
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      if constexpr (HOLD)
#pragma unroll
        for (int k = 0; k < 4; ++k) A[h][k] = a_op(h, k);
      xs[h] = *reinterpret_cast<const float *>(rec + (4 * h + G) * S::kRec);
    }
  }
  __device__ __forceinline__ void take(int t, int tile, int s, const uint8_t *cur) {
    const uint32_t o = FMT == kW_Q6_K
                           ? ((uint32_t)(tile * 16 + j) * g.row_bytes + 210u * (uint32_t)s) & 15u
                           : 0u;
    bg::BOps B;
    bg::decode<FMT>(cur + j * 16 * S::kChunks, o, G, B);
    // HP A tiles at a time: 2 HP independent accumulator chains (one for
    // Q4_K at HT 8, whose minima take the registers)
    constexpr int HP = HT < 2 || (HT == 8 && FMT == kW_Q4_K) ? 1 : 2;
#pragma unroll
    for (int h0 = 0; h0 < HT; h0 += HP) {
      v4i hi[HP], lw[HP];
#pragma unroll
      for (int h = 0; h < HP; ++h) hi[h] = lw[h] = v4i{0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int h = 0; h < HP; ++h) {
          const v4i a = HOLD ? A[HOLD ? h0 + h : 0][k] : a_op(h0 + h, k);
          hi[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, B.hi[k], hi[h], 0, 0, 0);
          lw[h] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, B.lo[k], lw[h], 0, 0, 0);
        }
#pragma unroll
      for (int h = 0; h < HP; ++h) {
        // times a power of two (d times that could pass the binary32 range
        // where no product of x does)
        const float val = bg::limb_sum(hi[h] * 256 + lw[h]) * xs[h0 + h];
        if constexpr (FMT == kW_Q4_K) {   // the minima: - dmin sum_s m_s (sub-block s's sum of x)
          const float4 *xr = reinterpret_cast<const float4 *>(rec + (4 * (h0 + h) + G) * S::kRec + 16);
          const float4 u = xr[0], v = xr[1];
          const float sa = fmaf(B.mf[1], u.y, B.mf[0] * u.x), sb = fmaf(B.mf[3], u.w, B.mf[2] * u.z);
          const float sc = fmaf(B.mf[5], v.y, B.mf[4] * v.x), sd = fmaf(B.mf[7], v.w, B.mf[6] * v.z);
          acc[t][h0 + h] += fmaf(B.d, val, -B.dmin * ((sa + sb) + (sc + sd)));
        } else {
          acc[t][h0 + h] = fmaf(B.d, val, acc[t][h0 + h]);
        }
      }
    }
    if (__builtin_expect(more != 0u, 0)) {   // (wave-uniform; read from the table itself)
      const uint8_t *a2 = second + (int64_t)s * kA + lane * 16;
#pragma unroll
      for (int h = 0; h < HT; ++h) {
        if (!(more >> (4 * h) & 15u)) continue;
        v4i hi = v4i{0, 0, 0, 0}, lw = hi;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const v4i a = *reinterpret_cast<const v4i *>(a2 + h * 4096 + k * 1024);
          hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, B.hi[k], hi, 0, 0, 0);
          lw = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, B.lo[k], lw, 0, 0, 0);
        }
        const float xs2 = *reinterpret_cast<const float *>(rec + (4 * h + G) * S::kRec + 4);
        acc[t][h] = fmaf(B.d, bg::limb_sum(hi * 256 + lw) * xs2, acc[t][h]);
      }
    }
  }
  __device__ __forceinline__ void put(int t, int tile) {
    const int row = tile * 16 + j;
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      const int m = slice * 4 * HT + 4 * h + G;
      if (row < g.N && m < g.M) g.y[(int64_t)m * g.ldy + row] = acc[t][h];
    }
  }
};

template <int FMT, int HT, int RT, int NW, int NB, bool HOLD>
__global__ __launch_bounds__(64 * NW, NW / 4) void gemv_batch_kq_kernel(GemvArgs g, const uint8_t *tab,
                                                                        int slices, int groups) {
  extern __shared__ uint4 blds[];
  const int slice = batch_slice(slices), NS = g.K / 256;
  tab += (int64_t)slice * NS * bg::a_bytes<FMT>(HT);
  KqBatch<FMT, HT, RT, HOLD> body(g, tab, slice);
  batch_stream<KqBatch<FMT, HT, RT, HOLD>, RT, NW, NB>(body, tab, NS, g.N, slices, groups,
                                                       reinterpret_cast<uint8_t *>(blds));
}

// ---- Q1_0, PQ2_0, PTQ1_0: the codes are bytes as they are
//
// A weight is d * (c1 * code - 1) per block of 128 positions (tern_gemv.h),
// x four int8 limbs per block, an A tile again four limbs of four rows.  A
// slab is four blocks; of each block lane group G decodes 32 codes, two B
// operands, in the order their bytes decode most cheaply:
//   Q1_0    dword G of the block, step a: bits 4a + w of its bytes;
//   PQ2_0   dwords 2G + a, codes w of their bytes;
//   PTQ1_0  step 0 trits 0..3 of bytes 4G .. 4G + 3; step 1 trits 0..3 of
//           bytes 16..19 (G 0) and 20..23 (G 1), trit 4 of bytes 0..15 (G 2),
//           trit 4 of bytes 16..23 and the trits of bytes 24 and 25 (G 3).
// A trit is ((b 3^n mod 256) 3) >> 8, two 16-bit products each for two bytes.
// The accumulators start at minus the block's limb totals, so the result's
// lane holds c1 sum a code - sum a, exact, two limbs to a 32-bit sum.
namespace bg {
constexpr int kTernA = 8192, kTernRec = 128;   // per A tile and step; per row and step
constexpr int tern_a_bytes(int ht) { return ht * (kTernA + 4 * kTernRec); }
template <int FMT> constexpr int tern_row() { return 4 * tern_quant_bytes(FMT); }   // slab bytes of a row
// position p of a block: its step, lane group, B dword and byte
template <int FMT>
__device__ __forceinline__ void tern_place(int p, int &a, int &G, int &w, int &m) {
  if constexpr (FMT == kW_Q1_0) {
    G = p >> 5; m = (p >> 3) & 3; a = (p >> 2) & 1; w = p & 3;
  } else if constexpr (FMT == kW_PQ2_0) {
    G = p >> 5; a = (p >> 4) & 1; m = (p >> 2) & 3; w = p & 3;
  } else if (p < 64) {
    a = 0; w = p >> 4; G = (p >> 2) & 3; m = p & 3;
  } else if (p < 80) {
    a = 1; G = 2; w = (p >> 2) & 3; m = p & 3;
  } else if (p < 112) {
    a = 1; w = (p - 80) >> 3; G = (p >> 2) & 1; m = p & 3;
  } else if (p < 120) {
    a = 1; G = 3; w = (p >> 2) & 1; m = p & 3;
  } else {
    a = 1; G = 3; w = 2 + ((p >> 2) & 1); m = p & 3;
  }
}
// four trits, one of each byte of s: byte 0 and 2 of 3^n in `mul` (as 16-bit
// halves), bytes 1 and 3 alike
__device__ __forceinline__ int trits(uint32_t s, uint32_t mul) {
  const v2s f = __builtin_bit_cast(v2s, mul), three = v2s{3, 3};
  const v2s e = __builtin_bit_cast(v2s, s & 0x00FF00FFu) * f;
  const v2s o = __builtin_bit_cast(v2s, (s >> 8) & 0x00FF00FFu) * f;
  const v2s te = __builtin_bit_cast(v2s, __builtin_bit_cast(uint32_t, e) & 0x00FF00FFu) * three;
  const v2s to = __builtin_bit_cast(v2s, __builtin_bit_cast(uint32_t, o) & 0x00FF00FFu) * three;
  return (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, to), __builtin_bit_cast(uint32_t, te),
                                    0x07030501u);
}
}  // namespace bg

// one wave per (block, row), two positions a lane.  tab: [slice][K / 512]
// [tern_a_bytes(ht)]; a row's record per block: minus its four limb totals,
// the scales of the two limb pairs.
template <int FMT>
__global__ __launch_bounds__(64) void tern_limbs_kernel(const float *x, int64_t ldx, int NS, int ht,
                                                        uint8_t *tab) {
  constexpr int C1 = FMT == kW_Q1_0 ? 2 : 1;
  const int blk = (int)blockIdx.x, m = (int)blockIdx.y, lane = (int)threadIdx.x;
  const float *xp = x + (int64_t)m * ldx + 128 * blk;
  float v[2] = {xp[lane], xp[64 + lane]};
  float mx = fmaxf(fabsf(v[0]), fabsf(v[1]));
  const bool fin = __all(__builtin_isfinite(v[0]) && __builtin_isfinite(v[1]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  int E = 0;
  (void)frexpf(fin ? mx : 1.f, &E);   // mx < 2^E
  // Q1_0 takes its limbs doubled (c1 = 2 folded into A): one more bit of
  // headroom keeps 2 a within int8
  E += C1 == 2 ? 1 : 0;
  const int hid = m % (4 * ht), b = blk & 3;
  uint8_t *tb = tab + ((int64_t)(m / (4 * ht)) * NS + (blk >> 2)) * bg::tern_a_bytes(ht);
  uint8_t *d = tb + (hid >> 2) * bg::kTernA + b * 2048 + 4 * (hid & 3) * 16;
  int tot[4] = {0, 0, 0, 0};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    // x rounded to a multiple of 2^(E - 27), then its balanced base-128
    // digits (as in tern_gemv.h)
    int nn = fin ? (int)rintf(ldexpf(v[h], 27 - E)) : 0;
    int dig[4];
#pragma unroll
    for (int t = 3; t > 0; --t) {
      dig[t] = ((nn + 64) & 127) - 64;
      nn = (nn - dig[t]) >> 7;
    }
    dig[0] = nn;
    int a, G, w, mm;
    bg::tern_place<FMT>(64 * h + lane, a, G, w, mm);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      d[a * 1024 + (16 * G + t) * 16 + 4 * w + mm] = (uint8_t)(C1 * dig[t]);
      tot[t] += dig[t];
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) tot[t] += __shfl_xor(tot[t], o);
  if (lane == 0) {
    int *rec = reinterpret_cast<int *>(tb + ht * bg::kTernA + hid * bg::kTernRec + b * 32);
#pragma unroll
    for (int t = 0; t < 4; ++t) rec[t] = -tot[t];
    rec[4] = __float_as_int(fin ? ldexpf(1.f, E - 13) : __builtin_nanf(""));
    rec[5] = __float_as_int(ldexpf(1.f, E - 27));
  }
}

template <int FMT, int HT, int RT>
struct TernBatch {
  using v4i = bg::v4i;
  static constexpr int kRow = bg::tern_row<FMT>();
  // PTQ1_0's slabs (26 dwords a row, 4-byte aligned) go in loads of 4 bytes a
  // lane, the others' in loads of 16; then the 16 rows' four binary16 scales
  static constexpr int kQuant = FMT == kW_PTQ1_0 ? (16 * kRow / 4 + 63) / 64 : 16 * kRow / 1024;
  static constexpr int kLoads = kQuant + 1;
  static constexpr int kSlab = 16 * kRow + 128;
  static constexpr int kA = bg::tern_a_bytes(HT);
  const GemvArgs &g;
  const int slice, lane, j, G;
  const uint32_t nb;     // blocks of a row
  const v4i rw, rs;
  uint32_t vo[kQuant], so;
  uint32_t mul[4];       // PTQ1_0: step 1's powers of three of the lane group
  const uint8_t *ab;
  float acc[RT][HT];

  __device__ __forceinline__ TernBatch(const GemvArgs &args, int sl)
      : g(args), slice(sl), lane(threadIdx.x & 63), j(lane & 15), G(lane >> 4), nb((uint32_t)(args.K / 128)),
        rw(bg::rsrc(args.w, (args.w_bytes + 3u) & ~3u)), rs(bg::rsrc(args.scales, (args.s_bytes + 3u) & ~3u)) {
    if constexpr (FMT == kW_PTQ1_0) {
      mul[0] = G < 2 ? 0x00010001u : 0x00510051u;
      mul[1] = G < 2 ? 0x00030003u : 0x00510051u;
      mul[2] = G < 2 ? 0x00090009u : G == 2 ? 0x00510051u : 0x00030001u;
      mul[3] = G < 2 ? 0x001B001Bu : G == 2 ? 0x00510051u : 0x001B0009u;
    }
  }
  // (16-byte pieces of a row are stored in the order piece ^ (row's bits), so
  // that the 16 rows' reads of one piece spread over the banks)
  // the lane group's of four values (by value: a choice of lvalues would be a
  // choice of addresses)
  __device__ __forceinline__ uint32_t by_group(uint32_t a, uint32_t b, uint32_t c, uint32_t d) const {
    const uint32_t ab2 = G & 1 ? b : a, cd = G & 1 ? d : c;
    return G & 2 ? cd : ab2;
  }
  static __device__ __forceinline__ int mix(int row) { return FMT == kW_Q1_0 ? (row >> 2) & 3 : row & 7; }
  __device__ __forceinline__ void at(int s) {
#pragma unroll
    for (int c = 0; c < kQuant; ++c) {
      const int q = c * 64 + lane;
      if constexpr (FMT == kW_PTQ1_0) {
        const int rj = q / (kRow / 4), cc = q % (kRow / 4);
        vo[c] = (uint32_t)rj * g.row_bytes + (uint32_t)(s * kRow) + 4u * (uint32_t)cc;
      } else {
        constexpr int P = kRow / 16;
        const int rj = q / P, cc = (q % P) ^ mix(rj);
        vo[c] = (uint32_t)rj * g.row_bytes + (uint32_t)(s * kRow) + 16u * (uint32_t)cc;
      }
    }
    so = ((uint32_t)(lane >> 1) * nb + 4u * (uint32_t)s) * 2u + 4u * (uint32_t)(lane & 1);
  }
  __device__ __forceinline__ void go(int tile, uint32_t dst) {
    const uint32_t base = (uint32_t)tile * 16u * g.row_bytes;
#pragma unroll
    for (int c = 0; c < kQuant; ++c) {
      if constexpr (FMT == kW_PTQ1_0) {
        if (c + 1 < kQuant || lane < 16 * kRow / 4 - 64 * (kQuant - 1)) bg::to_lds4(rw, base + vo[c], dst + c * 256);
      } else {
        bg::to_lds(rw, base + vo[c], dst + c * 1024);
      }
    }
    if (lane < 32) bg::to_lds4(rs, (uint32_t)tile * 32u * nb + so, dst + 16 * kRow);
  }
  __device__ __forceinline__ void zero(int t) {
#pragma unroll
    for (int h = 0; h < HT; ++h) acc[t][h] = 0.f;
  }
  __device__ __forceinline__ void step(const uint8_t *a) { ab = a; }
  __device__ __forceinline__ void take(int t, int, int, const uint8_t *cur) {
    const uint8_t *rowb = cur + j * kRow;
    const uint2 sc = *reinterpret_cast<const uint2 *>(cur + 16 * kRow + 8 * j);
    uint32_t q[4][FMT == kW_PTQ1_0 ? 7 : FMT == kW_PQ2_0 ? 2 : 1];
    auto read = [&](int b) {
      if constexpr (FMT == kW_Q1_0) {
        q[b][0] = *reinterpret_cast<const uint32_t *>(rowb + 16 * (b ^ mix(j)) + 4 * G);
      } else if constexpr (FMT == kW_PQ2_0) {
        const uint2 x = *reinterpret_cast<const uint2 *>(rowb + 16 * ((2 * b + (G >> 1)) ^ mix(j)) + 8 * (G & 1));
        q[b][0] = x.x;
        q[b][1] = x.y;
      } else {
        const uint32_t *p = reinterpret_cast<const uint32_t *>(rowb) + (26 * b) / 4;
        uint32_t d[7];
#pragma unroll
        for (int i = 0; i < 7; ++i) d[i] = p[i];
#pragma unroll
        for (int i = 0; i < 7; ++i)   // block b starts 2 (b & 1) bytes into its first dword
          q[b][i] = b & 1 ? (i < 6 ? __builtin_amdgcn_alignbyte(d[i + 1 < 7 ? i + 1 : 6], d[i], 2) : d[6] >> 16)
                          : d[i];
      }
    };
    // (PTQ1_0: one block ahead)
#pragma unroll
    for (int b = 0; b < (FMT == kW_PTQ1_0 ? 1 : 4); ++b) read(b);
    float sum[HT];   // the slab's four blocks, then added to the row's sum
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if (FMT == kW_PTQ1_0 && b < 3) read(b + 1);
      v4i B[2];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if constexpr (FMT == kW_Q1_0) {
          B[0][w] = (int)((q[b][0] >> w) & 0x01010101u);
          B[1][w] = (int)((q[b][0] >> (4 + w)) & 0x01010101u);
        } else if constexpr (FMT == kW_PQ2_0) {
          B[0][w] = (int)((q[b][0] >> (2 * w)) & 0x03030303u);
          B[1][w] = (int)((q[b][1] >> (2 * w)) & 0x03030303u);
        } else {
          constexpr uint32_t pw[4] = {0x00010001u, 0x00030003u, 0x00090009u, 0x001B001Bu};
          uint32_t x[7];
#pragma unroll
          for (int i = 0; i < 7; ++i) x[i] = q[b][i];
          const uint32_t tail = (x[6] & 0xFFFFu) | (x[6] << 16);
          const uint32_t s0 = by_group(x[0], x[1], x[2], x[3]);
          const uint32_t s1 = by_group(x[4], x[5], x[w], w == 0 ? x[4] : w == 1 ? x[5] : tail);
          B[0][w] = bg::trits(s0, pw[w]);
          B[1][w] = bg::trits(s1, mul[w]);
        }
      }
      const float d = q6m::h2f(b & 1 ? (b < 2 ? sc.x : sc.y) >> 16 : (b < 2 ? sc.x : sc.y));
#pragma unroll
      for (int h = 0; h < HT; ++h) {
        const uint8_t *at_ = ab + h * bg::kTernA + b * 2048 + lane * 16;
        const uint8_t *rec = ab + HT * bg::kTernA + (4 * h + G) * bg::kTernRec + b * 32;
        v4i D = *reinterpret_cast<const v4i *>(rec);
        const float2 ls = *reinterpret_cast<const float2 *>(rec + 16);
        D = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const v4i *>(at_), B[0], D, 0, 0, 0);
        D = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const v4i *>(at_ + 1024), B[1], D, 0, 0, 0);
        const int H = (D[0] << 7) + D[1], Lo = (D[2] << 7) + D[3];   // (|.| < 2^23)
        const float val = fmaf((float)Lo, ls.y, (float)H * ls.x);
        sum[h] = b == 0 ? val * d : fmaf(val, d, sum[h]);
      }
    }
#pragma unroll
    for (int h = 0; h < HT; ++h) acc[t][h] += sum[h];
  }
  __device__ __forceinline__ void put(int t, int tile) {
    const int row = tile * 16 + j;
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      const int m = slice * 4 * HT + 4 * h + G;
      if (row < g.N && m < g.M) g.y[(int64_t)m * g.ldy + row] = acc[t][h];
    }
  }
};

template <int FMT, int HT, int RT, int NW, int NB>
__global__ __launch_bounds__(64 * NW, NW / 4) void gemv_batch_tern_kernel(GemvArgs g, const uint8_t *tab,
                                                                          int slices, int groups) {
  extern __shared__ uint4 blds[];
  using Body = TernBatch<FMT, HT, RT>;
  const int slice = batch_slice(slices), NS = g.K / 512;
  Body body(g, slice);
  batch_stream<Body, RT, NW, NB>(body, tab + (int64_t)slice * NS * Body::kA, NS, g.N, slices, groups,
                                 reinterpret_cast<uint8_t *>(blds));
}

// ---- Q4_0, Q4_1: blocks of 32 on v_mfma_i32_16x16x32_i8
//
// A weight is d * (q - 8) or d * q + m with a binary16 d (and m) per block of
// 32, so a block's limb sums leave the matrix cores each: one MFMA of 32
// positions per block and A tile, B the block's q - 8 or q of 16 rows.  Lane
// (j, G) takes the low, then the high nibbles of dword G of its row's block.
// x as for the K-quants, limbs per 256 positions (eight blocks, one slab), so
// 2^(E - 7) multiplies the slab's sum once.
template <int FMT, int HT, int RT>
struct Q4Batch {
  using S = bg::Slab<FMT>;
  using v4i = bg::v4i;
  static constexpr int kLoads = bg::slab_loads<FMT>(), kSlab = bg::slab_bytes<FMT>();
  static constexpr int kA = bg::a_bytes<FMT>(HT);
  const GemvArgs &g;
  const int slice, lane, j, G;
  const v4i rw;
  uint32_t vo[kLoads];
  const uint8_t *ab;
  const uint8_t *second;   // as KqBatch's
  uint32_t more;
  float acc[RT][HT];

  __device__ __forceinline__ Q4Batch(const GemvArgs &args, const uint8_t *tab, int sl)
      : g(args), slice(sl), lane(threadIdx.x & 63), j(lane & 15), G(lane >> 4),
        rw(bg::rsrc(args.w, (args.w_bytes + 15u) & ~15u)), second(tab + kBatchTabBytes) {}
  __device__ __forceinline__ void at(int s) {
#pragma unroll
    for (int c = 0; c < kLoads; ++c) {
      const int q = c * 64 + lane, rj = q / S::kChunks, cc = q % S::kChunks;
      vo[c] = (uint32_t)rj * g.row_bytes + (uint32_t)(S::kBytes * s) + 16u * (uint32_t)cc;
    }
  }
  __device__ __forceinline__ void go(int tile, uint32_t dst) {
    const uint32_t base = (uint32_t)tile * 16u * g.row_bytes;
#pragma unroll
    for (int c = 0; c < kLoads; ++c)
      if (c + 1 < kLoads || 16 * S::kChunks % 64 == 0 || lane < 16 * S::kChunks % 64)
        bg::to_lds(rw, base + vo[c], dst + c * 1024);
  }
  __device__ __forceinline__ void zero(int t) {
#pragma unroll
    for (int h = 0; h < HT; ++h) acc[t][h] = 0.f;
  }
  __device__ __forceinline__ void step(const uint8_t *a) {
    ab = a;
    more = bg::second_rows<FMT, HT>(a + HT * 4096, lane, g.M - slice * 4 * HT);
  }
  // block b's q - 8 or q of this lane, low then high nibbles
  static __device__ __forceinline__ int64_t quants(uint32_t q) {
    uint32_t lo = q & 0x0F0F0F0Fu, hi = (q >> 4) & 0x0F0F0F0Fu;
    if constexpr (FMT == kW_Q4_0) {   // q - 8 as a signed byte
      lo = ((lo | 0x80808080u) - 0x08080808u) ^ 0x80808080u;
      hi = ((hi | 0x80808080u) - 0x08080808u) ^ 0x80808080u;
    }
    return (int64_t)(((unsigned long long)hi << 32) | lo);
  }
  __device__ __forceinline__ void take(int t, int, int s, const uint8_t *cur) {
    const uint32_t *rowb = reinterpret_cast<const uint32_t *>(cur + j * 16 * S::kChunks);
    const uint8_t *rec = ab + HT * 4096;
    float sum[HT];          // the slab's
    uint32_t hd[8], q[8];   // d (and m); the lane group's dword
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if constexpr (FMT == kW_Q4_0) {   // block b from byte 18 b: d, 16 bytes
        const uint32_t w = rowb[18 * b / 4];
        hd[b] = b & 1 ? w >> 16 : w;
        const uint32_t *p = rowb + 18 * b / 4 + G;
        q[b] = b & 1 ? p[1] : __builtin_amdgcn_alignbyte(p[1], p[0], 2);
      } else {
        hd[b] = rowb[5 * b];
        q[b] = rowb[5 * b + 1 + G];
      }
    }
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const int64_t B = quants(q[b]);
      const float d = q6m::h2f(hd[b]);
#pragma unroll
      for (int h = 0; h < HT; ++h) {
        const int64_t A = *reinterpret_cast<const int64_t *>(ab + h * 4096 + b * 512 + lane * 8);
        const v4i D = __builtin_amdgcn_mfma_i32_16x16x32_i8(A, B, v4i{0, 0, 0, 0}, 0, 0, 0);
        const float val = bg::limb_sum(D);
        if constexpr (FMT == kW_Q4_1) {   // (d q and m cancel within the block, as in a row alone)
          const float sx = *reinterpret_cast<const float *>(rec + (4 * h + G) * S::kRec + 16 + 4 * b);
          const float w = fmaf(val, d, q6m::h2f(hd[b] >> 16) * sx);
          sum[h] = b == 0 ? w : sum[h] + w;
        } else {
          sum[h] = b == 0 ? val * d : fmaf(val, d, sum[h]);
        }
      }
    }
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      const float xs = *reinterpret_cast<const float *>(rec + (4 * h + G) * S::kRec);
      acc[t][h] = fmaf(sum[h], xs, acc[t][h]);   // times a power of two
    }
    if (__builtin_expect(more != 0u, 0)) {
      const uint8_t *a2 = second + (int64_t)s * kA + lane * 8;
#pragma unroll
      for (int h = 0; h < HT; ++h) {
        if (!(more >> (4 * h) & 15u)) continue;
        float sum2 = 0.f;
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const int64_t A = *reinterpret_cast<const int64_t *>(a2 + h * 4096 + b * 512);
          const v4i D = __builtin_amdgcn_mfma_i32_16x16x32_i8(A, quants(q[b]), v4i{0, 0, 0, 0}, 0, 0, 0);
          sum2 = fmaf(bg::limb_sum(D), q6m::h2f(hd[b]), sum2);
        }
        acc[t][h] = fmaf(sum2, *reinterpret_cast<const float *>(rec + (4 * h + G) * S::kRec + 4), acc[t][h]);
      }
    }
  }
  // A row's result in plain binary32, unit by unit as the one-row kernel
  // forms them: what a row with a non-finite input is (the limbs, which
  // cannot hold one, leave NaN; d q x + m x may be an infinity).
  __device__ __forceinline__ float plain(int m, int row) const {
    const float *x = g.x + (int64_t)m * g.ldx;
    const uint32_t *w = static_cast<const uint32_t *>(g.w) + (int64_t)row * (g.row_bytes / 4u);
    float r = 0.f;
#pragma nounroll
    for (int b = 0; b < g.K / 32 && r == r; ++b, x += 32, w += 5) {
      float lo = 0.f, hi = 0.f, sum = 0.f;
#pragma nounroll
      for (int v = 0; v < 4; ++v) {
        const uint32_t q4 = w[1 + v];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float xl = x[4 * v + i], xh = x[16 + 4 * v + i];
          lo = fmaf(xl, (float)((q4 >> (8 * i)) & 15u), lo);
          hi = fmaf(xh, (float)((q4 >> (8 * i + 4)) & 15u), hi);
          sum += xl + xh;
        }
      }
      r += fmaf(q6m::h2f(w[0]), lo + hi, q6m::h2f(w[0] >> 16) * sum);
    }
    return r;
  }
  __device__ __forceinline__ void put(int t, int tile) {
    const int row = tile * 16 + j, m0 = slice * 4 * HT + G;
    uint32_t nan = 0;
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      const int m = m0 + 4 * h;
      if (row < g.N && m < g.M) {
        g.y[(int64_t)m * g.ldy + row] = acc[t][h];
        if (FMT == kW_Q4_1 && acc[t][h] != acc[t][h]) nan |= 1u << h;
      }
    }
    if constexpr (FMT == kW_Q4_1)
      while (__builtin_expect(nan != 0u, 0)) {
        const int m = m0 + 4 * (__ffs(nan) - 1);
        g.y[(int64_t)m * g.ldy + row] = plain(m, row);
        nan &= nan - 1u;
      }
  }
};

template <int FMT, int HT, int RT, int NW, int NB>
__global__ __launch_bounds__(64 * NW, NW / 4) void gemv_batch_q4_kernel(GemvArgs g, const uint8_t *tab,
                                                                        int slices, int groups) {
  extern __shared__ uint4 blds[];
  using Body = Q4Batch<FMT, HT, RT>;
  const int slice = batch_slice(slices), NS = g.K / 256;
  tab += (int64_t)slice * NS * Body::kA;
  Body body(g, tab, slice);
  batch_stream<Body, RT, NW, NB>(body, tab, NS, g.N, slices, groups, reinterpret_cast<uint8_t *>(blds));
}

// ---- F32: binary32 on v_mfma_f32_16x16x4_f32
//
// A tile is 16 activation rows x 4 positions, B 4 positions x 16 weight rows,
// every product a binary32 fused multiply-add as on the vector units.  A slab
// is 64 positions, lane group kk of a wave takes positions 16 kk .. 16 kk + 15,
// its i-th weight the B operand of MFMA i; x lies in LDS in the same order.
// Two chains of eight MFMAs per slab; the slabs are added up with a
// compensated sum (plain, the error against binary64 was 1.3e-7 at K 1024
// against the vector units' 1.2e-7).
namespace bg {
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int kFSP = 64;                                   // positions of a slab
constexpr int f32_a_bytes(int ht) { return ht * 16 * 4 * kFSP; }
}  // namespace bg

// x of row i of a slice's tile: 16-byte piece c of its slab at piece c ^ i
// (the 16 rows' reads of one piece spread over the banks), 16 lanes a slab.
// tab: [slice][K / 64][f32_a_bytes(ht)]
__global__ __launch_bounds__(64) void xpack_kernel(const float *x, int64_t ldx, int NS, int ht, uint8_t *tab) {
  const int s = 4 * (int)blockIdx.x + ((int)threadIdx.x >> 4), m = (int)blockIdx.y, c = (int)threadIdx.x & 15;
  if (s >= NS) return;
  const float *xp = x + (int64_t)m * ldx + bg::kFSP * s + 4 * c;
  const int hid = m % (16 * ht), i = hid & 15;
  uint8_t *d = tab + ((int64_t)(m / (16 * ht)) * NS + s) * bg::f32_a_bytes(ht) + hid * bg::kFSP * 4;
  *reinterpret_cast<float4 *>(d + (c ^ i) * 16) = make_float4(xp[0], xp[1], xp[2], xp[3]);
}

template <int HT, int RT>
struct F32Batch {
  using v4i = bg::v4i;
  using v4f = bg::v4f;
  static constexpr int kLoads = 4, kSlab = 4096;
  static constexpr int kA = bg::f32_a_bytes(HT);
  const GemvArgs &g;
  const int slice, lane, j, kk;
  const v4i rw;
  uint32_t vo[kLoads];
  const uint8_t *ab;
  v4f acc[RT][HT], low[RT][HT];   // sums, and what their roundings lost

  __device__ __forceinline__ F32Batch(const GemvArgs &args, int sl)
      : g(args), slice(sl), lane(threadIdx.x & 63), j(lane & 15), kk(lane >> 4),
        rw(bg::rsrc(args.w, (args.w_bytes + 15u) & ~15u)) {}
  __device__ __forceinline__ void at(int s) {
#pragma unroll
    for (int c = 0; c < kLoads; ++c) {   // four rows a load, their pieces as x's
      const int rj = 4 * c + (lane >> 4);
      vo[c] = (uint32_t)rj * g.row_bytes + 256u * (uint32_t)s + 16u * (uint32_t)((lane & 15) ^ rj);
    }
  }
  __device__ __forceinline__ void go(int tile, uint32_t dst) {
    const uint32_t base = (uint32_t)tile * 16u * g.row_bytes;
#pragma unroll
    for (int c = 0; c < kLoads; ++c) bg::to_lds(rw, base + vo[c], dst + c * 1024);
  }
  __device__ __forceinline__ void zero(int t) {
#pragma unroll
    for (int h = 0; h < HT; ++h) acc[t][h] = low[t][h] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ void step(const uint8_t *a) { ab = a; }
  __device__ __forceinline__ void take(int t, int, int, const uint8_t *cur) {
    v4f D[HT][2];
#pragma unroll
    for (int h = 0; h < HT; ++h) D[h][0] = D[h][1] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int c = (4 * kk + v) ^ j;
      const float4 w = *reinterpret_cast<const float4 *>(cur + j * 256 + c * 16);
#pragma unroll
      for (int h = 0; h < HT; ++h) {
        const float4 xv = *reinterpret_cast<const float4 *>(ab + h * 4096 + j * 256 + c * 16);
        D[h][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv.x, w.x, D[h][0], 0, 0, 0);
        D[h][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv.y, w.y, D[h][1], 0, 0, 0);
        D[h][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv.z, w.z, D[h][0], 0, 0, 0);
        D[h][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv.w, w.w, D[h][1], 0, 0, 0);
      }
    }
#pragma unroll
    for (int h = 0; h < HT; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float a = acc[t][h][r], x = (D[h][0][r] + D[h][1][r]) - low[t][h][r];
        const float n = a + x;
        // (where the sum is infinite, Inf - Inf: any finite value does, and one
        // that cannot overflow the next x)
        low[t][h][r] = __builtin_amdgcn_fmed3f((n - a) - x, -0x1p100f, 0x1p100f);
        acc[t][h][r] = n;
      }
  }
  __device__ __forceinline__ void put(int t, int tile) {
    const int row = tile * 16 + j;
#pragma unroll
    for (int h = 0; h < HT; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = slice * 16 * HT + 16 * h + 4 * kk + r;
        if (row < g.N && m < g.M) g.y[(int64_t)m * g.ldy + row] = acc[t][h][r];
      }
  }
};

template <int HT, int RT, int NW, int NB>
__global__ __launch_bounds__(64 * NW, NW / 4) void gemv_batch_f32_kernel(GemvArgs g, const uint8_t *tab,
                                                                         int slices, int groups) {
  extern __shared__ uint4 blds[];
  using Body = F32Batch<HT, RT>;
  const int slice = batch_slice(slices), NS = g.K / bg::kFSP;
  Body body(g, slice);
  batch_stream<Body, RT, NW, NB>(body, tab + (int64_t)slice * NS * Body::kA, NS, g.N, slices, groups,
                                 reinterpret_cast<uint8_t *>(blds));
}

namespace {

// slabs per wave of a 16-wave workgroup (half as many bytes in flight a slab
// for Q4_K)
template <int FMT> constexpr int kRing16 = FMT == kW_Q6_K ? 2 : 3;

// The tables' kernel, then the GEMV's: LDS of two steps' A operands and the
// rings, one workgroup a CU, slices of `rows` activation rows.
template <class Pre, class Main>
hipError_t launch_two(const GemvArgs &g, Pre pre, dim3 pre_grid, int pre_threads, Main kernel, int NW,
                      size_t lds, int rows, int pre_arg, hipStream_t stream, hipEvent_t start,
                      hipEvent_t stop, int NS) {
  const int res = resident_blocks(reinterpret_cast<const void *>(kernel), (uint32_t)lds, 64 * NW);
  const int slices = (g.M + rows - 1) / rows, ntiles = (g.N + 15) / 16;
  // groups of tiles: whole multiples of eight (one per XCD)
  int groups = res / slices / 8 * 8;
  const int most = ((ntiles + NW - 1) / NW + 7) / 8 * 8;
  groups = groups < 8 ? 8 : groups;
  groups = groups < most ? groups : most;
  const dim3 grid((unsigned)(groups * slices)), block(64 * NW);
  uint8_t *tab = static_cast<uint8_t *>(g.tab);
  if (start)
    hipExtLaunchKernelGGL(pre, pre_grid, dim3(pre_threads), 0, stream, start, nullptr, 0u, g.x, g.ldx, NS,
                          pre_arg, tab);
  else
    hipLaunchKernelGGL(pre, pre_grid, dim3(pre_threads), 0, stream, g.x, g.ldx, NS, pre_arg, tab);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (stop)
    hipExtLaunchKernelGGL(kernel, grid, block, lds, stream, nullptr, stop, 0u, g, tab, slices, groups);
  else
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, g, tab, slices, groups);
  return hipGetLastError();
}

template <int FMT, int HT, int RT, int NW, int NB, bool HOLD>
constexpr size_t kq_lds() {
  constexpr size_t b = 2 * (size_t)bg::a_bytes<FMT>(HT) + (size_t)NW * NB * bg::slab_bytes<FMT>();
  static_assert(b <= 160 * 1024, "LDS");
  return b;
}
template <int FMT, int HT, int RT, int NW, int NB, bool HOLD>
hipError_t launch_kq(const GemvArgs &g, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  return launch_two(g, limbs_kernel<FMT>, dim3((unsigned)(g.K / 256), (unsigned)g.M), 64,
                    gemv_batch_kq_kernel<FMT, HT, RT, NW, NB, HOLD>, NW, kq_lds<FMT, HT, RT, NW, NB, HOLD>(),
                    4 * HT, HT, stream, start, stop, g.K / 256);
}

// By the number of activation rows: A tiles HT (four rows each) per slice,
// tiles RT per pass, waves NW per workgroup (one a CU), slabs NB per wave's
// ring, and whether a wave holds a super-block's A operands in registers for
// its RT tiles or reads them from LDS for each (at 32 rows they are 128
// registers: holding them leaves 8 waves a CU; 16 rows and 16 waves: read).
// Measured at 151936 x 2048 Q6_K, us per call: 16 rows 87 (held, 8 waves 90),
// 64 rows 199 (held, 8 waves 210; RT 3 202), 2 rows 70 (RT 1 74, 8 waves 75).
template <int FMT>
hipError_t launch_kq_m(const GemvArgs &g, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (g.M <= 4) return launch_kq<FMT, 1, 3, 16, kRing16<FMT>, true>(g, stream, start, stop);
  if (g.M <= 8) return launch_kq<FMT, 2, 3, 16, kRing16<FMT>, true>(g, stream, start, stop);
  if (g.M <= 16) return launch_kq<FMT, 4, 3, 16, kRing16<FMT>, false>(g, stream, start, stop);
  return launch_kq<FMT, 8, 4, 12, 2, false>(g, stream, start, stop);
}

template <int FMT, int HT, int RT, int NW, int NB, bool HOLD>
hipError_t prep_kq() {
  return hipFuncSetAttribute(reinterpret_cast<const void *>(gemv_batch_kq_kernel<FMT, HT, RT, NW, NB, HOLD>),
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)kq_lds<FMT, HT, RT, NW, NB, HOLD>());
}

template <int FMT>
hipError_t prep_kq_m() {
  hipError_t e = prep_kq<FMT, 1, 3, 16, kRing16<FMT>, true>();
  if (e == hipSuccess) e = prep_kq<FMT, 2, 3, 16, kRing16<FMT>, true>();
  if (e == hipSuccess) e = prep_kq<FMT, 4, 3, 16, kRing16<FMT>, false>();
  if (e == hipSuccess) e = prep_kq<FMT, 8, 4, 12, 2, false>();
  return e;
}

// The other formats' instances: launched (go) or their LDS limit raised.
template <int FMT, int HT, int RT, int NW, int NB>
hipError_t tern_one(const GemvArgs *g, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  using Body = TernBatch<FMT, HT, RT>;
  constexpr size_t lds = 2 * (size_t)Body::kA + (size_t)NW * NB * Body::kSlab;
  static_assert(lds <= 160 * 1024, "LDS");
  const auto k = gemv_batch_tern_kernel<FMT, HT, RT, NW, NB>;
  if (!g)
    return hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds);
  return launch_two(*g, tern_limbs_kernel<FMT>, dim3((unsigned)(g->K / 128), (unsigned)g->M), 64, k, NW, lds,
                    4 * HT, HT, stream, start, stop, g->K / 512);
}
template <int FMT>
hipError_t tern_m(const GemvArgs *g, int M, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (M <= 4) return tern_one<FMT, 1, 3, 16, 4>(g, stream, start, stop);
  if (M <= 8) return tern_one<FMT, 2, 3, 16, 3>(g, stream, start, stop);
  // (16 waves a CU, 128 registers each, spill some of them)
  return tern_one<FMT, 4, 3, 12, 3>(g, stream, start, stop);
}
template <int FMT, int HT, int RT, int NW, int NB>
hipError_t q4_one(const GemvArgs *g, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  using Body = Q4Batch<FMT, HT, RT>;
  constexpr size_t lds = 2 * (size_t)Body::kA + (size_t)NW * NB * Body::kSlab;
  static_assert(lds <= 160 * 1024, "LDS");
  const auto k = gemv_batch_q4_kernel<FMT, HT, RT, NW, NB>;
  if (!g)
    return hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds);
  return launch_two(*g, limbs_kernel<FMT>, dim3((unsigned)(g->K / 256), (unsigned)g->M), 64, k, NW, lds,
                    4 * HT, HT, stream, start, stop, g->K / 256);
}
template <int FMT>
hipError_t q4_m(const GemvArgs *g, int M, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (M <= 4) return q4_one<FMT, 1, 3, 16, 3>(g, stream, start, stop);
  if (M <= 8) return q4_one<FMT, 2, 3, 16, 3>(g, stream, start, stop);
  return q4_one<FMT, 4, 3, 16, 3>(g, stream, start, stop);
}
template <int HT, int RT, int NW, int NB>
hipError_t f32_one(const GemvArgs *g, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  using Body = F32Batch<HT, RT>;
  constexpr size_t lds = 2 * (size_t)Body::kA + (size_t)NW * NB * Body::kSlab;
  static_assert(lds <= 160 * 1024, "LDS");
  const auto k = gemv_batch_f32_kernel<HT, RT, NW, NB>;
  if (!g)
    return hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds);
  return launch_two(*g, xpack_kernel, dim3((unsigned)((g->K / bg::kFSP + 3) / 4), (unsigned)g->M), 64, k, NW, lds,
                    16 * HT, HT, stream, start, stop, g->K / bg::kFSP);
}
hipError_t f32_m(const GemvArgs *g, int M, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (M <= 16) return f32_one<1, 3, 16, 2>(g, stream, start, stop);
  if (M <= 32) return f32_one<2, 3, 16, 2>(g, stream, start, stop);
  return f32_one<4, 3, 8, 3>(g, stream, start, stop);
}

}  // namespace

hipError_t prepare_gemv_batch() {
  hipError_t e = prep_kq_m<kW_Q6_K>();
  if (e == hipSuccess) e = prep_kq_m<kW_Q4_K>();
  for (const int M : {4, 8, 16, 32, 64}) {   // every instance
    if (e == hipSuccess) e = tern_m<kW_Q1_0>(nullptr, M, nullptr, nullptr, nullptr);
    if (e == hipSuccess) e = tern_m<kW_PQ2_0>(nullptr, M, nullptr, nullptr, nullptr);
    if (e == hipSuccess) e = tern_m<kW_PTQ1_0>(nullptr, M, nullptr, nullptr, nullptr);
    if (e == hipSuccess) e = q4_m<kW_Q4_0>(nullptr, M, nullptr, nullptr, nullptr);
    if (e == hipSuccess) e = q4_m<kW_Q4_1>(nullptr, M, nullptr, nullptr, nullptr);
    if (e == hipSuccess) e = f32_m(nullptr, M, nullptr, nullptr, nullptr);
  }
  return e;
}

hipError_t launch_gemv_batch(GemvArgs g, hipStream_t stream, hipEvent_t *ev, hipEvent_t done) {
  // the tables hold kBatchRows activation rows: more go in parts, one after
  // another on the stream
  const int M = g.M;
  for (int m = 0; m < M; m += kBatchRows) {
    GemvArgs p = g;
    p.x = g.x + (int64_t)m * g.ldx;
    p.y = g.y + (int64_t)m * g.ldy;
    p.M = M - m < kBatchRows ? M - m : kBatchRows;
    const bool last = m + kBatchRows >= M;
    const hipEvent_t start = ev && m == 0 ? ev[0] : nullptr;
    const hipEvent_t stop = !last ? nullptr : ev ? ev[1] : done;
    hipError_t e = hipErrorInvalidValue;
    switch (g.type) {
      case kW_Q6_K: e = launch_kq_m<kW_Q6_K>(p, stream, start, stop); break;
      case kW_Q4_K: e = launch_kq_m<kW_Q4_K>(p, stream, start, stop); break;
      case kW_Q1_0: e = tern_m<kW_Q1_0>(&p, p.M, stream, start, stop); break;
      case kW_PQ2_0: e = tern_m<kW_PQ2_0>(&p, p.M, stream, start, stop); break;
      case kW_PTQ1_0: e = tern_m<kW_PTQ1_0>(&p, p.M, stream, start, stop); break;
      case kW_Q4_0: e = q4_m<kW_Q4_0>(&p, p.M, stream, start, stop); break;
      case kW_Q4_1: e = q4_m<kW_Q4_1>(&p, p.M, stream, start, stop); break;
      case kW_F32: e = f32_m(&p, p.M, stream, start, stop); break;
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace hs
