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
// int8 limbs per super-block, as in the one-row kernels (there per 16
// positions): with 2^E above the block's largest |x|, a_t = rint(r_{t-1} *
// 2^(6 + 7t - E)), r_t the exact remainder, |a_t| <= 64.  An A tile (16 x 64)
// holds four limbs of four activation rows, A row 4 h + t limb t of row h; B
// (64 x 16) one of the two bytes of 16 weight rows.  Eight MFMAs per
// super-block and A tile (four steps of 64 positions, hi and lo) leave in
// lane (j, h) of the result the four exact limb sums of (weight row j,
// activation row h), in magnitude at most 2^26: one product per lane, so the
// running binary32 sum of a tile takes one register per A tile.
// (One row on the same instruction fills a quarter of an A tile with zeros
// around its four limbs; four rows fill it.)
//
// The limbs are made by a kernel of their own (limbs_kernel) into the
// context's workspace, laid out as the A operands are read; a workgroup
// stages one super-block's A operands at a time in LDS (two buffers, one
// barrier per super-block), each of its waves streams the weights of its own
// tiles through a ring in LDS, as the one-row kernels do.
//
// What bounds it: up to 8 rows the weights' reads (151936 x 2048 Q6_K, 2
// rows: 70 us a call, of which 3 us are limbs_kernel; one row at a time 96
// us; 7 rows 75 and 284 us; Q4_K at K 4096, 7 rows 112 and 453 us), beyond
// that the instructions of a tile: about 250 vector instructions to take it
// apart, 13 per A tile to add its results up, 8 MFMAs per A tile (counters
// at 64 rows: vector units busy 45 % of the cycles, matrix cores 31 %, hardly
// overlapping).  16 rows 87 us (620 one at a time), 64 rows 199 us (2417).
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
  static constexpr int kRec = 16;                        // bytes of an activation row's record
};
template <> struct Slab<kW_Q4_K> {
  static constexpr int kBytes = 144;
  static constexpr int kChunks = q4m::kRowChunks;
  static constexpr int kRec = 48;                        // 2^(E - 6), then eight sums of x
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

// The A operands of activation rows 0..M-1: one wave per (super-block, row),
// four positions a lane.  tab: [ceil(M / 4 ht)][K / 256][a_bytes(ht)].  A
// block with a non-finite element gets a NaN scale, which makes every result
// of its row NaN.
template <int FMT>
__global__ __launch_bounds__(64) void limbs_kernel(const float *x, int64_t ldx, int NS, int ht,
                                                   uint8_t *tab) {
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
  float sum = (v[0] + v[1]) + (v[2] + v[3]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
#pragma unroll
  for (int o = 4; o > 0; o >>= 1) sum += __shfl_xor(sum, o);   // of the 32 positions of 8 lanes
  fin = __all(fin);
  int E = 0;
  (void)frexpf(fin ? mx : 1.f, &E);   // mx < 2^E
  uint32_t limb[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    float r = fin ? v[b] : 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float a = rintf(ldexpf(r, 6 + 7 * t - E));
      r -= ldexpf(a, E - 6 - 7 * t);   // exact: a 2^(E-6-7t) is within half a step of r
      limb[t] |= ((uint32_t)(int)a & 0xFFu) << (8 * b);
    }
  }
  // where the weights of position p sit in B: step and lane group (Q6_K:
  // p = 128 n + 32 step + 16 h + b in group 2 n + h, the quarters of a half
  // share their bytes; Q4_K: in order)
  const int p = 4 * lane;
  const int step = FMT == kW_Q6_K ? (p >> 5) & 3 : p >> 6;
  const int G = FMT == kW_Q6_K ? 2 * (p >> 7) + ((p >> 4) & 1) : (p >> 4) & 3;
  const int hid = m % (4 * ht);
  uint8_t *a = tab + ((int64_t)(m / (4 * ht)) * NS + s) * bg::a_bytes<FMT>(ht);
  uint8_t *d = a + (hid >> 2) * 4096 + step * 1024 + (16 * G + 4 * (hid & 3)) * 16 + (p & 15);
#pragma unroll
  for (int t = 0; t < 4; ++t) *reinterpret_cast<uint32_t *>(d + 16 * t) = limb[t];
  float *rec = reinterpret_cast<float *>(a + ht * 4096 + hid * bg::Slab<FMT>::kRec);
  if (lane == 0) rec[0] = fin ? ldexpf(1.f, E - 6) : __builtin_nanf("");
  if (FMT == kW_Q4_K && (lane & 7) == 0) rec[4 + (lane >> 3)] = sum;
}

// The wave's tiles are gw, gw + nwx, ... (at any time the waves read
// neighbouring tiles, and the tiles of a last, partial round spread over all
// workgroups), taken in passes of at most RT; a pass goes through the
// row's super-blocks in order, each over the pass's tiles.  Items (pass,
// super-block, tile) stream through the wave's ring of NB slabs.
template <int FMT, int HT, int RT, int NW, int NB, bool HOLD>
__global__ __launch_bounds__(64 * NW, NW / 4) void gemv_batch_kq_kernel(GemvArgs g, const uint8_t *tab,
                                                                        int slices, int groups) {
  using namespace bg;
  using S = Slab<FMT>;
  constexpr int L = slab_loads<FMT>(), SB = slab_bytes<FMT>();
  constexpr int AB = a_bytes<FMT>(HT);
  // A loads of a wave (1 KiB each; past the last piece a wave reads that one
  // again, so that every wave has the same count in flight)
  constexpr int AP = (AB + 1023) / 1024, AL = (AP + NW - 1) / NW;
  extern __shared__ uint4 blds[];
  uint8_t *abuf = reinterpret_cast<uint8_t *>(blds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint8_t *ring = abuf + 2 * AB + wave * NB * SB;
  const uint32_t abuf_a = lds_addr(abuf), ring_a = lds_addr(ring);
  // Workgroups b, b + 8, ... of one XCD: the slices (16 activation rows) of
  // one group of tiles are neighbours there and share the weights in its L2
  const int b = (int)blockIdx.x, r = b >> 3;
  const int slice = r % slices, xg = (r / slices) * 8 + (b & 7);
  const int NS = g.K / 256;
  const int ntiles = (g.N + 15) >> 4;
  const int nwx = groups * NW, gw = wave * groups + xg;
  const int cnt = gw < ntiles ? (ntiles - 1 - gw) / nwx + 1 : 0;
  const int maxcnt = (ntiles - 1) / nwx + 1;
  const int np = (maxcnt + RT - 1) / RT;
  auto plo = [&](int p) {   // first tile of pass p
    const int i = p * maxcnt / np;
    return i < cnt ? i : cnt;
  };
  const int total = cnt * NS;
  const int j = lane & 15, G = lane >> 4;
  const v4i rw = rsrc(g.w, (g.w_bytes + 15u) & ~15u);
  const uint8_t *atab = tab + (int64_t)slice * NS * AB;
  const v4i ra = rsrc(atab, (uint32_t)(NS * AB));

  // next slab to issue: its tile, super-block and ring slot
  int iz = 0, is = 0, ip = 0, ilo = 0, ihi = plo(1), ii = 0, islot = 0;
  // (a lane's byte offset in a tile, per load, for super-block `is`; rows at
  // and past N lie past the resource, or wrap to its start: unused)
  uint32_t vo[L];
  auto lane_offsets = [&]() {
#pragma unroll
    for (int c = 0; c < L; ++c) {
      const int q = c * 64 + lane, rj = q / S::kChunks, cc = q % S::kChunks;
      vo[c] = (((uint32_t)rj * g.row_bytes + (uint32_t)S::kBytes * (uint32_t)is) & ~15u) + 16u * (uint32_t)cc;
    }
  };
  lane_offsets();
  auto issue = [&]() {
    const uint32_t base = (uint32_t)(gw + ii * nwx) * 16u * g.row_bytes;   // a multiple of 16
    const uint32_t dst = ring_a + islot * SB;
#pragma unroll
    for (int c = 0; c < L; ++c)
      if (c + 1 < L || 16 * S::kChunks % 64 == 0 || lane < 16 * S::kChunks % 64)
        to_lds(rw, base + vo[c], dst + c * 1024);
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
      lane_offsets();
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
  float acc[RT][HT];
  for (int p = 0; p < np; ++p) {
    const int lo = plo(p), n = plo(p + 1) - lo;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int h = 0; h < HT; ++h) acc[t][h] = 0.f;
    for (int s = 0; s < NS; ++s) {
      const int q = p * NS + s;
      const uint8_t *ab = abuf + (q & 1) * AB;
      // this wave's share of A has arrived (the slabs issued after it may
      // still be in flight), its reads of the other buffer are done
      wait_slabs<L, 0>(iz - iza < iz - z ? iz - iza : iz - z);
      wait_lds();
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (q + 1 < np * NS) {
        issue_a(s + 1 == NS ? 0 : s + 1, abuf_a + ((q + 1) & 1) * AB);
        iza = iz;
      }
      v4i A[HOLD ? HT : 1][4];
      float xs[HT];
      const uint8_t *rec = ab + HT * 4096;
      auto a_op = [&](int h, int k) {
        return *reinterpret_cast<const v4i *>(ab + h * 4096 + k * 1024 + lane * 16);
      };
#pragma unroll
      for (int h = 0; h < HT; ++h) {
        if constexpr (HOLD)
#pragma unroll
          for (int k = 0; k < 4; ++k) A[h][k] = a_op(h, k);
        xs[h] = *reinterpret_cast<const float *>(rec + (4 * h + G) * S::kRec);
      }
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        if (t < n) {
          wait_lds();   // the previous slab's reads are done: its slot is free
          if (iz < total) issue();
          // slab z has arrived: the later slabs may be in flight, and the A
          // loads where they were issued after it
          if (z < iza && q + 1 < np * NS) wait_slabs<L, AL>(iz - z - 1);
          else wait_slabs<L, 0>(iz - z - 1);
          const uint8_t *cur = ring + slot * SB;
          slot = slot + 1 == NB ? 0 : slot + 1;
          ++z;
          const int row = (gw + (lo + t) * nwx) * 16 + j;
          const uint32_t o =
              FMT == kW_Q6_K ? ((uint32_t)row * g.row_bytes + 210u * (uint32_t)s) & 15u : 0u;
          BOps B;
          decode<FMT>(cur + j * 16 * S::kChunks, o, G, B);
          // HP A tiles at a time: 2 HP independent accumulator chains
          // (one for Q4_K at HT 8, whose minima take the registers)
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
              float &sum = acc[t][h0 + h];
              if constexpr (FMT == kW_Q4_K) {   // the minima: - dmin sum_s m_s (sub-block s's sum of x)
                const float4 *xr = reinterpret_cast<const float4 *>(rec + (4 * (h0 + h) + G) * S::kRec + 16);
                const float4 u = xr[0], v = xr[1];
                float sm = B.mf[0] * u.x;
                sm = fmaf(B.mf[1], u.y, sm);
                sm = fmaf(B.mf[2], u.z, sm);
                sm = fmaf(B.mf[3], u.w, sm);
                sm = fmaf(B.mf[4], v.x, sm);
                sm = fmaf(B.mf[5], v.y, sm);
                sm = fmaf(B.mf[6], v.z, sm);
                sm = fmaf(B.mf[7], v.w, sm);
                sum = fmaf(-B.dmin, sm, sum);
              }
              const v4i dt = hi[h] * 256 + lw[h];
              float val = fmaf((float)dt[3], 0x1p-7f, (float)dt[2]);
              val = fmaf(val, 0x1p-7f, (float)dt[1]);
              val = fmaf(val, 0x1p-7f, (float)dt[0]);
              sum = fmaf(B.d * xs[h0 + h], val, sum);   // d times a power of two
            }
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      if (t < n) {
        const int row = (gw + (lo + t) * nwx) * 16 + j;
#pragma unroll
        for (int h = 0; h < HT; ++h) {
          const int m = slice * 4 * HT + 4 * h + G;
          if (row < g.N && m < g.M) g.y[(int64_t)m * g.ldy + row] = acc[t][h];
        }
      }
    }
  }
}

namespace {

// slabs per wave of a 16-wave workgroup (half as many bytes in flight a slab
// for Q4_K)
template <int FMT> constexpr int kRing16 = FMT == kW_Q6_K ? 2 : 3;

template <int FMT, int HT, int RT, int NW, int NB, bool HOLD>
hipError_t launch_kq(const GemvArgs &g, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  const size_t lds = 2 * (size_t)bg::a_bytes<FMT>(HT) + (size_t)NW * NB * bg::slab_bytes<FMT>();
  static_assert(2 * bg::a_bytes<FMT>(HT) + NW * NB * bg::slab_bytes<FMT>() <= 160 * 1024, "LDS");
  static_assert(NB <= 4, "wait_slabs counts three later slabs");
  const auto kernel = gemv_batch_kq_kernel<FMT, HT, RT, NW, NB, HOLD>;
  const int res = resident_blocks(reinterpret_cast<const void *>(kernel), (uint32_t)lds, 64 * NW);
  const int slices = (g.M + 4 * HT - 1) / (4 * HT), ntiles = (g.N + 15) / 16;
  // groups of tiles: whole multiples of eight (one per XCD)
  int groups = res / slices / 8 * 8;
  const int most = ((ntiles + NW - 1) / NW + 7) / 8 * 8;
  groups = groups < 8 ? 8 : groups;
  groups = groups < most ? groups : most;
  const dim3 grid((unsigned)(groups * slices)), block(64 * NW);
  uint8_t *tab = static_cast<uint8_t *>(g.tab);
  const dim3 lgrid((unsigned)(g.K / 256), (unsigned)g.M);
  if (start)
    hipExtLaunchKernelGGL(limbs_kernel<FMT>, lgrid, dim3(64), 0, stream, start, nullptr, 0u, g.x, g.ldx,
                          g.K / 256, HT, tab);
  else
    hipLaunchKernelGGL(limbs_kernel<FMT>, lgrid, dim3(64), 0, stream, g.x, g.ldx, g.K / 256, HT, tab);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (stop)
    hipExtLaunchKernelGGL(kernel, grid, block, lds, stream, nullptr, stop, 0u, g, tab, slices, groups);
  else
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, g, tab, slices, groups);
  return hipGetLastError();
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
                             2 * bg::a_bytes<FMT>(HT) + NW * NB * bg::slab_bytes<FMT>());
}

template <int FMT>
hipError_t prep_kq_m() {
  hipError_t e = prep_kq<FMT, 1, 3, 16, kRing16<FMT>, true>();
  if (e == hipSuccess) e = prep_kq<FMT, 2, 3, 16, kRing16<FMT>, true>();
  if (e == hipSuccess) e = prep_kq<FMT, 4, 3, 16, kRing16<FMT>, false>();
  if (e == hipSuccess) e = prep_kq<FMT, 8, 4, 12, 2, false>();
  return e;
}

}  // namespace

hipError_t prepare_gemv_batch() {
  hipError_t e = prep_kq_m<kW_Q6_K>();
  if (e == hipSuccess) e = prep_kq_m<kW_Q4_K>();
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
    if (g.type == kW_Q6_K) e = launch_kq_m<kW_Q6_K>(p, stream, start, stop);
    else if (g.type == kW_Q4_K) e = launch_kq_m<kW_Q4_K>(p, stream, start, stop);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace hs
