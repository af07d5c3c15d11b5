// gemm_rows16.hip -- a7 / a9 for short prompts (17 to a few hundred tokens at a few
// thousand weight rows), straight from plain rows of any 2-byte alignment and any
// block count: one 16 x 16 output tile a wave.
//
// What bounds it: an output's n/32 fmas run in order, so a wave walks all of K, and
// with one wave a SIMD it issues one VALU instruction per ~5 cycles whatever it is
// (2.6 with two waves).  32 x 32 tiles take half the VALU per output but leave
// half the SIMDs without a wave at 4096 rows x 128 tokens; 16 x 16 tiles put two
// on each.  A work-group of 4 or 8 waves (32 or 64 weight rows x 32 tokens)
// shares its rows through LDS:
//   - K in chunks of 16 blocks, the raw row spans loaded in 16-byte pieces (whole
//     rows side by side), a chunk ahead in registers, into one of two LDS
//     buffers: one barrier a chunk, nothing repacked;
//   - the operands come from the raw spans as aligned dwords, each lane group
//     the dwords of a block pair that need one funnel shift (two for tokens against
//     Q4_0) to make its eight quants, in an order both operands share;
//   - v_mfma_i32_16x16x32_i8 gives the block sums, v_mfma_f32_16x16x16_f16 the
//     exact scale products (Q8_0) or the weights' scales spread over the tile
//     (Q4_0); the pair after next is read and the next pair's MFMAs issued while
//     a pair is folded.
// Measured (us, K 4096, Q4_0 / Q8_0; before it gemm_rows_few, gemm_batch past 24
// tokens, and for odd block counts gemm_batch): 4096 x 64 17.2 / 18.5 -> 13.3 /
// 12.4, 4096 x 128 31.0 / 26.7 -> 18.4 / 16.6, 4096 x 192 31.2 / 26.8 -> 28.1 /
// 26.0; 3001 x 333 x 2912 53 / 58 -> 36 / 43.  At 4096 x 128 the LDS is busy two
// thirds of the time (Q4_0) and a wave waits a third of it, for barriers mostly.
#include "tcrv_hip_internal.h"
#include "mfma_fold.h"
#include "tile_order.h"

namespace tcrv {

typedef uint32_t u32x4a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kR16Chunk = 16;  // blocks (8 measured 1-3 us slower at 4096 x 128: twice the barriers)

// A lane group's dwords of a block pair (17 dwords of a Q8_0 row, 9 of a Q4_0 one, the
// even block's quants 2 bytes off a dword, the odd block's on one).
struct R16Words {
  uint32_t e[4], o[2], z, y;
};
// The MFMA operands of the pair: quants of the even and the odd block, and the words
// holding d_even (low half) and d_odd (high half).
struct R16Ops {
  uint32_t e0, e1, o0, o1, se, so;
};

// Q8_0 against Q8_0: lane group k takes the even block's dword 2k + 1 and the halves
// around it (quants 8k .. 8k + 7 in the order 0 1 6 7 2 3 4 5), the odd block's
// dwords 2k, 2k + 1.  d_even is in group 0's words, d_odd in group 3's.
__device__ __forceinline__ void r16_read_q8(const uint32_t *w, int k, R16Words &r) {
  const uint32_t *e = w + 2 * k;
  r.e[0] = e[0];
  r.e[1] = e[1];
  r.e[2] = e[2];
  r.o[0] = e[9];
  r.o[1] = e[10];
}
__device__ __forceinline__ R16Ops r16_q8(const R16Words &r) {
  return {funnel16(r.e[0], r.e[2]), r.e[1], r.o[0], r.o[1], r.e[0], r.e[2]};
}

// Q8_0 against Q4_0, whose byte j holds quants j and 16 + j: group k takes quants 4k .. 4k + 3
// and 16 + 4k .. 16 + 4k + 3, and every group the scales.
__device__ __forceinline__ void r16_read_q8_for_q4(const uint32_t *w, int k, R16Words &r) {
  const uint32_t *e = w + k;
  r.e[0] = e[0];
  r.e[1] = e[1];
  r.e[2] = e[4];
  r.e[3] = e[5];
  r.o[0] = e[9];
  r.o[1] = e[13];
  r.z = w[0];
  r.y = w[8];
}
__device__ __forceinline__ R16Ops r16_q8_for_q4(const R16Words &r) {
  return {funnel16(r.e[0], r.e[1]), funnel16(r.e[2], r.e[3]), r.o[0], r.o[1], r.z, r.y};
}

// Q4_0: the same quants, as 16 (n - 8) (the offset-binary nibble with its top bit
// flipped, left in the byte's high half).  d_even is in group 0's word, d_odd in group 3's.
__device__ __forceinline__ void r16_read_q4(const uint32_t *w, int k, R16Words &r) {
  const uint32_t *e = w + k;
  r.e[0] = e[0];
  r.e[1] = e[1];
  r.o[0] = e[5];
}
__device__ __forceinline__ R16Ops r16_q4(const R16Words &r) {
  const uint32_t ev = funnel16(r.e[0], r.e[1]) ^ 0x88888888u, od = r.o[0] ^ 0x88888888u;
  return {(ev << 4) & 0xf0f0f0f0u, ev & 0xf0f0f0f0u, (od << 4) & 0xf0f0f0f0u, od & 0xf0f0f0f0u,
          r.e[0], r.e[1]};
}

__device__ __forceinline__ v4i r16_sums(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) {
  const long a = static_cast<long>((static_cast<uint64_t>(a1) << 32) | a0);
  const long b = static_cast<long>((static_cast<uint64_t>(b1) << 32) | b0);
  return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, v4i{}, 0, 0, 0);
}

// a0 b0 + a1 b1 of the operands' first two halves (k-slots 4k, 4k + 1 of group k): with one
// nonzero slot in all, one exact product.
__device__ __forceinline__ v4f r16_scales(uint32_t a, uint32_t b) {
  const v2h z = {};
  const v4h ha = __builtin_shufflevector(__builtin_bit_cast(v2h, a), z, 0, 1, 2, 3);
  const v4h hb = __builtin_shufflevector(__builtin_bit_cast(v2h, b), z, 0, 1, 2, 3);
  return __builtin_amdgcn_mfma_f32_16x16x16f16(ha, hb, v4f{}, 0, 0, 0);
}

// Work-group (x, y, z): the tile of XCD x's slot (y, z), tile_order.h.
template <bool kQ4, int kWM>
__global__ __launch_bounds__(kWM * 2 * 64, 2) void gemm_rows16(
    uint32_t units, uint32_t inv, const uint8_t *vx,
    size_t bx, const uint8_t *vy, size_t by, uint32_t nr, uint32_t nc, size_t nb, float *s,
    size_t bs) {
  constexpr int kWN = 2;
  constexpr int kCB = kR16Chunk;
  constexpr int kThreads = kWM * kWN * 64;
  constexpr int kBM = 16 * kWM, kBN = 16 * kWN;
  constexpr int kXBlock = kQ4 ? kQ4Bytes : kQ8Bytes;
  constexpr int kXSpan = kCB * kXBlock, kYSpan = kCB * kQ8Bytes;
  // row strides in LDS: 12 dwords past a multiple of the 64 banks
  constexpr int kXS = kXSpan + 16, kYS = kYSpan + 16;
  constexpr int kXL = kXSpan / 16 / 8 * 8, kYL = kYSpan / 16 / 8 * 8;  // pieces of whole-row loads
  constexpr int kXT = kXSpan / 16 - kXL, kYT = kYSpan / 16 - kYL;  // left over a row: 1 or 2
  constexpr int kXMain = (kBM * kXL + kThreads - 1) / kThreads;
  constexpr int kYMain = (kBN * kYL + kThreads - 1) / kThreads;
  constexpr int kTailPieces = kBM * kXT + kBN * kYT;
  constexpr int kTails = (kTailPieces + kThreads - 1) / kThreads;
  constexpr int kLoads = kXMain + kYMain + kTails;
  constexpr int kStage = kBM * kXS + kBN * kYS;
  __shared__ __align__(16) uint8_t lds[2][kStage];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % kWM, wn = wave / kWM;
  const TilePos tile = xcd_tile(units, (nr + kBM - 1) / kBM,
                                (nc + kBN - 1) / kBN, inv, blockIdx.x, blockIdx.y,
                                blockIdx.z);
  if (!tile.live)
    return;
  const size_t m0 = static_cast<size_t>(tile.tm) * kBM, n0 = static_cast<size_t>(tile.tn) * kBN;
  const uint32_t xlast = static_cast<uint32_t>(min(static_cast<size_t>(kBM), nr - m0)) - 1;
  const uint32_t ylast = static_cast<uint32_t>(min(static_cast<size_t>(kBN), nc - n0)) - 1;
  const uint8_t *xbase = vx + m0 * bx, *ybase = vy + n0 * by;
  const uint32_t bx32 = static_cast<uint32_t>(bx), by32 = static_cast<uint32_t>(by);

  uint32_t off[kLoads], dst[kLoads];
  int at[kLoads];
  bool isx[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    uint32_t r;
    bool x;
    if (j < kXMain) {
      const int f = min(j * kThreads + tid, kBM * kXL - 1);
      x = true;
      r = f / kXL;
      at[j] = 16 * (f % kXL);
    } else if (j < kXMain + kYMain) {
      const int f = min((j - kXMain) * kThreads + tid, kBN * kYL - 1);
      x = false;
      r = f / kYL;
      at[j] = 16 * (f % kYL);
    } else {
      const int f = min((j - kXMain - kYMain) * kThreads + tid, kTailPieces - 1);
      x = f < kBM * kXT;
      const int g = x ? f : f - kBM * kXT;
      r = x ? g / kXT : g / kYT;
      at[j] = 16 * (x ? kXL + g % kXT : kYL + g % kYT);
    }
    isx[j] = x;
    off[j] = x ? min(r, xlast) * bx32 : min(r, ylast) * by32;
    dst[j] = x ? r * kXS : kBM * kXS + r * kYS;
  }
  u32x4a2 raw[kLoads];
  // a partial chunk's pieces past its end repeat its last 16 bytes (a block is 18 at least)
  auto in_span = [&](int j, int nbc) {
    return static_cast<uint32_t>(min(at[j], nbc * (isx[j] ? kXBlock : kQ8Bytes) - 16));
  };
  auto load = [&](size_t c, int nbc) {
    const uint8_t *xc = xbase + c * kXSpan, *yc = ybase + c * kYSpan;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const uint8_t *base = j < kXMain ? xc : j < kXMain + kYMain ? yc : isx[j] ? xc : yc;
      raw[j] = *reinterpret_cast<const u32x4a2 *>(base + (off[j] + in_span(j, nbc)));
    }
  };
  auto put = [&](uint8_t *buf, int nbc) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      *reinterpret_cast<u32x4a2 *>(buf + dst[j] + in_span(j, nbc)) = raw[j];
  };

  const int li = lane & 15, k = lane >> 4;
  const uint32_t m_even = k == 0 ? 0xffffu : 0u, m_odd = k == 3 ? 0xffff0000u : 0u;
  // 1/16 beside a weight's scale (the Q4_0 sums are 16 sumi)
  const uint32_t one_even = 0x2c00u & m_even, one_odd = 0x2c000000u & m_odd;
  const int xo = (16 * wm + li) * kXS, yo = kBM * kXS + (16 * wn + li) * kYS;

  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // rows 4k .. 4k + 3 of token li

  struct Words {
    R16Words x, y;
  };
  struct Step {  // of a pair: the block sums, scale products and (Q4_0) token scales
    v4i e, o;
    v4f pe, po;
    float de, dy;
  };
  auto read = [&](const uint8_t *buf, int pp) {
    Words w;
    const uint32_t *xw = reinterpret_cast<const uint32_t *>(buf + xo) + pp * (2 * kXBlock / 4);
    const uint32_t *yw = reinterpret_cast<const uint32_t *>(buf + yo) + pp * (2 * kQ8Bytes / 4);
    if constexpr (kQ4) {
      r16_read_q4(xw, k, w.x);
      r16_read_q8_for_q4(yw, k, w.y);
    } else {
      r16_read_q8(xw, k, w.x);
      r16_read_q8(yw, k, w.y);
    }
    return w;
  };
  auto issue = [&](const Words &w) {
    Step st;
    const R16Ops x = kQ4 ? r16_q4(w.x) : r16_q8(w.x);
    const R16Ops y = kQ4 ? r16_q8_for_q4(w.y) : r16_q8(w.y);
    st.e = r16_sums(x.e0, x.e1, y.e0, y.e1);
    st.o = r16_sums(x.o0, x.o1, y.o0, y.o1);
    st.pe = r16_scales(x.se & m_even, kQ4 ? one_even : y.se & m_even);
    st.po = r16_scales(x.so & m_odd, kQ4 ? one_odd : y.so & m_odd);
    if constexpr (kQ4) {
      st.de = fp16_bits_to_f32(y.se & 0xffffu);
      st.dy = fp16_bits_to_f32(y.so >> 16);
    }
    return st;
  };
  auto fold = [&](const v4i &sums, const v4f &p, float dy) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (kQ4)
        acc[e] = fmaf(static_cast<float>(sums[e]) * p[e], dy, acc[e]);
      else
        acc[e] = fmaf(static_cast<float>(sums[e]), p[e], acc[e]);
    }
  };

  const size_t nchunks = (nb + kCB - 1) / kCB;
  auto blocks = [&](size_t c) { return static_cast<int>(min(nb - c * kCB, static_cast<size_t>(kCB))); };
  load(0, blocks(0));
  put(lds[0], blocks(0));
  if (nchunks > 1)
    load(1, blocks(1));
  __syncthreads();
  for (size_t c = 0; c < nchunks; ++c) {
    const uint8_t *buf = lds[c & 1];
    const int nbc = blocks(c);
    if (nbc == kCB) {
      // pair pp is folded, pair pp + 1's MFMAs issued and pair pp + 2 read in one step
      Words w = read(buf, 0);
      Step cur = issue(w);
      w = read(buf, 1);
#pragma unroll
      for (int pp = 0; pp < kCB / 2; ++pp) {
        Step nxt;
        if (pp + 1 < kCB / 2)
          nxt = issue(w);
        if (pp + 2 < kCB / 2)
          w = read(buf, pp + 2);
        fold(cur.e, cur.pe, cur.de);
        fold(cur.o, cur.po, cur.dy);
        __builtin_amdgcn_sched_barrier(0);
        if (pp + 1 < kCB / 2)
          cur = nxt;
      }
    } else {
      for (int pp = 0; 2 * pp < nbc; ++pp) {
        const Step st = issue(read(buf, pp));
        fold(st.e, st.pe, st.de);
        if (2 * pp + 1 < nbc)
          fold(st.o, st.po, st.dy);
      }
    }
    if (c + 1 < nchunks) {
      put(lds[(c + 1) & 1], blocks(c + 1));
      if (c + 2 < nchunks)
        load(c + 2, blocks(c + 2));
      __syncthreads();
    }
  }
  const size_t col = n0 + 16 * wn + li;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const size_t row = m0 + 16 * wm + 4 * k + e;
    if (row < nr && col < nc)
      s[row * bs + col] = acc[e];
  }
}

}  // namespace tcrv

namespace tcrv_host {

// 32- or 64-row work-groups, by rounds of 256 (a CU holds one or two of either).  Measured over
// 400 sizes, us a block of K beyond 1-3 us, Q4_0 / Q8_0: 32 rows, 1 to 4 rounds 0.085 / 0.082,
// 0.135 / 0.116, 0.193 / 0.193, 0.257 / 0.245, 7 rounds 0.43 / 0.41; 64 rows 0.125 / 0.113,
// 0.221 / 0.229, 0.337 / 0.373, 4 rounds 0.40 / 0.44.  Where a last 64-row tile is half empty the
// two have nearly as many work-groups: 31 x 9893 x 3840 Q8_0 24.5 / 31.9, 212 x 4169 x 2176 Q8_0
// 24.0 / 31.9, 2317 x 211 x 4960 Q4_0 26.0 / 37.6.
bool rows16_by_32(bool q4, size_t w32, size_t w64) {
  if (w64 <= 256)
    return w32 <= 256;
  if (w64 <= 512)
    return w32 <= 768;
  return w32 <= (q4 ? 1024 : 1792);
}

int gemm_rows16(bool q4, size_t nb, float *s, const uint8_t *vx, size_t bx, const uint8_t *vy,
                size_t by, size_t nr, size_t nc, size_t bs, void *stream) {
  // 32-bit row offsets within a work-group's 64 rows, and row and token counts
  if (bx > 0x03ffffffu || by > 0x03ffffffu || nr > 0xffffffffu || nc > 0xffffffffu)
    return TCRV_HIP_ERR_UNSUPPORTED;
  const size_t w32 = (nr + 31) / 32 * ((nc + 31) / 32), w64 = (nr + 63) / 64 * ((nc + 31) / 32);
  const bool rows32 = rows16_by_32(q4, w32, w64);
  const size_t mt = rows32 ? (nr + 31) / 32 : (nr + 63) / 64;
  tcrv::TileOrder o;
  if (!tcrv::tile_order(mt, (nc + 31) / 32, &o))
    return TCRV_HIP_ERR_UNSUPPORTED;
  const dim3 g(tcrv::kXcds, o.slots_y, o.slots_z);
  auto run = [&](auto kernel, int waves) {
    kernel<<<g, dim3(waves * 64), 0, as_stream(stream)>>>(
        o.units, o.inv, vx, bx, vy, by, static_cast<uint32_t>(nr),
        static_cast<uint32_t>(nc), nb, s, bs);
  };
  if (rows32)
    q4 ? run(tcrv::gemm_rows16<true, 2>, 4) : run(tcrv::gemm_rows16<false, 2>, 4);
  else
    q4 ? run(tcrv::gemm_rows16<true, 4>, 8) : run(tcrv::gemm_rows16<false, 4>, 8);
  return launch_status();
}

// Whether gemm_rows16 runs a shape of 4-byte aligned rows.  Measured over the same sizes, us:
//   - against gemm_rows_few, where that serves: up to two rounds of 32-row work-groups (4096 x 128
//     x 4096 18.4 / 16.6 against 31.0 / 26.7), four where its 64 x 64 ones, half empty at few tokens,
//     take two (18006 x 21 x 1792 Q8_0 13.7 / 18.9, 790 x 1238 x 3584 Q4_0 27.9 / 34.6), and three of
//     Q4_0 (0.193 against 0.214 a block) but for K 256, half a chunk (1166 x 596 5.8 / 5.0); three
//     of Q8_0 with K of whole chunks, a part chunk costing nearly a whole one (150 sizes, by
//     gemm_rows_few's time: 16 blocks 0.90, 64 0.93, 128 and 320 0.97, but 8 blocks 1.15, 24 1.08, 40
//     1.04, 72 1.02; 4245 x 142 x 2048 13.5 / 14.8 us);
//   - else, under 256 weight rows, against the 128 x 128 tiles (one round 0.40 / 0.36 a block): three
//     rounds of 64-row work-groups (Q4_0), five of 32-row ones (Q8_0) (190 x 8881 x 10432 Q8_0
//     138 / 125, 120 x 14581 x 960 Q4_0 19.7 / 17.4);
//   - else against the 256-row tiles (0.67 / 0.63 a block, few as they may be): four rounds of
//     64-row work-groups (K 4160, 4096 x 512 61 / 70 against 101 / 93.6, 4096 x 1000 118 / 138
//     against 101 / 92.5), five of 32-row ones of Q8_0 at K under 1024 (6192 x 244 x 640 17.9 / 16.9,
//     but 8672 x 116 x 576 13.4 / 15.3; Q4_0 977 x 1672 x 320 9.9 / 12.3).
bool rows16_first(bool q4, size_t nb, size_t nr, size_t nc, bool few_serves) {
  const size_t w32 = (nr + 31) / 32 * ((nc + 31) / 32), w64 = (nr + 63) / 64 * ((nc + 31) / 32);
  if (few_serves) {
    if (w32 <= 512 || (nr + 63) / 64 * ((nc + 63) / 64) > 256)
      return w32 <= 1024;
    return w32 <= 768 && (q4 ? nb >= 16 : nb % 16 == 0);
  }
  if (nr < 256)
    return q4 ? w64 <= 768 : w32 <= 1280;
  return nc <= 64 || (!q4 && nb < 32 ? w32 <= 1280 : w64 <= 1024);
}

int gemm_small(bool q4, bool rows4, size_t nb, float *s, const uint8_t *vx, size_t bx,
               const uint8_t *vy, size_t by, size_t nr, size_t nc, size_t bs, void *stream) {
  if (batch_first(rows4, nb, nr, nc))
    return gemm_batch(q4, nb, s, vx, bx, vy, by, nr, nc, bs, stream);
  if (nr > 1 && nc > 4 && (!rows4 || rows16_first(q4, nb, nr, nc,
                                                  rows_few_serves(nb, vx, bx, vy, by, nr, nc)))) {
    const int st = gemm_rows16(q4, nb, s, vx, bx, vy, by, nr, nc, bs, stream);
    if (st != TCRV_HIP_ERR_UNSUPPORTED)
      return st;
  }
  return rows4 ? TCRV_HIP_ERR_UNSUPPORTED
               : gemm_batch(q4, nb, s, vx, bx, vy, by, nr, nc, bs, stream);
}

}  // namespace tcrv_host
