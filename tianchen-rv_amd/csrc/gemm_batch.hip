// gemm_batch.hip -- a7 / a9 for a few tokens (batched decode), and for rows that are
// only 2-byte aligned (odd block counts) at any number of tokens: the reference GEMMs
// s[ir*bs + col] = block_dot(weight row ir, token col) straight from plain rows.
//
// What bounds it: each output is one serial fold of n/32 fmas (the reference's
// ascending-block order, RVVToEmitCBlockQuantLinear.cpp:322-356, :7538-7575), but
// the integer block sums under it are free of order.  So a work-group of 8 (or
// 16) waves owns a 16-row x 16-token tile (256 outputs: 4096 weight rows give
// one work-group a CU), its waves split K for the sums, and only the fmas run
// in order, one output a lane:
//   - K in chunks of 8 blocks a wave.  The wave loads its 8-block spans of the
//     16 weight rows and the tokens in 16-byte pieces (whole rows side by side:
//     a few cache lines an instruction), the next chunk's while this one is
//     computed, and writes them to its own LDS region;
//   - v_mfma_i32_16x16x32_i8 gives a block's 256 sums.  Its operands are read
//     from the raw spans as aligned dwords (an LDS read at a 2-byte offset
//     takes 32 cycles a wave against 4.6): a block pair is 17 dwords (Q8_0) or
//     9 (Q4_0), the odd block's quants dword aligned and the even block's
//     shifted by 2 bytes, so lane group k takes the pair's dwords in an order
//     that needs one funnel shift a pair instead of one a dword -- a dot
//     product does not care about the order of its terms as long as both
//     operands agree;
//   - the sums go back to LDS (over the raw spans) four blocks of an output
//     together, and after a work-group barrier waves 0-3 fold 64 outputs each,
//     one a lane, the scales beside them as the rows hold them.
// Measured (us, 4096 weight rows x K 4096 unless named; before it the
// multi-column GEMVs, the 64-row-tile kernel past 24 tokens, and for odd block
// counts a kernel of one wave an output or the raw 128 x 128 tiles):
//   8 tokens Q4_0 7.8 -> 6.2, Q8_0 8.8 -> 7.0; 16 tokens 15.4 -> 6.2, 15.8 ->
//   7.0; 32 tokens 30.6 -> 10.0, 26.4 -> 11.0; 3001 x 6 x 2912 (91 blocks)
//   27.5 -> 7.0, 397 -> 7.5; one token, Q8_0 4096 x 14304 (447 blocks) 2110 -> 21
//   (Q4_0 decodes on gemv.hip's LDS-staged kernel, and its few outputs of odd block
//   counts a wave each, block_dot.hip).
#include "tcrv_hip_internal.h"
#include "mfma_fold.h"
#include "tile_order.h"

#include <type_traits>

namespace tcrv {

constexpr int kBtRows = 16, kBtToks = 16;     // work-group tile
constexpr int kBtSlice = 8;                   // blocks of a wave in a chunk
constexpr int kBtYSpan = kBtSlice * kQ8Bytes; // 272: a token's span of a slice
constexpr int kBtQuad = 16 * 272;             // four blocks' sums of 256 outputs (17 float4 a token)
constexpr int kBtRegion = 2 * kBtQuad;        // 8704: a wave's raw spans, then its sums

typedef uint32_t u32x4a2 __attribute__((ext_vector_type(4), aligned(2)));

// The operands of a block pair in MFMA form: quants of the even and the odd
// block (two dwords each) and the pair's scales (d_even | d_odd << 16, valid in
// lane group 3).
struct BtPair {
  uint32_t e0, e1, o0, o1, d;
};

// A Q8_0 pair (17 dwords at w) against another Q8_0 operand: lane group k takes
// the even block's dwords 1 + 2k, 2 + 2k (group 3 the last dword's first half
// beside dword 0's second: quants 30, 31, 0, 1) and the odd block's 9 + 2k, 10 + 2k.
__device__ __forceinline__ BtPair bt_q8_pair(const uint32_t *w, int k) {
  BtPair p;
  const uint32_t z = w[0];
  p.e0 = w[1 + 2 * k];
  const uint32_t e1 = w[2 + 2 * k];
  p.o0 = w[9 + 2 * k];
  p.o1 = w[10 + 2 * k];
  p.e1 = k == 3 ? funnel16(z, e1) : e1;
  p.d = (z & 0xffffu) | (e1 & 0xffff0000u);
  return p;
}

// A Q8_0 pair against a Q4_0 one, whose byte j carries quants j and 16 + j:
// group k takes quants p, 16 + p for its four byte positions p -- even block
// 2 + 4k .. 5 + 4k (group 3: 0, 1, 14, 15), odd block 4k .. 4k + 3.
__device__ __forceinline__ BtPair bt_q8_pair_for_q4(const uint32_t *w, int k) {
  BtPair p;
  const uint32_t z = w[0], a = w[1 + k], b = w[5 + k];
  p.o0 = w[9 + k];
  p.o1 = w[13 + k];
  p.e0 = k == 3 ? funnel16(z, a) : a;
  p.e1 = k == 3 ? funnel16(a, b) : b;
  p.d = (z & 0xffffu) | (b & 0xffff0000u);
  return p;
}

// A Q4_0 pair (9 dwords): the same byte positions, the nibbles as 16 (n - 8) --
// the offset-binary nibble with its top bit flipped, left in the byte's high
// half.  Sums, terms and the running fold are then 16 times the reference's, exactly (a power
// of two, and nothing comes near either end of the exponent range: terms are
// multiples of 2^-48 below 2^47), and the stored value is acc / 16.
__device__ __forceinline__ BtPair bt_q4_pair(const uint32_t *w, int k) {
  BtPair p;
  const uint32_t z = w[0], a = w[1 + k];
  const uint32_t ev = (k == 3 ? funnel16(z, a) : a) ^ 0x88888888u;
  const uint32_t od = w[5 + k] ^ 0x88888888u;
  p.e0 = (ev << 4) & 0xf0f0f0f0u;
  p.e1 = ev & 0xf0f0f0f0u;
  p.o0 = (od << 4) & 0xf0f0f0f0u;
  p.o1 = od & 0xf0f0f0f0u;
  p.d = (z & 0xffffu) | (a & 0xffff0000u);
  return p;
}

__device__ __forceinline__ v4i bt_sums(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) {
  const long a = static_cast<long>((static_cast<uint64_t>(a1) << 32) | a0);
  const long b = static_cast<long>((static_cast<uint64_t>(b1) << 32) | b0);
  return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, v4i{}, 0, 0, 0);
}

// The tile of rows row0.. and tokens tok0..  At most four waves a SIMD (the kernels' bounds): two
// work-groups of 8 waves a CU, one of 16.  kWide: row strides past 256 MB.
template <bool kQ4, int kWaves, bool kWide>
__device__ __forceinline__ void batch_tile(size_t row0, unsigned tok0, const uint8_t *vx, size_t bx,
                                           const uint8_t *vy, size_t by, size_t nr, size_t nb,
                                           unsigned nc, float *s, size_t bs) {
  using Off = std::conditional_t<kWide, size_t, uint32_t>;  // of a row from the tile's first
  constexpr int kChunk = kWaves * kBtSlice;  // blocks
  constexpr int kXBlock = kQ4 ? kQ4Bytes : kQ8Bytes;
  constexpr int kXSpan = kBtSlice * kXBlock;                 // 144 or 272
  constexpr int kXPieces = kXSpan / 16;
  constexpr int kXLanes = kXPieces - 1;                      // 8 or 16 lanes a row
  constexpr int kXMain = kBtRows * kXLanes / 64, kYMain = 4; // whole-row instructions
  constexpr int kLoads = kXMain + kYMain + 1;                // 7 or 9 a lane
  constexpr int kXAll = kBtRows * kXSpan;                    // the tokens' spans follow
  constexpr int kSRow = kChunk / 2 + 4;                    // scale pairs of a row (+ pad)
  static_assert(kXAll + kBtToks * kBtYSpan <= kBtRegion, "raw spans fit the region");
  __shared__ __align__(16) uint8_t lds[kWaves * kBtRegion];
  __shared__ __align__(16) uint32_t sx[kBtRows][kSRow], sy[kBtToks][kSRow];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int ntok = static_cast<int>(min(nc - tok0, static_cast<unsigned>(kBtToks)));
  uint8_t *region = lds + wave * kBtRegion;

  // This lane's pieces: instruction j < kXMain + kYMain moves the first 16 (8 for
  // Q4_0 weights) pieces of several rows, whole rows side by side; the last one
  // the rows' last pieces (lanes 0-15 the weights', 16-31 the tokens', twice).
  // Rows past nr and tokens past nc repeat the last one (never stored).
  const uint8_t *xbase = vx + row0 * bx + wave * kXSpan;
  const uint8_t *ybase = vy + static_cast<size_t>(tok0) * by + wave * kBtYSpan;
  const int xlast = static_cast<int>(min(static_cast<size_t>(kBtRows), nr - row0)) - 1;
  const Off bxo = static_cast<Off>(bx), byo = static_cast<Off>(by);
  auto piece_row = [&](int j) {
    return j < kXMain           ? j * (64 / kXLanes) + lane / kXLanes
           : j < kXMain + kYMain ? (j - kXMain) * 4 + lane / 16
                                 : lane & 15;
  };
  const bool tail_x = (lane & 16) == 0;
  Off off[kLoads];       // of the row from its operand's base
  uint32_t dst[kLoads];  // of the row's span in the region
  int at[kLoads];        // of the piece in the span
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const bool x = j < kXMain || (j == kLoads - 1 && tail_x);
    const int r = piece_row(j);
    at[j] = j < kXMain           ? 16 * (lane % kXLanes)
            : j < kXMain + kYMain ? 16 * (lane % 16)
                                  : (x ? kXSpan : kBtYSpan) - 16;
    off[j] = x ? static_cast<Off>(min(r, xlast)) * bxo : static_cast<Off>(min(r, ntok - 1)) * byo;
    dst[j] = x ? r * kXSpan : kXAll + r * kBtYSpan;
  }
  // blocks of chunk c, and of this wave's slice of it
  auto chunk_blocks = [&](size_t c) {
    return static_cast<int>(min(nb - c * kChunk, static_cast<size_t>(kChunk)));
  };
  auto slice_blocks = [&](size_t c) {
    return min(max(chunk_blocks(c) - wave * kBtSlice, 0), kBtSlice);
  };
  // A partial slice's pieces past its end repeat its last 16 bytes (a block is
  // 18 at least), so no load leaves the span.
  auto in_span = [&](int j, int nbw) {
    const bool x = j < kXMain || (j == kLoads - 1 && tail_x);
    return static_cast<uint32_t>(min(at[j], nbw * (x ? kXBlock : kQ8Bytes) - 16));
  };
  u32x4a2 raw[kLoads];
  auto load = [&](size_t c, int nbw) {
    const uint8_t *xc = xbase + c * (kChunk * kXBlock);
    const uint8_t *yc = ybase + c * (kChunk * kQ8Bytes);
    const uint8_t *tc = tail_x ? xc : yc;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const uint8_t *base = j < kXMain ? xc : j < kXMain + kYMain ? yc : tc;
      raw[j] = *reinterpret_cast<const u32x4a2 *>(base + (off[j] + in_span(j, nbw)));
    }
  };
  auto put = [&](int nbw) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      *reinterpret_cast<u32x4a2 *>(region + dst[j] + in_span(j, nbw)) = raw[j];
  };

  const int li = lane & 15, k = lane >> 4;  // MFMA row / token, lane group
  const uint32_t *xrow = reinterpret_cast<const uint32_t *>(region + li * kXSpan);
  const uint32_t *yrow = reinterpret_cast<const uint32_t *>(region + kXAll + li * kBtYSpan);
  // the fold's output of this lane (waves 0-3): row 4 wave + lane / 16, token lane % 16
  const int fr = 4 * (wave & 3) + k;
  const uint8_t *ft = lds + li * 272 + fr * 16;
  float acc = 0.0f;
  struct Eight {  // a slice's blocks of the output: sums and scale pairs
    float4 v[2];
    uint4 dx, dy;
  };
  auto read8 = [&](int w) {
    Eight t;
    t.v[0] = *reinterpret_cast<const float4 *>(ft + w * kBtRegion);
    t.v[1] = *reinterpret_cast<const float4 *>(ft + w * kBtRegion + kBtQuad);
    t.dx = *reinterpret_cast<const uint4 *>(&sx[fr][4 * w]);
    t.dy = *reinterpret_cast<const uint4 *>(&sy[li][4 * w]);
    return t;
  };
  // products with an fp16 scale as fma(., ., -0): v_fma_mix_f32 reads the half in
  // place, and adding -0 changes no product, zero signs included
  auto step = [&](float fs, uint32_t dx, uint32_t dy) {
    const float x = fp16_bits_to_f32(dx), y = fp16_bits_to_f32(dy);
    if constexpr (kQ4)
      acc = fmaf(fmaf(fs, x, -0.0f), y, acc);
    else
      acc = fmaf(fs, fmaf(x, y, -0.0f), acc);
  };
  auto fold_pair = [&](float f0, float f1, uint32_t dx, uint32_t dy, int n) {
    if (n > 0)
      step(f0, dx & 0xffffu, dy & 0xffffu);
    if (n > 1)
      step(f1, dx >> 16, dy >> 16);
  };
  auto fold8 = [&](const Eight &t, int n) {
    fold_pair(t.v[0].x, t.v[0].y, t.dx.x, t.dy.x, n);
    fold_pair(t.v[0].z, t.v[0].w, t.dx.y, t.dy.y, n - 2);
    fold_pair(t.v[1].x, t.v[1].y, t.dx.z, t.dy.z, n - 4);
    fold_pair(t.v[1].z, t.v[1].w, t.dx.w, t.dy.w, n - 6);
  };

  const size_t nchunks = (nb + kChunk - 1) / kChunk;
  int nbw = slice_blocks(0);
  if (nbw > 0)
    load(0, nbw);
  for (size_t c = 0; c < nchunks; ++c) {
    if (nbw > 0) {
      put(nbw);
      const int nbn = c + 1 < nchunks ? slice_blocks(c + 1) : 0;
      if (nbn > 0)
        load(c + 1, nbn);
      nbw = nbn;
      wave_lds_sync();
      float f[2][4][4];  // quad, block, output row of the lane's four
      uint32_t dx[4], dy[4];
#pragma unroll
      for (int pp = 0; pp < kBtSlice / 2; ++pp) {
        BtPair x, y;
        if constexpr (kQ4) {
          x = bt_q4_pair(xrow + pp * (2 * kQ4Bytes / 4), k);
          y = bt_q8_pair_for_q4(yrow + pp * (2 * kQ8Bytes / 4), k);
        } else {
          x = bt_q8_pair(xrow + pp * (2 * kQ8Bytes / 4), k);
          y = bt_q8_pair(yrow + pp * (2 * kQ8Bytes / 4), k);
        }
        dx[pp] = x.d;
        dy[pp] = y.d;
        const v4i se = bt_sums(x.e0, x.e1, y.e0, y.e1);
        const v4i so = bt_sums(x.o0, x.o1, y.o0, y.o1);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f[pp >> 1][2 * (pp & 1)][e] = static_cast<float>(se[e]);
          f[pp >> 1][2 * (pp & 1) + 1][e] = static_cast<float>(so[e]);
        }
      }
      wave_lds_sync();  // every raw read is issued before the sums overwrite the spans
      if (k == 3) {
        *reinterpret_cast<uint4 *>(&sx[li][4 * wave]) = make_uint4(dx[0], dx[1], dx[2], dx[3]);
        *reinterpret_cast<uint4 *>(&sy[li][4 * wave]) = make_uint4(dy[0], dy[1], dy[2], dy[3]);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *reinterpret_cast<float4 *>(region + q * kBtQuad + li * 272 + (4 * k + e) * 16) =
              make_float4(f[q][0][e], f[q][1][e], f[q][2][e], f[q][3][e]);
    }
    __syncthreads();
    if (wave < 4) {
      const int nbc = chunk_blocks(c);
      if (nbc == kChunk) {  // each slice read two ahead of its fold
        Eight t[2] = {read8(0), read8(1)};
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          const Eight u = t[w & 1];
          if (w + 2 < kWaves)
            t[w & 1] = read8(w + 2);
          fold8(u, 8);
        }
      } else {
        const int nw = nbc >> 3, rest = nbc & 7;
        Eight t = read8(0);
        for (int w = 0; w < nw; ++w) {
          const Eight u = t;
          t = read8(min(w + 1, kWaves - 1));
          fold8(u, 8);
        }
        fold8(t, rest);
      }
    }
    __syncthreads();
  }
  if (wave < 4 && row0 + fr < nr && li < ntok)
    s[(row0 + fr) * bs + tok0 + li] = kQ4 ? acc * 0.0625f : acc;
}

// Work-group (x, y, z): the tile of XCD x's slot (y, z), tile_order.h.
template <bool kQ4, int kWaves, bool kWide>
__global__ __launch_bounds__(kWaves * 64, 4) void gemm_batch(
    const uint8_t *vx, size_t bx, const uint8_t *vy, size_t by, size_t nb, uint32_t nr, uint32_t nc,
    uint32_t units, uint32_t inv, float *s, size_t bs) {
  const TilePos tile = xcd_tile(units, (nr + kBtRows - 1) / kBtRows, (nc + kBtToks - 1) / kBtToks,
                                inv, blockIdx.x, blockIdx.y, blockIdx.z);
  if (tile.live)
    batch_tile<kQ4, kWaves, kWide>(static_cast<size_t>(tile.tm) * kBtRows, tile.tn * kBtToks, vx, bx,
                                   vy, by, nr, nb, nc, s, bs);
}

// One token group: the row tiles dealt in turn, which is as even and spares a wave the order's
// arithmetic (1-2 % of a 4-7 us kernel).
template <bool kQ4, int kWaves>
__global__ __launch_bounds__(kWaves * 64, 4) void gemm_batch_one(
    const uint8_t *vx, size_t bx, const uint8_t *vy, size_t by, size_t nr, size_t nb, unsigned nc,
    float *s, size_t bs) {
  const unsigned tile = blockIdx.x + kXcds * blockIdx.y;
  const size_t row0 = static_cast<size_t>(tile) * kBtRows;
  if (row0 < nr)
    batch_tile<kQ4, kWaves, false>(row0, 0, vx, bx, vy, by, nr, nb, nc, s, bs);
}

}  // namespace tcrv

namespace tcrv_host {

int gemm_batch(bool q4, size_t nb, float *s, const uint8_t *vx, size_t bx, const uint8_t *vy,
               size_t by, size_t nr, size_t nc, size_t bs, void *stream) {
  // a launch takes 65535 x 8 row tiles, then as many token groups as its tiles allow
  constexpr size_t kMaxRows = static_cast<size_t>(65535) * 8 * tcrv::kBtRows;
  const bool wide = bx > 0x0fffffffu || by > 0x0fffffffu;
  hipStream_t st = as_stream(stream);
  for (size_t r0 = 0; r0 < nr; r0 += kMaxRows) {
    const size_t rows = nr - r0 < kMaxRows ? nr - r0 : kMaxRows;
    const size_t tiles = (rows + tcrv::kBtRows - 1) / tcrv::kBtRows;
    const size_t max_toks = (tcrv::kMaxTiles - 1) / tiles * tcrv::kBtToks;
    for (size_t c0 = 0; c0 < nc; c0 += max_toks) {
      const size_t toks = nc - c0 < max_toks ? nc - c0 : max_toks;
      const size_t groups = (toks + tcrv::kBtToks - 1) / tcrv::kBtToks;
      const uint8_t *x = vx + r0 * bx, *y = vy + c0 * by;
      float *out = s + r0 * bs + c0;
      const uint32_t nt = static_cast<uint32_t>(toks);
      // 16 waves where they hold all of K in one chunk and 8 would not, and a CU
      // has one work-group at most (4096 x 16 x 4096 Q4_0 6.2 against 6.8 us,
      // Q8_0 7.0 against 8.0); with more work-groups two of 8 waves overlap
      // each other's loads (4096 x 32: 10.1 against 11.2; 4096 x 16 x 14336
      // 17.6 against 21.2)
      const bool w16 = nb > 64 && nb <= 128 && tiles * groups <= 256;
      if (groups == 1 && !wide) {
        auto run = [&](auto kernel, int waves) {
          kernel<<<dim3(tcrv::kXcds, static_cast<unsigned>((tiles + 7) / 8)), dim3(waves * 64), 0,
                   st>>>(x, bx, y, by, rows, nb, nt, out, bs);
        };
        if (w16)
          q4 ? run(tcrv::gemm_batch_one<true, 16>, 16) : run(tcrv::gemm_batch_one<false, 16>, 16);
        else
          q4 ? run(tcrv::gemm_batch_one<true, 8>, 8) : run(tcrv::gemm_batch_one<false, 8>, 8);
      } else {
        tcrv::TileOrder o;
        if (!tcrv::tile_order(tiles, groups, &o))
          return TCRV_HIP_ERR_TOO_LARGE;
        auto run = [&](auto kernel, int waves) {
          kernel<<<dim3(tcrv::kXcds, o.slots_y, o.slots_z), dim3(waves * 64), 0, st>>>(
              x, bx, y, by, nb, static_cast<uint32_t>(rows), nt, o.units, o.inv, out, bs);
        };
        if (wide)
          q4 ? run(tcrv::gemm_batch<true, 8, true>, 8) : run(tcrv::gemm_batch<false, 8, true>, 8);
        else if (w16)
          q4 ? run(tcrv::gemm_batch<true, 16, false>, 16)
             : run(tcrv::gemm_batch<false, 16, false>, 16);
        else
          q4 ? run(tcrv::gemm_batch<true, 8, false>, 8)
             : run(tcrv::gemm_batch<false, 8, false>, 8);
      }
      const int rc = launch_status();
      if (rc != TCRV_HIP_OK)
        return rc;
    }
  }
  return TCRV_HIP_OK;
}

}  // namespace tcrv_host
