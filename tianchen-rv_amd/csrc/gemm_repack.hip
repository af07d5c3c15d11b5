// gemm_repack.hip -- tcrv_rvv.repack_gemm_q4_0_q8_0 (x16 Q4_0 weights, 4-row interleaved
// Q8_0 activations; RVVOps.td:4228-4338) for prompts: the 256 x 128 tiles of
// gemm_repack_q4_0 give nr / 256 * nc / 128 work-groups, 64 for 4096 weight rows x
// 512 tokens, one round of ~87 us at K 4096 however few.
//
// Here a wave folds one 32 x 32 tile and a work-group 64 x 64 (4 waves) or 128 x 64 (8
// waves, two a SIMD) outputs.  K in chunks of 8 blocks, two chunks ahead in
// registers, turned into row-major int8 rows in one of two LDS buffers:
//   - weights: a thread takes four byte positions of four rows of a block (four
//     dwords), one 4 x 4 byte transpose, the nibbles as 16 (n - 8) -- the x16
//     bytes are already offset by ^0x88, so a shift and two masks decode eight
//     quants; every sum and the running fold is then 16 times the reference's, exactly
//     (a power of two, and the folds stay far from either end of the exponent
//     range: the terms are multiples of 2^-48 below 2^47), and the stored value
//     is acc / 16;
//   - activations: a lane takes 8 elements of four rows (32 consecutive bytes, a
//     wave two whole spans side by side), two transposes, one 8-byte LDS write a row.
// The steps are gemm_wide's: the next block's MFMAs issued before a block is folded.
// Measured (us, K 4096, the GEMM alone): 4096 x 64 83 -> 24, 4096 x 256 87 -> 26.4, 4096
// x 512 88 -> 33.6, 4096 x 1024 89 -> 65; 11968 x 304 x 9088 184 -> 133.  Bound
// by its VALU (47 a wave and block, 32 of them the fold) and a quarter of a wave's time in
// waits; one chunk ahead instead of two cost 2 us.
#include "tcrv_hip_internal.h"
#include "mfma_fold.h"
#include "tile_order.h"

namespace tcrv {

constexpr int kRpX16 = 288, kRpX4 = 136;  // bytes of a block_q4_0x16, a block_q8_0x4
constexpr int kRpKB = 8;                  // blocks per K chunk
constexpr int kRpRow = kRpKB * kQK + 16;  // quant bytes per staged row (+16 pad: 16-byte reads of
                                          // 16 consecutive rows hit distinct banks)

struct RpOps {
  v4i a, b;
  uint32_t ux, uy;
};
struct RpStep {
  v16i sumi;
  v16f dxy;
};

// Work-group (x, y, z): the tile of XCD x's slot (y, z), tile_order.h.  Weight groups past ngw and token groups past nga repeat the last one
// (never stored).
template <int kWM, int kWN>
__global__ __launch_bounds__(kWM * kWN * 64, 2) void gemm_repack_mid(
    uint32_t units, uint32_t inv, size_t nb,
    const uint8_t *vx, const uint8_t *vy, size_t ngw, size_t nga, float *s, size_t bs,
    bool vec_out) {
  constexpr int kThreads = kWM * kWN * 64;
  constexpr int kBM = 32 * kWM, kBN = 32 * kWN, kRows = kBM + kBN;
  constexpr int kHRow = kRows + 32;  // fp16 scales of a block (+ 32 zero rows)
  constexpr int kWTasks = kBM / 16 * kRpKB * 16;  // (x16 block, position quad, row quad)
  constexpr int kWEach = kWTasks / kThreads;      // 1 or 2 a thread
  constexpr int kAEach = kBN / 8 / (kWM * kWN);   // x4 group pairs a wave
  static_assert(kAEach * 8 * kWM * kWN == kBN, "whole group pairs");
  constexpr int kScales = kBM / 16 * kRpKB * 4 + kBN / 4 * kRpKB;  // 8-byte scale loads
  static_assert(kWTasks % kThreads == 0 && kScales <= kThreads, "tasks");
  __shared__ __align__(16) int8_t q[2][kRows * kRpRow];
  __shared__ __align__(16) uint16_t dsh[2][kRpKB][kHRow];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % kWM, wn = wave / kWM;
  const int li = lane & 31, h = lane >> 5;
  const size_t nrw = ngw * 16, ntok = nga * 4;
  const TilePos tile = xcd_tile(units, static_cast<uint32_t>((nrw + kBM - 1) / kBM),
                                static_cast<uint32_t>((ntok + kBN - 1) / kBN), inv, blockIdx.x, blockIdx.y,
                                blockIdx.z);
  if (!tile.live)
    return;
  const size_t m0 = static_cast<size_t>(tile.tm) * kBM, n0 = static_cast<size_t>(tile.tn) * kBN;

  // weight tasks: lane order (group, block, position quad, row quad)
  const uint8_t *wsrc[kWEach];
  int wdst[kWEach], wblk[kWEach];
#pragma unroll
  for (int j = 0; j < kWEach; ++j) {
    const int t = j * kThreads + tid;
    const int rq = t & 3, pq = (t >> 2) & 3, b = (t >> 4) & (kRpKB - 1), g = t / (16 * kRpKB);
    wsrc[j] = vx + (min(m0 / 16 + g, ngw - 1) * nb + b) * kRpX16 + 32 + 64 * pq + 4 * rq;
    wdst[j] = (16 * g + 4 * rq) * kRpRow + kQK * b + 4 * pq;
    wblk[j] = b;
  }
  // activation tasks: lane = (group of the pair, block, 8 elements x 4 rows: 32 bytes)
  const int ab = (lane >> 2) & 7, ap = lane & 3;
  const uint8_t *asrc[kAEach];
  int adst[kAEach];
#pragma unroll
  for (int j = 0; j < kAEach; ++j) {
    const int g = 2 * (wave * kAEach + j) + (lane >> 5);
    asrc[j] = vy + (min(n0 / 4 + g, nga - 1) * nb + ab) * kRpX4 + 8 + 32 * ap;
    adst[j] = (kBM + 4 * g) * kRpRow + kQK * ab + 8 * ap;
  }
  // scales: four rows' (8 bytes) a thread, the weights' first
  constexpr int kSW = kBM / 16 * kRpKB * 4;
  const bool sw = tid < kSW;
  const int st_ = sw ? tid : tid - kSW;
  const int sb = sw ? (st_ >> 2) & (kRpKB - 1) : st_ & (kRpKB - 1);
  const int sg = sw ? st_ / (4 * kRpKB) : st_ / kRpKB;
  const bool has_scale = tid < kScales;
  const uint8_t *ssrc = sw ? vx + (min(m0 / 16 + sg, ngw - 1) * nb + sb) * kRpX16 + 8 * (st_ & 3)
                           : vy + (min(n0 / 4 + sg, nga - 1) * nb + sb) * kRpX4;
  const int sdst = sw ? 16 * sg + 4 * (st_ & 3) : kBM + 4 * sg;

  struct Regs {
    uint32_t w[kWEach][4], a[kAEach][8], s[2];
  };
  // chunk c, nbc of its blocks present: a task of an absent block repeats the chunk's first
  auto load = [&](Regs &r, size_t c, int nbc) {
#pragma unroll
    for (int j = 0; j < kWEach; ++j) {
      const uint8_t *p = wsrc[j] + (c * kRpKB - (wblk[j] < nbc ? 0 : wblk[j])) * kRpX16;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r.w[j][i] = *reinterpret_cast<const uint32_t *>(p + 16 * i);
    }
#pragma unroll
    for (int j = 0; j < kAEach; ++j) {
      const uint32_t *p = reinterpret_cast<const uint32_t *>(
          asrc[j] + (c * kRpKB - (ab < nbc ? 0 : ab)) * kRpX4);
      typedef uint32_t u32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
      const u32x4a4 v = *reinterpret_cast<const u32x4a4 *>(p);
      const u32x4a4 u = *reinterpret_cast<const u32x4a4 *>(p + 4);
      r.a[j][0] = v.x; r.a[j][1] = v.y; r.a[j][2] = v.z; r.a[j][3] = v.w;
      r.a[j][4] = u.x; r.a[j][5] = u.y; r.a[j][6] = u.z; r.a[j][7] = u.w;
    }
    if (has_scale) {
      const uint32_t *p = reinterpret_cast<const uint32_t *>(
          ssrc + (c * kRpKB - (sb < nbc ? 0 : sb)) * (sw ? kRpX16 : kRpX4));
      r.s[0] = p[0];
      r.s[1] = p[1];
    }
  };
  auto put = [&](const Regs &r, int st) {
#pragma unroll
    for (int j = 0; j < kWEach; ++j) {
      uint32_t rows[4];
      transpose4x4(r.w[j], rows);  // rows[rr]: positions 4pq .. 4pq + 3 of row 4rq + rr
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        int8_t *d = q[st] + wdst[j] + rr * kRpRow;
        *reinterpret_cast<uint32_t *>(d) = (rows[rr] << 4) & 0xf0f0f0f0u;
        *reinterpret_cast<uint32_t *>(d + 16) = rows[rr] & 0xf0f0f0f0u;
      }
    }
#pragma unroll
    for (int j = 0; j < kAEach; ++j) {
      uint32_t lo[4], hi[4];
      transpose4x4(&r.a[j][0], lo);  // lo[c], hi[c]: elements 8ap .. 8ap + 7 of row c
      transpose4x4(&r.a[j][4], hi);
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *reinterpret_cast<uint2 *>(q[st] + adst[j] + c * kRpRow) = make_uint2(lo[c], hi[c]);
    }
    if (has_scale)
      *reinterpret_cast<uint2 *>(&dsh[st][sb][sdst]) = make_uint2(r.s[0], r.s[1]);
  };

  for (int t = tid; t < 2 * kRpKB * 32; t += kThreads)  // the zero rows of both stages
    dsh[t / (kRpKB * 32)][t / 32 % kRpKB][kRows + t % 32] = 0;

  const int qa = (32 * wm + li) * kRpRow + 16 * h, qb = (kBM + 32 * wn + li) * kRpRow + 16 * h;
  const int hx = h ? kRows + li : 32 * wm + li, hy = h ? kRows + li : kBM + 32 * wn + li;
  auto ops = [&](int st, int b) {
    RpOps o;
    o.a = *reinterpret_cast<const v4i *>(q[st] + qa + b * kQK);
    o.b = *reinterpret_cast<const v4i *>(q[st] + qb + b * kQK);
    o.ux = dsh[st][b][hx];
    o.uy = dsh[st][b][hy];
    return o;
  };
  auto issue = [&](const RpOps &o) {
    RpStep t;
    t.sumi = q8_sumi(o.a, o.b);
    t.dxy = q8_dxy(o.ux, o.uy);
    return t;
  };
  float acc[16];
#pragma unroll
  for (int e = 0; e < 16; ++e)
    acc[e] = 0.0f;

  const size_t nchunks = (nb + kRpKB - 1) / kRpKB;
  auto blocks = [&](size_t c) {
    return static_cast<int>(min(nb - c * kRpKB, static_cast<size_t>(kRpKB)));
  };
  // chunk c (its buffer ready): chunk c + 2 loaded into `in`, chunk c + 1 in `out` staged
  auto chunk = [&](size_t c, Regs &in, const Regs &out) {
    const int st = static_cast<int>(c & 1);
    const int nbc = blocks(c);
    if (c + 2 < nchunks)
      load(in, c + 2, blocks(c + 2));
    if (nbc == kRpKB) {
      RpOps o = ops(st, 0);
      RpStep cur = issue(o);
      o = ops(st, 1);
#pragma unroll
      for (int b = 0; b < kRpKB; ++b) {
        RpStep nxt;
        if (b + 1 < kRpKB)
          nxt = issue(o);
        if (b + 2 < kRpKB)
          o = ops(st, b + 2);
        q8_fold<true>(acc, cur.sumi, cur.dxy);
        __builtin_amdgcn_sched_barrier(0);
        if (b + 1 < kRpKB)
          cur = nxt;
      }
    } else {
      for (int b = 0; b < nbc; ++b) {
        const RpStep t = issue(ops(st, b));
        q8_fold(acc, t.sumi, t.dxy);
      }
    }
    if (c + 1 < nchunks) {
      put(out, st ^ 1);
      __syncthreads();
    }
  };
  Regs r0, r1;
  load(r0, 0, blocks(0));
  if (nchunks > 1)
    load(r1, 1, blocks(1));
  put(r0, 0);
  __syncthreads();
  for (size_t c = 0; c < nchunks; c += 2) {
    chunk(c, r0, r1);
    if (c + 1 < nchunks)
      chunk(c + 1, r1, r0);
  }

  const size_t tok = n0 + 32 * wn + li;
  if (tok < ntok) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const size_t row = m0 + 32 * wm + 8 * g + 4 * h;
      if (row >= nrw)
        continue;
      float *d = s + tok * bs + row;
      if (vec_out) {
        *reinterpret_cast<float4 *>(d) =
            make_float4(acc[4 * g] * 0.0625f, acc[4 * g + 1] * 0.0625f, acc[4 * g + 2] * 0.0625f,
                        acc[4 * g + 3] * 0.0625f);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          d[e] = acc[4 * g + e] * 0.0625f;
      }
    }
  }
}

}  // namespace tcrv

namespace tcrv_host {

int gemm_repack_mid(size_t nb, float *s, const uint8_t *vx, const uint8_t *vy, size_t ngw,
                    size_t nga, size_t bs, bool vec_out, size_t wide_tiles, void *stream) {
  const size_t nrw = ngw * 16, ntok = nga * 4;
  const size_t nt = (ntok + 63) / 64;
  const size_t t64 = (nrw + 63) / 64 * nt, t128 = (nrw + 127) / 128 * nt;
  // Rounds times a round's time at K 4096 (us): 256 work-groups of 128 x 64 outputs 33; of
  // 64 x 64, up to 256 26, then 512 (two a CU) 38; of the 256 x 128 kernel 87.
  // Measured, 64 / 128 / 256 rows: 4096 x 256 26.4 / 32.6 / 87, 4096 x 512 38.8 / 33.6 / 88,
  // 4096 x 1024 74 / 65 / 89, 4096 x 2048 137 / 129 / 96, 14336 x 512 119 / 126 / 92,
  // 3024 x 2584 x 2304 84 / 79 / 60.
  const size_t c64 = t64 <= 256 ? 26 : (t64 + 511) / 512 * 38;
  const size_t c128 = (t128 + 255) / 256 * 33, c256 = (wide_tiles + 255) / 256 * 87;
  if (c256 < c64 && c256 < c128)
    return TCRV_HIP_ERR_UNSUPPORTED;
  const bool rows64 = c64 <= c128;
  tcrv::TileOrder o;
  if (!tcrv::tile_order(rows64 ? (nrw + 63) / 64 : (nrw + 127) / 128, nt, &o))
    return TCRV_HIP_ERR_UNSUPPORTED;
  auto run = [&](auto kernel, int waves) {
    kernel<<<dim3(tcrv::kXcds, o.slots_y, o.slots_z), dim3(waves * 64), 0, as_stream(stream)>>>(
        o.units, o.inv, nb, vx, vy, ngw, nga, s, bs, vec_out);
  };
  if (rows64)
    run(tcrv::gemm_repack_mid<2, 2>, 4);
  else
    run(tcrv::gemm_repack_mid<4, 2>, 8);
  return launch_status();
}

}  // namespace tcrv_host
