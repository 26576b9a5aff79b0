// Batched LM head (at most 64 activation rows, K = 1024): final RMSNorm, tied Q4 table on
// MFMA, per-row argmax partials (gfx950).
//
// The tiled GEMM read the table through 1187 blocks that each staged activations and weight
// tiles through LDS behind a barrier per 64 columns (24 rows of 151936 x 1024: 54 us for 83
// MB, plus a launch for the norm).  Here one block per CU stays resident: its waves normalise
// the activation rows once (the arithmetic of rms_norm_kernel) into LDS as fp16, and after
// one barrier every wave streams its own 16-row tiles of the table, the next tile's codes in
// flight while a tile is unpacked (q4d_mfma_dev.h) and multiplied, with the best (score,
// index) per row kept in registers.  Tiles are dealt in pairs of waves (waves 2j and 2j + 1
// of every block take neighbours, then the next pair of waves): the waves that take one more
// are spread over the CUs, and the two 64-byte halves of a line of logits meet in one L2.
//
// What bounds it (24 / 64 rows, a call among others with its argmax rows 35 / 57 us, 65 / 71 on
// the tiled GEMM with the norm's launch): of the time, the activations' LDS reads are about 15 /
// 29 %, the logits' stores 8 / 12 %; without either, the unpacking and the argmax two thirds are
// left at 24 rows.  Two table tiles per read of the activations took as long at 24 rows and 8 %
// longer at 64: fewer, longer steps per wave cost what they save.
//
// The products and their order are the tiled kernel's: fp16 operands (weights rounded once),
// 32 columns per MFMA in order, fp32 accumulation.
#include <math.h>

#include <type_traits>

#include "q4d_internal.h"
#include "q4d_mfma_dev.h"

namespace q4d {

namespace {

constexpr int kLbK = 1024, kLbUnits = kLbK / 128;
constexpr int kLbLd = kLbK + 16;  // LDS row stride in fp16

template <int MT, int NW>
__global__ __launch_bounds__(NW * 64) void lm_batch_kernel(const LmBatchArgs a) {
  __shared__ __attribute__((aligned(16))) _Float16 xs[16 * MT * kLbLd];
  __shared__ float sbest[NW][16 * MT];
  __shared__ int sidx[NW][16 * MT];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nl = lane & 15, G = lane >> 4;
  const int tiles = a.N / 16, stride = (int)gridDim.x * NW;
  int tile = (w >> 1) * 2 * (int)gridDim.x + 2 * (int)blockIdx.x + (w & 1);

  u32x4 c[kLbUnits];
  uint32_t sc[kLbUnits];
  const auto load = [&](int u, int tl) {  // unit u of a tile (past the end: the last tile, not used)
    const size_t row = (size_t)16 * min(tl, tiles - 1) + nl;
    sc[u] = reinterpret_cast<const uint32_t*>(a.s + row * (kLbK / 64))[u];
    c[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(a.w + row * (kLbK / 2) + 16 * G + 64 * u));
  };

  // RMSNorm of rows w, w + NW, ...: lane holds columns 64 j + lane; sums in the order of
  // rms_norm_kernel (four partial sums over every fourth j)
  for (int m = w; m < a.M; m += NW) {
    const float* xr = a.hidden + (size_t)m * kLbK + lane;
    float x[16], g[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = xr[64 * j];
#pragma unroll
    for (int j = 0; j < 16; ++j) g[j] = a.gamma[64 * j + lane];
    float ss[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ss[q] = 0.f;
#pragma unroll
      for (int j = q; j < 16; j += 4) ss[q] = fmaf(x[j], x[j], ss[q]);
      ss[q] = wave_sum(ss[q]);
    }
    const float inv = 1.0f / sqrtf(((ss[0] + ss[1]) + (ss[2] + ss[3])) / (float)kLbK + a.eps);
    // pair order within eight columns: 0 4 1 5 2 6 3 7
    _Float16* d = xs + m * kLbLd + (lane & ~7) + ((lane & 3) << 1) + ((lane >> 2) & 1);
#pragma unroll
    for (int j = 0; j < 16; ++j) d[64 * j] = (_Float16)((x[j] * inv) * g[j]);
  }
#pragma unroll
  for (int u = 0; u < kLbUnits; ++u) load(u, tile);
  block_sync_lds();

  float best[MT][4];
  int bidx[MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      best[i][r] = -INFINITY;
      bidx[i][r] = 0x7fffffff;
    }
  for (; tile < tiles; tile += stride) {
    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    const auto units = [&](auto wide) {
#pragma unroll
      for (int u = 0; u < kLbUnits; ++u) {
        uint32_t d[4] = {c[u][0], c[u][1], c[u][2], c[u][3]};
        rows_transpose4(d);
        const W16Scale lo = w16_scale(sc[u] & 0xFFFFu), hi = w16_scale(sc[u] >> 16);
        load(u, tile + stride);  // the next tile's unit takes its place
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const h8 q = __builtin_bit_cast(h8, dequant8_pairs<decltype(wide)::value>(d[s], s < 2 ? lo : hi));
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            const h8 xv = *reinterpret_cast<const h8*>(xs + (16 * i + nl) * kLbLd + 128 * u + 32 * s + 8 * G);
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, q, acc[i], 0, 0, 0);
          }
        }
      }
    };
    uint32_t most = 0;
#pragma unroll
    for (int u = 0; u < kLbUnits; ++u) most = max(most, max(sc[u] & 0xFFFFu, sc[u] >> 16));
    if (scale_wide(most))
      units(std::true_type{});
    else
      units(std::false_type{});
    // lane holds rows 16 i + 4G + r of table row n
    const int n = 16 * tile + nl;
    const uint32_t lofs = (uint32_t)(4 * G) * a.N + n;  // the rest of the row offset is the wave's
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * i + 4 * G + r;
        const float v = acc[i][r];
        if (a.logits && m < a.M) (a.logits + (size_t)(16 * i + r) * a.N)[lofs] = v;
        if (arg_better(v, n, best[i][r], bidx[i][r])) {
          best[i][r] = v;
          bidx[i][r] = n;
        }
      }
  }

  // the 16 lanes of a row, then the block's waves
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float bs = best[i][r];
      int bi = bidx[i][r];
#pragma unroll
      for (int msk = 8; msk >= 1; msk >>= 1) {
        const float os = shfl_xor_f(bs, msk);
        const int oi = __shfl_xor(bi, msk, kWave);
        if (arg_better(os, oi, bs, bi)) {
          bs = os;
          bi = oi;
        }
      }
      if (nl == 0) {
        sbest[w][16 * i + 4 * G + r] = bs;
        sidx[w][16 * i + 4 * G + r] = bi;
      }
    }
  __syncthreads();
  if (t < 16 * MT && t < a.M) {
    float bs = sbest[0][t];
    int bi = sidx[0][t];
#pragma unroll
    for (int v = 1; v < NW; ++v)
      if (arg_better(sbest[v][t], sidx[v][t], bs, bi)) {
        bs = sbest[v][t];
        bi = sidx[v][t];
      }
    a.part_score[(size_t)t * gridDim.x + blockIdx.x] = bs;
    a.part_idx[(size_t)t * gridDim.x + blockIdx.x] = bi;
  }
}

}  // namespace

bool lm_batch_applies(const LmBatchArgs& a, int K) {
  return K == kLbK && a.M >= 1 && a.M <= 64 && a.N >= 128 && a.N % 128 == 0 && aligned(a.w, 16) && aligned(a.s, 4);
}

int launch_lm_batch(const LmBatchArgs& a, int* nparts, hipStream_t st) {
  if (!a.w || !a.s || !a.hidden || !a.gamma || !a.part_score || !a.part_idx) return Q4D_ERR_NULL;
  if (!lm_batch_applies(a, kLbK)) return Q4D_ERR_SHAPE;
  // one block per CU, fewer where that leaves waves without a tile; the partial buffers hold
  // N / 128 entries per row
  const int blocks = min(device_cus(), a.N / 128);
  *nparts = blocks;
  // waves per block: as many as the registers allow, where that measured faster
  // (24 rows: 4 % slower with 8 than with 16; 16 rows: 7 % slower with 16 than with 8)
  const auto go = [&](auto kernel, int nw) { hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64 * nw), 0, st, a); };
  switch ((a.M + 15) / 16) {
    case 1: go(lm_batch_kernel<1, 8>, 8); break;
    case 2: go(lm_batch_kernel<2, 16>, 16); break;
    case 3: go(lm_batch_kernel<3, 12>, 12); break;
    default: go(lm_batch_kernel<4, 8>, 8); break;
  }
  return check_launch();
}

}  // namespace q4d
