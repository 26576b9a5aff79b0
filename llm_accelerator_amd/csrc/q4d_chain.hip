// Q4 GEMMs of a short prefill on MFMA (gfx950): the sums of q4d_gemm.hip's tiled kernels,
// bit for bit, without their chain of staged K steps.
//
// A short prompt gives the tiled kernels few blocks (75 tokens: 16-48 on 256 CUs), each
// walking K in 64-column steps with a barrier and a dequantised LDS tile per step: 15-22 us
// per GEMM for 1-3 MB of weights.  Here every wave computes 16 weight rows x 16 MT tokens
// over the whole K (of its split) by itself: its codes and scales go to registers with all
// loads issued at entry, the block's 16 MT token rows go to LDS once, and after that one
// barrier the wave unpacks and multiplies without waiting for anybody.  The MFMA sequence
// per output (32 columns a step, in order, from zero) is the tiled kernels', so a prompt in
// chunks equals one call whichever kernel a chunk's size picks.
//
// The 16 NW columns of a block meet in LDS for the epilogue, which then stores whole rows: a
// head's RMSNorm + RoPE (128 columns are one head), SwiGLU (waves 0-3 gate, 4-7 up rows), or
// the raw partial tile of a K split.
//
// What bounds it: the launch, one memory round trip and the unpacking VALU work of the two
// waves on each SIMD (75 tokens, kernel times: q|k|v 8.0 us, was 17.0; gate / up 7.7, 15.4;
// o_proj and down 5.7 on average, 16.0 and 21.9; the 28 layers and LM head 2385 -> 1131 us).
#include <type_traits>

#include "q4d_internal.h"
#include "q4d_mfma_dev.h"

namespace q4d {

namespace {

constexpr int kChUnit = 128;  // K columns per code load (16 bytes per lane of each 16 x 128 tile)

// NU units per split; NW waves per block, 16 weight rows each.
template <int EP, int MT, int NW, int NU>
__global__ __launch_bounds__(NW * 64) void q4_chain_kernel(const GemmArgs a) {
  constexpr bool PAIR = EP == EP_SWIGLU;
  static_assert(EP == EP_RESID || NW == 8, "a head or a gate / up tile is 128 columns");
  constexpr int NT = NW * 64, KS = NU * kChUnit, LD = KS + 16;  // row stride 32 B past a multiple of 64: no conflicts
  constexpr int CPR = KS / 8, XL = 16 * MT * CPR / NT;          // 16-byte chunks per token row, loads per thread
  constexpr int TLD = 16 * NW + 4;
  static_assert(16 * MT * CPR % NT == 0, "chunks per thread");
  constexpr int kX = 16 * MT * LD * 2, kT = 16 * MT * TLD * 4;
  __shared__ __attribute__((aligned(16))) char lds[kX > kT ? kX : kT];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nl = lane & 15, G = lane >> 4;
  const int nblk = blockIdx.x, m0 = blockIdx.y * 16 * MT, k0 = blockIdx.z * KS;

  // token rows (past the end: the last one, not stored), then this wave's codes and scales
  u32x4 x[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int c = t + NT * i, m = min(m0 + c / CPR, a.M - 1);
    x[i] = *reinterpret_cast<const u32x4*>(a.x + (size_t)m * a.K + k0 + (c % CPR) * 8);
  }
  const uint8_t* wb;
  const uint16_t* sb;
  int grow;
  if (PAIR) {
    grow = nblk * 64 + 16 * (w & 3) + nl;
    wb = w >= 4 ? a.w[1] : a.w[0];
    sb = w >= 4 ? a.s[1] : a.s[0];
  } else {
    const int r = nblk * 16 * NW + 16 * w;  // segment ends are multiples of 128
    if (r < a.seg_end[0]) {
      grow = r + nl; wb = a.w[0]; sb = a.s[0];
    } else if (r < a.seg_end[1]) {
      grow = r + nl - a.seg_end[0]; wb = a.w[1]; sb = a.s[1];
    } else {
      grow = r + nl - a.seg_end[1]; wb = a.w[2]; sb = a.s[2];
    }
  }
  wb += (size_t)grow * (a.K / 2) + k0 / 2 + 16 * G;
  sb += (size_t)grow * (a.K / 64) + k0 / 64;
  u32x4 c[NU];
  uint32_t sc[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    c[u] = *reinterpret_cast<const u32x4*>(wb + u * (kChUnit / 2));
    sc[u] = *reinterpret_cast<const uint32_t*>(sb + 2 * u);
  }
  __builtin_amdgcn_sched_barrier(0);  // every load goes out before the first wait
  _Float16* xs = reinterpret_cast<_Float16*>(lds);
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int q = t + NT * i;
    *reinterpret_cast<u32x4*>(xs + (q / CPR) * LD + (q % CPR) * 8) = to_pairs(x[i]);
  }
  block_sync_lds();

  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  const auto units = [&](auto wide) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      uint32_t d[4] = {c[u][0], c[u][1], c[u][2], c[u][3]};
      rows_transpose4(d);
      const W16Scale lo = w16_scale(sc[u] & 0xFFFFu), hi = w16_scale(sc[u] >> 16);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const h8 q = __builtin_bit_cast(h8, dequant8_pairs<decltype(wide)::value>(d[s], s < 2 ? lo : hi));
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const h8 xv = *reinterpret_cast<const h8*>(xs + (16 * i + nl) * LD + kChUnit * u + 32 * s + 8 * G);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, q, acc[i], 0, 0, 0);
        }
      }
    }
  };
  uint32_t most = 0;
#pragma unroll
  for (int u = 0; u < NU; ++u) most = max(most, max(sc[u] & 0xFFFFu, sc[u] >> 16));
  if (scale_wide(most))
    units(std::true_type{});
  else
    units(std::false_type{});

  // lane holds token rows 16 i + 4G + r of column 16 w + l % 16
  __syncthreads();
  float* T = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) T[(16 * i + 4 * G + r) * TLD + 16 * w + nl] = acc[i][r];
  __syncthreads();
  if constexpr (EP == EP_RESID) {  // raw tile of the split: [z][m][n]
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = 16 * i + t / (4 * NW), cq = 4 * (t % (4 * NW)), m = m0 + row;
      if (m < a.M)
        *reinterpret_cast<f32x4*>(a.part + ((size_t)blockIdx.z * a.M + m) * a.N + nblk * 16 * NW + cq) =
            *reinterpret_cast<const f32x4*>(T + row * TLD + cq);
    }
  } else if constexpr (EP == EP_SWIGLU) {
    const int cp = 2 * (t & 31);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = 16 * i + (t >> 5), m = m0 + row;
      if (m >= a.M) continue;
      const float* g = T + row * TLD + cp;
      const h2 v = make_h2(swiglu(g[0], g[64]), swiglu(g[1], g[65]));
      *reinterpret_cast<h2*>(static_cast<_Float16*>(a.y) + (size_t)m * a.ldy + nblk * 64 + cp) = v;
    }
  } else {
    // one head per block: 32 lanes per token row, as rope_epilogue deals a row's columns
    const PrefillArgs& R = a.rope;
    const int h = nblk, cl = t & 15, wn = (t >> 4) & 1;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = 16 * i + (t >> 5), tok = m0 + row;
      const float* p = T + row * TLD + 32 * wn + cl;
      float v[4] = {p[0], p[16], p[64], p[80]};
      if (h < R.qh + R.kvh) {
        float ss = rope_half_ss(v[0], v[1], v[2], v[3]);
        ss += shfl_xor_f(ss, 16);
        const float inv = rope_inv(ss, R.eps);
        const float* gam = h < R.qh ? R.q_gamma : R.k_gamma;
        const size_t tb = (size_t)(R.p0 + min(tok, a.M - 1)) * 64 + 32 * wn + cl;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int d = 32 * wn + 16 * j + cl;
          rope_pair(v[j], v[j + 2], inv, gam[d], gam[d + 64], R.rope_cos[tb + 16 * j], R.rope_sin[tb + 16 * j]);
        }
      }
      if (tok >= a.M) continue;
      _Float16* dst;
      _Float16 o[4] = {(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
      if (h < R.qh) {
        dst = R.q16 + ((size_t)h * R.n + tok) * 128;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          o[j] = rope_q_lo(v[j], R.qscale);
          o[j + 2] = rope_q_hi(v[j + 2], R.qscale);
        }
      } else if (h < R.qh + R.kvh) {
        dst = reinterpret_cast<_Float16*>(R.kcache) + ((size_t)(h - R.qh) * R.max_ctx + R.p0 + tok) * 128;
      } else {
        dst = reinterpret_cast<_Float16*>(R.vcache) + ((size_t)(h - R.qh - R.kvh) * R.max_ctx + R.p0 + tok) * 128;
      }
      dst += 32 * wn + cl;
      dst[0] = o[0];
      dst[16] = o[1];
      dst[64] = o[2];
      dst[80] = o[3];
    }
  }
}

template <int EP, int NW, int NU>
int launch_mt(const GemmArgs& a, hipStream_t st) {
  const int nb = EP == EP_SWIGLU ? a.N / 64 : a.N / (16 * NW), z = EP == EP_RESID ? a.ksplit : 1;
  const auto blocks = [&](int mt) { return (long)nb * z * ((a.M + 16 * mt - 1) / (16 * mt)); };
  const auto go = [&](auto kernel, int mt) {
    hipLaunchKernelGGL(kernel, dim3(nb, (a.M + 16 * mt - 1) / (16 * mt), z), dim3(64 * NW), 0, st, a);
    return check_launch();
  };
  // more tokens per block while most CUs keep one (each unpacked weight serves MT tiles):
  // 256 tokens 1.63 ms at 200 blocks, 1.69 at 120, 1.76 at 320
  constexpr long kMinBlocks = 200;
  constexpr int kWide = NU * 4 <= 40 ? 4 : 2;  // 64 tokens x 1536 columns do not fit the LDS
  if (kWide == 4 && blocks(4) >= kMinBlocks) return go(q4_chain_kernel<EP, kWide, NW, NU>, kWide);
  if (blocks(2) >= kMinBlocks) return go(q4_chain_kernel<EP, 2, NW, NU>, 2);
  return go(q4_chain_kernel<EP, 1, NW, NU>, 1);
}

}  // namespace

bool chain_applies(const GemmArgs& a, int ep, bool pair) {
  // tokens up to which it wins, kernel times against the tiled kernels': q|k|v 10.7 / 13.6 us
  // against 17.3 / 18.0 at 256 / 512 tokens, o_proj 8.9 / 9.2 against 16.7 / 18.2, down
  // 8.9 / 16.8 against 22.7 / 23.3, gate / up 14.7 / 21.3 against 16.0 / 16.7
  if (a.M > (ep == EP_SWIGLU ? 256 : 512) || (ep == EP_SWIGLU) != pair) return false;
  for (int i = 0; i < a.nseg; ++i)
    if (!aligned(a.s[i], 4)) return false;
  if (ep == EP_ROPE || ep == EP_SWIGLU)
    return a.K == 1024 && !a.part && a.ksplit <= 1 && (ep == EP_ROPE || (a.ldy % 2 == 0 && aligned(a.y, 4)));
  if (ep != EP_RESID || a.nseg != 1 || a.ksplit < 2 || !a.part || !aligned(a.part, 16) ||
      (size_t)a.ksplit * a.M * a.N > a.part_cap || a.K % a.ksplit)
    return false;
  const int ks = a.K / a.ksplit;
  return ks == 512 || ks == 1024 || ks == 1536;
}

int launch_chain(const GemmArgs& a, int ep, bool pair, hipStream_t st) {
  if (!chain_applies(a, ep, pair)) return Q4D_ERR_SHAPE;
  if (ep == EP_ROPE) return launch_mt<EP_ROPE, 8, 8>(a, st);
  if (ep == EP_SWIGLU) return launch_mt<EP_SWIGLU, 8, 8>(a, st);
  switch (a.K / a.ksplit) {
    case 512: return launch_mt<EP_RESID, 4, 4>(a, st);
    case 1024: return launch_mt<EP_RESID, 4, 8>(a, st);
    default: return launch_mt<EP_RESID, 4, 12>(a, st);
  }
}

}  // namespace q4d
