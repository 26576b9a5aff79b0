// Q4 linear over several activation rows on MFMA, at the GEMV's precision (gfx950).
//
//   y[m, n] = sum_g scale[n, g] * sum_{k in group g} q[n, k] x[m, k]      (4 rows and more: rows_linear)
//
// The GEMV (q4d_gemv.hip) reads and unpacks every weight again for each activation row: at
// 211 rows of a 1024 x 3072 matrix its VALU work took 142 us.  Here 16 rows share each
// unpacked weight.  The arithmetic keeps the GEMV's precision: the int4 codes enter the MFMA
// as exact fp16 integers, fp32 activations as an fp16 hi + fp16 lo pair (~22 significant
// bits, two MFMAs; fp16 activations and activation precision 1 take one), products are
// exact, a 64-column group is summed in fp32 by its own MFMA accumulator and multiplied by
// its Q2.14 scale in fp32.
//
// Work split: a block owns 16 MT activation rows x 16 NT weight rows; its waves split K in
// units of 128 columns (two scale groups) and their partial tiles are summed through LDS in
// wave order, so the result is deterministic.  A unit's activations are read as whole
// 512-byte row pieces, split into hi / lo and laid out for the MFMA in LDS that belongs to
// the wave alone (no barrier); read straight into the MFMA operand layout, each load
// instruction would touch 64 separate cache lines.  The codes go to registers: 16 bytes per
// lane, transposed across the four lane rows as in the skinny GEMM (q4d_gemm.hip).
//
// What bounds it: a few rows, the launch and one memory round trip (16 rows of 3072 x 1024
// fp32: 3.1 us, 9.4 as 16 GEMVs); many, the unpacking and splitting VALU work per MFMA and
// the activations' re-reads from L2 (211 rows of 1024 x 3072: 8.6 us, was 142; 1024 rows of
// 3072 x 1024: 32 us, was 466).
#include <type_traits>

#include "q4d_internal.h"
#include "q4d_mfma_dev.h"

namespace q4d {

namespace {

constexpr int kRwUnit = 128;           // K columns per wave and step
constexpr int kRwLd = kRwUnit + 16;    // LDS row stride in fp16: 288 B, conflict-free MFMA operand reads
constexpr int kRwRed = 17;             // LDS row stride (floats) of the partial tiles

// Up to kRowsGroupMax matrices of one shape in a launch (matrix blockIdx.z); a's pointers unused.
constexpr int kRowsGroupMax = 64;
struct RowsGroupArgs {
  RowsArgs a;
  const uint8_t* w[kRowsGroupMax];
  const uint16_t* s[kRowsGroupMax];
  const void* x[kRowsGroupMax];
  void* y[kRowsGroupMax];
};

__device__ __forceinline__ RowsArgs rows_of(const RowsArgs& a) { return a; }
__device__ __forceinline__ RowsArgs rows_of(const RowsGroupArgs& g) {
  const int z = blockIdx.z;
  return RowsArgs{g.w[z], g.s[z], g.x[z], g.y[z], nullptr, g.a.M, g.a.N, g.a.K};
}

// XF32: fp32 activations (else fp16).  XP: 2 = hi + lo halves, 1 = one fp16 value, 0 = one fp16
// value and the weights rounded to fp16 as q4d_gemm states it (one rounding of code x scale,
// so no scale is applied to the sums).  The block's
// tile is 16 MT activation rows x 16 NT weight rows.  UPW > 0: every wave has UPW units and
// issues all their loads at entry; 0: any number, the next unit's loads in flight.
template <bool XF32, int XP, int EP, int MT, int NT, int NW, int UPW, class Args>
__global__ __launch_bounds__(NW * 64) void rows_kernel(const Args args) {
  const RowsArgs a = rows_of(args);
  static_assert(XF32 ? XP != 0 : XP != 2, "fp16 activations are one value");
  constexpr int kH = XP == 2 ? 2 : 1;
  constexpr int kX = NW * kH * 16 * MT * kRwLd * 2, kR = NW * MT * NT * 16 * kRwRed * 4;
  __shared__ __attribute__((aligned(16))) char lds[kX > kR ? kX : kR];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nl = lane & 15, G = lane >> 4;
  const int n0 = blockIdx.x * 16 * NT, m0 = blockIdx.y * 16 * MT;
  const int nu = a.K / kRwUnit;
  const int u0 = w * nu / NW, u1 = (w + 1) * nu / NW;
  _Float16* xs = reinterpret_cast<_Float16*>(lds) + (size_t)w * kH * 16 * MT * kRwLd;

  // rows past the end read the last one; their results are not stored
  // (32-bit offsets from the block's first rows: one address register per load)
  const uint8_t* wb = a.w + (size_t)n0 * (a.K / 2);
  const char* sb = reinterpret_cast<const char*>(a.s) + (size_t)n0 * (a.K / 32);
  uint32_t wo[NT], so[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const uint32_t n = min(16 * j + nl, a.N - 1 - n0);
    wo[j] = n * (a.K / 2) + 16 * G;
    so[j] = n * (a.K / 32);
  }
  // activation loads of a unit: 16 lanes per row, 8 columns each (fp32: two 16-byte loads)
  constexpr int XB = XF32 ? 4 : 2, XR = 4 * MT, XL = XR * (XB / 2);
  const int xr = lane >> 4, xc = lane & 15;
  const char* xb = static_cast<const char*>(a.x) + (size_t)m0 * a.K * XB;
  uint32_t xo[XR];
#pragma unroll
  for (int i = 0; i < XR; ++i) xo[i] = (uint32_t)min(4 * i + xr, a.M - 1 - m0) * a.K * XB + 8 * XB * xc;

  // where the wave stores them in LDS.  Other lanes of the wave read them: its LDS operations
  // run in program order, and the empty asm holds the compiler to that order, since it cannot
  // tell an opaque offset apart from any load's.  (A wave barrier with fences does too, but
  // stops the scheduler: 211 fp32 rows of 1024 x 3072 8.6 -> 9.4 us.)
  uint32_t xw = (uint32_t)w * kH * 16 * MT * kRwLd;
  asm("" : "+s"(xw));

  struct Unit {
    u32x4 x[XL];
    u32x4 c[NT];
    uint32_t s[NT];
  } U[UPW > 0 ? UPW : 1];
  auto load_scales = [&](Unit& L, int u) {
#pragma unroll
    for (int j = 0; j < NT; ++j) L.s[j] = *reinterpret_cast<const uint32_t*>(sb + 4 * u + so[j]);
  };
  auto load = [&](Unit& L, int u) {
#pragma unroll
    for (int i = 0; i < XL; ++i)
      L.x[i] = *reinterpret_cast<const u32x4*>(xb + u * (kRwUnit * XB) + xo[i / (XB / 2)] + 16 * (i % (XB / 2)));
#pragma unroll
    for (int j = 0; j < NT; ++j) L.c[j] = *reinterpret_cast<const u32x4*>(wb + u * (kRwUnit / 2) + wo[j]);
  };
  // whether a unit's weights need the general fp16 conversion (a scale code past the fast one)
  auto wide_codes = [&](const Unit& L) {
    uint32_t most = 0;
#pragma unroll
    for (int j = 0; j < NT; ++j) most = max(most, max(L.s[j] & 0xFFFFu, L.s[j] >> 16));
    return most;
  };
  f32x4 tot[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) tot[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto step = [&](Unit& L, int u, auto wide) {
    // activations to LDS in pair order: row 4 i + xr, hi at 0, lo 16 MT rows further
#pragma unroll
    for (int i = 0; i < XR; ++i) {
      u32x4* d = reinterpret_cast<u32x4*>(reinterpret_cast<_Float16*>(lds) + xw + (4 * i + xr) * kRwLd + 8 * xc);
      if constexpr (XF32) {
        u32x4 hw, lw;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint32_t b0 = L.x[2 * i][p], b1 = L.x[2 * i + 1][p];
          const float f0 = __builtin_bit_cast(float, b0), f1 = __builtin_bit_cast(float, b1);
          const h2 h = make_h2((_Float16)f0, (_Float16)f1);
          hw[p] = __builtin_bit_cast(uint32_t, h);
          if constexpr (XP == 2)
            lw[p] = __builtin_bit_cast(uint32_t, make_h2((_Float16)(f0 - (float)h.x), (_Float16)(f1 - (float)h.y)));
        }
        *d = hw;
        if constexpr (XP == 2) d[16 * MT * kRwLd / 8] = lw;
      } else {
        *d = to_pairs(L.x[i]);
      }
    }
    uint32_t d4[NT][4], sc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      sc[j] = L.s[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) d4[j][e] = L.c[j][e];
    }
    if (UPW == 0 && u + 1 < u1) {
      load_scales(L, u + 1);
      load(L, u + 1);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) rows_transpose4(d4[j]);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      W16Scale sh[NT];
      if constexpr (XP == 0) {
#pragma unroll
        for (int j = 0; j < NT; ++j) sh[j] = w16_scale(g ? sc[j] >> 16 : sc[j] & 0xFFFFu);
      }
      f32x4 p[MT][NT];
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) p[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 2 * g; s < 2 * g + 2; ++s) {
        h8 xh[MT], xl[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const _Float16* xp = xs + (16 * i + nl) * kRwLd + 32 * s + 8 * G;
          xh[i] = *reinterpret_cast<const h8*>(xp);
          if constexpr (XP == 2) xl[i] = *reinterpret_cast<const h8*>(xp + 16 * MT * kRwLd);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if constexpr (XP == 0) {
            const h8 q = __builtin_bit_cast(h8, dequant8_pairs<decltype(wide)::value>(d4[j][s], sh[j]));
#pragma unroll
            for (int i = 0; i < MT; ++i)
              tot[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[i], q, tot[i][j], 0, 0, 0);
            continue;
          }
          const h8 q = __builtin_bit_cast(h8, codes8_pairs(d4[j][s]));
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            p[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[i], q, p[i][j], 0, 0, 0);
            if constexpr (XP == 2) p[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[i], q, p[i][j], 0, 0, 0);
          }
        }
      }
      if constexpr (XP == 0) continue;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const float f = 8.0f * scale_q2_14(g ? sc[j] >> 16 : sc[j] & 0xFFFFu);  // the codes are q / 8
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) tot[i][j][r] = fmaf(p[i][j][r], f, tot[i][j][r]);
      }
    }
  };
  constexpr bool kWideOnly = XP == 0 && MT * NT >= 8 && UPW > 1;
  const auto units = [&](auto wide) {
#pragma unroll
    for (int d = 0; d < UPW; ++d) step(U[d], u0 + d, wide);
  };
  if constexpr (UPW > 0) {
    // the scales first: the choice of conversion waits for them alone
#pragma unroll
    for (int d = 0; d < UPW; ++d) load_scales(U[d], u0 + d);
#pragma unroll
    for (int d = 0; d < UPW; ++d) load(U[d], u0 + d);
    uint32_t most = 0;
#pragma unroll
    for (int d = 0; d < UPW; ++d) most = max(most, wide_codes(U[d]));
    // (the largest tile over several units: the general conversion always; two copies of that
    // much code cost more than it saves: 768 x 1024 x 3072 17.4 us, 19.2 with both)
    if (XP == 0 && (kWideOnly || scale_wide(most)))
      units(std::true_type{});
    else if constexpr (!kWideOnly)
      units(std::false_type{});
  } else if (u0 < u1) {
    load_scales(U[0], u0);
    load(U[0], u0);
    for (int u = u0; u < u1; ++u) {
      if (XP == 0 && scale_wide(wide_codes(U[0])))
        step(U[0], u, std::true_type{});
      else
        step(U[0], u, std::false_type{});
    }
  }

  // lane holds activation rows 16 i + 4G + r of weight row 16 j + l % 16
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[(((w * NT + j) * MT + i) * 16 + 4 * G + r) * kRwRed + nl] = tot[i][j][r];
  __syncthreads();
  for (int o = t; o < MT * NT * 256; o += NW * 64) {
    const int c = o % (16 * NT), j = c >> 4, m = o / (16 * NT);
    if (m0 + m >= a.M || n0 + c >= a.N) continue;
    float v = red[(j * 16 * MT + m) * kRwRed + (c & 15)];
#pragma unroll
    for (int q = 1; q < NW; ++q) v += red[((q * NT + j) * 16 * MT + m) * kRwRed + (c & 15)];
    const size_t oo = (size_t)(m0 + m) * a.N + n0 + c;
    if constexpr (EP == EP_F16)
      static_cast<_Float16*>(a.y)[oo] = (_Float16)v;
    else if constexpr (EP == EP_RESID)
      static_cast<float*>(a.y)[oo] = a.resid[oo] + v;
    else
      static_cast<float*>(a.y)[oo] = v;
  }
}

template <bool XF32, int XP, int EP, int MT, int NT, class Args>
int launch_tile(const Args& args, const RowsArgs& a, int count, bool k12, hipStream_t st) {
  const dim3 grid((a.N + 16 * NT - 1) / (16 * NT), (a.M + 16 * MT - 1) / (16 * MT), count);
  const auto go = [&](auto kernel, int nw) { hipLaunchKernelGGL(kernel, grid, dim3(64 * nw), 0, st, args); };
  // Every unit of a wave in flight where K is one of the projections' widths and the
  // registers hold them (211 x 1024 x 3072, hi + lo: 8.6 us, 11.5 with the next unit only);
  // else the general loop, which q4d_linear needs for one tile and q4d_gemm for other widths.
  constexpr bool kDeep = XP < 2 || MT * NT <= 4, kGroup = std::is_same_v<Args, RowsGroupArgs>;
  constexpr bool k12Tile = MT == 1 && (NT == 1 || kGroup);  // the tiles that rows_tile gives 12 waves
  switch (a.K / kRwUnit) {
    case 8: go(rows_kernel<XF32, XP, EP, MT, NT, 8, 1, Args>, 8); return check_launch();
    case 16:
      if constexpr (kDeep) {
        go(rows_kernel<XF32, XP, EP, MT, NT, 8, 2, Args>, 8);
        return check_launch();
      }
      break;
    case 24:
      if constexpr (k12Tile)
        if (k12) {
          go(rows_kernel<XF32, XP, EP, MT, NT, 12, 2, Args>, 12);
          return check_launch();
        }
      if constexpr (kDeep && NT > 1) {
        go(rows_kernel<XF32, XP, EP, MT, NT, 8, 3, Args>, 8);
        return check_launch();
      }
      break;
    default: break;
  }
  if constexpr (XP != 0 && kDeep) return Q4D_ERR_SHAPE;  // q4d_linear's widths are above
  else go(rows_kernel<XF32, XP, EP, MT, NT, 8, 0, Args>, 8);
  return check_launch();
}

template <bool XF32, int XP, int EP>
int launch_nt(const RowsArgs& a, hipStream_t st) {
  const RowsTile t = rows_tile(a.M, a.N, a.K, 1);
  if (t.mt == 2) return launch_tile<XF32, XP, EP, 2, 4>(a, a, 1, t.k12, st);
  if (t.nt == 4) return launch_tile<XF32, XP, EP, 1, 4>(a, a, 1, t.k12, st);
  if (t.nt == 2) return launch_tile<XF32, XP, EP, 1, 2>(a, a, 1, t.k12, st);
  return launch_tile<XF32, XP, EP, 1, 1>(a, a, 1, t.k12, st);
}

template <bool XF32, int XP, int EP>
int launch_group_nt(const RowsGroupArgs& g, int count, hipStream_t st) {
  const RowsTile t = rows_tile(g.a.M, g.a.N, g.a.K, count);
  if (t.mt == 2) return launch_tile<XF32, XP, EP, 2, 4>(g, g.a, count, t.k12, st);
  if (t.nt == 4) return launch_tile<XF32, XP, EP, 1, 4>(g, g.a, count, t.k12, st);
  return launch_tile<XF32, XP, EP, 1, 1>(g, g.a, count, t.k12, st);
}

}  // namespace

// The largest tile (each split activation serves NT weight tiles, each unpacked weight MT row
// tiles) that still gives most CUs a block: 512 rows of 3072 x 1024, fp16: 24.4 us with
// MT = 1, 16.3 with 2; 64 rows of 2048 x 1024: 3.6 us on 256 blocks, 4.8 on 128.  Two row
// tiles only where there are two: 4 fp32 rows of 151936 x 1024 27.5 us, 48.4 with MT = 2.
// One matrix of K = 3072 on one-tile blocks: 12 waves of two units (4 rows: 5.1 us, 5.5 with 8
// of three), which groups the sums differently from 8 waves.  The matrices of a group count
// together, but each keeps its own launch's waves, so its bits are its own launch's (12 waves
// and two row tiles do not fit the LDS).
RowsTile rows_tile(int M, int N, int K, int count) {
  const int mt = (M + 15) / 16, nt = (N + 15) / 16;
  const auto blocks = [&](int m, int n) { return (long)((mt + m - 1) / m) * ((nt + n - 1) / n); };
  constexpr long kMinBlocks = 192;
  RowsTile t = {1, 1, false};
  if (mt > 1 && blocks(2, 4) >= kMinBlocks) t = {2, 4, false};
  else if (blocks(1, 4) >= kMinBlocks) t = {1, 4, false};
  else if (blocks(1, 2) >= kMinBlocks) t = {1, 2, false};
  else t.k12 = K == 24 * kRwUnit;
  if (count > 1 && t.nt < 4 && blocks(1, 4) * count >= kMinBlocks) t.nt = 4;
  if (count > 1 && !t.k12 && mt > 1 && blocks(2, 4) * count >= kMinBlocks) t = {2, 4, false};
  return t;
}

static int check_rows(const RowsArgs& a, bool xf32, int xp, int ep) {
  if (!a.w || !a.s || !a.x || !a.y || (ep == EP_RESID && !a.resid)) return Q4D_ERR_NULL;
  if (a.M <= 0 || a.M > 16 * 65535 || a.N <= 0 || a.K <= 0 || a.K % kRwUnit) return Q4D_ERR_SHAPE;
  if (!aligned(a.w, 16) || !aligned(a.s, 4) || !aligned(a.x, 16)) return Q4D_ERR_BAD_ADDR;
  if (ep != EP_F16 && ep != EP_F32 && ep != EP_RESID) return Q4D_ERR_SHAPE;
  if (xf32 ? xp < 1 || xp > 2 : xp < 0 || xp > 1) return Q4D_ERR_DTYPE;
  if (ep == EP_RESID && (xf32 || xp)) return Q4D_ERR_DTYPE;
  return Q4D_OK;
}

int launch_rows(const RowsArgs& a, bool xf32, int xp, int ep, hipStream_t st) {
  if (const int rc = check_rows(a, xf32, xp, ep)) return rc;
  if (xf32 && xp == 2) return ep == EP_F16 ? launch_nt<true, 2, EP_F16>(a, st) : launch_nt<true, 2, EP_F32>(a, st);
  if (xf32) return ep == EP_F16 ? launch_nt<true, 1, EP_F16>(a, st) : launch_nt<true, 1, EP_F32>(a, st);
  if (xp == 1) return ep == EP_F16 ? launch_nt<false, 1, EP_F16>(a, st) : launch_nt<false, 1, EP_F32>(a, st);
  switch (ep) {
    case EP_F16: return launch_nt<false, 0, EP_F16>(a, st);
    case EP_F32: return launch_nt<false, 0, EP_F32>(a, st);
    default: return launch_nt<false, 0, EP_RESID>(a, st);
  }
}

// 64 fp32 matrices, us a call (a launch per matrix: 190-350, bound by the host; in brackets the
// grouped GEMV, which reads and unpacks a matrix again for each row): 1024 x 1024 at 8 / 16 / 64
// rows 14.4 / 16.3 / 52 (47 / 88 / 317), 3072 x 1024 at 4 / 16 / 64 rows 33 / 35 / 125 (70 / 239
// / 951), 1024 x 3072 at 4 / 16 / 64 rows 35 / 42 / 137 (98 / 370 / 1467).
int launch_rows_group(int M, int N, int K, const uint8_t* const* w, const uint16_t* const* s, const void* const* x,
                      void* const* y, int count, bool xf32, int xp, int ep, hipStream_t st) {
  if (count <= 0 || !xp || (ep != EP_F16 && ep != EP_F32)) return Q4D_ERR_SHAPE;
  for (int i = 0; i < count; ++i)
    if (const int rc = check_rows(RowsArgs{w[i], s[i], x[i], y[i], nullptr, M, N, K}, xf32, xp, ep)) return rc;
  for (int i0 = 0; i0 < count; i0 += kRowsGroupMax) {
    const int n = count - i0 < kRowsGroupMax ? count - i0 : kRowsGroupMax;
    int rc;
    if (n == 1) {
      rc = launch_rows(RowsArgs{w[i0], s[i0], x[i0], y[i0], nullptr, M, N, K}, xf32, xp, ep, st);
    } else {
      RowsGroupArgs g;
      g.a = RowsArgs{nullptr, nullptr, nullptr, nullptr, nullptr, M, N, K};
      for (int k = 0; k < kRowsGroupMax; ++k) {
        const int i = i0 + (k < n ? k : 0);  // unused slots repeat the first matrix, never read
        g.w[k] = w[i];
        g.s[k] = s[i];
        g.x[k] = x[i];
        g.y[k] = y[i];
      }
      const bool f16 = ep == EP_F16;
      if (xf32 && xp == 2)
        rc = f16 ? launch_group_nt<true, 2, EP_F16>(g, n, st) : launch_group_nt<true, 2, EP_F32>(g, n, st);
      else if (xf32)
        rc = f16 ? launch_group_nt<true, 1, EP_F16>(g, n, st) : launch_group_nt<true, 1, EP_F32>(g, n, st);
      else
        rc = f16 ? launch_group_nt<false, 1, EP_F16>(g, n, st) : launch_group_nt<false, 1, EP_F32>(g, n, st);
    }
    if (rc) return rc;
  }
  return Q4D_OK;
}

}  // namespace q4d
