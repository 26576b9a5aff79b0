// Causal GQA attention of a prefill on MFMA (gfx950).
//
// The reference's prefill is serial: run_manual_one_token once per prompt
// token (10_validate_full_run_one_token.py:81-135), each call appending one
// K/V row and attending over the cache (common.py:231-298).  Here the n new
// tokens at positions p0 .. p0 + n - 1 go through each layer together; the
// projections are Q4 GEMMs (q4d_gemm.hip), whose q|k|v epilogue also applies
// the per-head q/k RMSNorm and RoPE, appends K/V to the cache and leaves q as
// fp16 [q_head][token][128] with the softmax scale and log2(e) folded in.
//
// prefill_attn_kernel: flash attention forward, causal, one block per (64-query tile, q
// head, sequence).  Four waves: 32 queries x one 32-key half of every 64-key tile each; the
// two halves' softmax states merge once at the end through LDS.
//   S^T = K . Q^T (32x32x16 f16 MFMA; K rows from LDS, Q^T from registers); online softmax
//   per query (exp2); O^T += V^T . P^T, where the S^T accumulator layout is already the
//   B operand layout of P^T (a lane holds 4 + 4 keys of each 16-key step for one query), so
//   P never leaves registers; V^T comes out of the row-major V tile with the transposing LDS
//   read (ds_read_b64_tr_b16: 4 keys of one dim per lane), for the same keys.
// K and V tiles go global -> LDS directly (global_load_lds_dwordx4, one tile ahead, two
// stages): no registers, no LDS store instructions, no transpose in registers, and one
// barrier per tile.  A DMA wave writes 64 consecutive 16-byte slots, so rows are unpadded;
// slot g of row r holds column group g ^ (r & 15) for K and g ^ 4 (r & 3) for V: the 16 rows
// (K) and 4 rows x 64 bytes (V) that a read touches at a time fall on all 64 banks.
//
// What bounds it: one layer of 2048 tokens 31.5 us (44.1 before, when a wave took 16 queries
// over whole tiles: 48 operand reads per 32 half-size MFMAs, 40 % of their cycles bank
// conflicts, and V transposed in registers in front of two barriers); the chain scores ->
// maximum -> exponentials -> P.V of a tile, with one or two waves per SIMD to fill its waits
// (the heavy query tiles run alone for half of their time).  Measured and not kept: the next
// tile's scores issued under this tile's exponentials (252 registers, 39.8 us), two
// accumulator chains for the scores, V read before the exponentials, raised priority around
// the MFMAs (equal or slower), a budget of one or three waves per SIMD (56.8 / 45.1 against
// 45.5 us for a call), MFMA results in accumulator registers (52.4).
#include <math.h>
#include <string.h>

#include <type_traits>

#include "q4d_device.h"
#include "q4d_internal.h"

namespace q4d {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kD = 128;
constexpr int kBQ = 64;  // queries per block
constexpr int kBK = 64;  // keys per tile
constexpr int kStage = 2 * kBK * kD * 2;  // bytes of a stage: K rows, then V rows
constexpr int kOld = kD + 4;              // float row stride of the output tile
constexpr float kRescale = 8.0f;  // log2 headroom of the lazily moved running max
constexpr float kNoMax = -1e30f;  // running max before the first visible key

struct AttnFwd {
  const _Float16* q16;  // [qh][n][128], scaled (F32 false)
  const float* q32;     // [batch][qh][n][128], scaled by qmul here (F32 true)
  float qmul;
  const uint16_t* k;    // per sequence [kvh][max_ctx][128]
  const uint16_t* v;
  _Float16* o16;        // [n][qh * 128]
  float* o32;           // [batch][qh][n][128]
  int n, p0, qh, kvh, max_ctx, batch;
};

// Max / sum of lanes l and l ^ 32, the same value in both: v_permlane32_swap(x, x) returns
// (x of lanes 0-31 in both halves, x of lanes 32-63 in both).  The result elements are copied
// to scalars before the bit casts (a bit cast of an ext-vector element expression reads
// element 0 with this compiler).
template <bool SUM>
__device__ __forceinline__ float halves_reduce(float v) {
  const uint32_t a = __builtin_bit_cast(uint32_t, v);
  const auto r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  const float x0 = __builtin_bit_cast(float, r0), x1 = __builtin_bit_cast(float, r1);
  return SUM ? x0 + x1 : fmaxf(x0, x1);
}

// Lane i of the wave writes 16 bytes from `src` at LDS address lds + 16 i (lds wave-uniform,
// through M0).  Issued by inline asm and ordered by the kernel's own wait and barrier, as in
// the pipelined GEMM (q4d_gemm.hip).
__device__ __forceinline__ void attn_dma16(const void* src, void* lds) {
  const uint32_t off = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(off), "v"(src) : "memory");
}

// 4 keys of one dim: lane i of each 16 addresses 4 dims (8 bytes) of key i / 4 and receives
// dim i of the four keys.
__device__ __forceinline__ h4 read_tr4(const char* p) {
  return __builtin_bit_cast(
      h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p)));
}

// Register budget of two waves per SIMD: the LDS holds two blocks of four waves per CU.
template <bool F32>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void prefill_attn_kernel(const AttnFwd a) {
  __shared__ __attribute__((aligned(16))) char lds[2 * kStage];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int qg = w >> 1, kh = w & 1;  // 32-query group, 32-key half

  // Block order.  Linear block b runs on XCD b % 8 (each XCD has its own L2), and an XCD's
  // blocks go round robin over its 32 CUs, two to a CU.  With 8 | heads each XCD takes
  // consecutive q heads (their kv heads' K/V stay in that L2), heaviest query tiles first;
  // the second block of each CU in the opposite order, so the first round's pairs are
  // complementary, and the rest as CUs become free.
  const int gx = gridDim.x, gy = gridDim.y, total = gx * gy * (int)gridDim.z;
  const int lin = (int)blockIdx.x + gx * ((int)blockIdx.y + gy * (int)blockIdx.z);
  const bool split = gy % 8 == 0;
  const int heads = split ? gy / 8 : gy, per = split ? total / 8 : total;
  int rank = split ? lin >> 3 : lin;
  constexpr int kCus = 32;  // per XCD
  if (split && rank >= kCus && rank < 2 * kCus) {
    const int end = min(2 * kCus, per);
    rank = kCus + end - 1 - rank;
  }
  const int other = heads * a.batch;
  const int qt = gx - 1 - rank / other, hb = rank % other;
  const int h = (split ? (lin & 7) * heads : 0) + hb % heads, bt = hb / heads;

  const int j = h / (a.qh / a.kvh);
  const int i0 = qt * kBQ, q_lo = i0 + 32 * qg;
  const int kend = a.p0 + min(a.n, i0 + kBQ);  // keys [0, kend) can be attended by the block
  const int ntiles = (kend + kBK - 1) / kBK;
  const size_t plane = ((size_t)bt * a.kvh + j) * a.max_ctx * kD;
  const uint16_t* kb = a.k + plane;
  const uint16_t* vb = a.v + plane;

  // Q^T operand: lane (query q_lo + l % 32, half l / 32) holds dims 16 s + 8 half .. +7
  const int qc = lane & 31, hf = lane >> 5;
  const int my_q = q_lo + qc, my_pos = a.p0 + my_q;
  h8 qop[8];
  {
    const int qrow = min(my_q, a.n - 1);
    if constexpr (F32) {
      const float* qp = a.q32 + (((size_t)bt * a.qh + h) * a.n + qrow) * kD + 8 * hf;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const f32x4 x0 = *reinterpret_cast<const f32x4*>(qp + 16 * s), x1 = *reinterpret_cast<const f32x4*>(qp + 16 * s + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          qop[s][e] = (_Float16)(x0[e] * a.qmul);
          qop[s][e + 4] = (_Float16)(x1[e] * a.qmul);
        }
      }
    } else {
      const _Float16* qp = a.q16 + ((size_t)h * a.n + qrow) * kD + 8 * hf;
#pragma unroll
      for (int s = 0; s < 8; ++s) qop[s] = *reinterpret_cast<const h8*>(qp + 16 * s);
    }
  }

  // DMA of a tile: wave w brings rows 16 w .. 16 w + 15 of K and V, four per instruction;
  // lane l fills slot l % 16 of row l / 16.  Rows past the end read the last one (masked).
  const int drow = lane >> 4, dslot = lane & 15;
  const auto issue = [&](int kt, int st) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * w + 4 * i + drow;
      const size_t key = min(kt * kBK + row, kend - 1);
      attn_dma16(kb + key * kD + ((dslot ^ (row & 15)) << 3), lds + st * kStage + (16 * w + 4 * i) * (kD * 2));
      attn_dma16(vb + key * kD + ((dslot ^ (4 * (row & 3))) << 3),
                 lds + st * kStage + kStage / 2 + (16 * w + 4 * i) * (kD * 2));
    }
  };

  // LDS offsets of this lane's operands.  K: row 32 kh + l % 32, column group 2 s + half.
  // V: 16-lane group (dim block l / 16 % 2, half), key 4 half + l % 16 / 4 (+ 16 per step,
  // + 8 for the second four), dims 32 dt + 16 block + 4 (l % 4).
  uint32_t ko[8], vo[4];
#pragma unroll
  for (int s = 0; s < 8; ++s) ko[s] = (32 * kh + qc) * (kD * 2) + (((2 * s + hf) ^ (qc & 15)) << 4);
  {
    const int i = lane & 15, key = 4 * hf + (i >> 2), db = (lane >> 4) & 1;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      vo[dt] = kStage / 2 + (32 * kh + key) * (kD * 2) + (((4 * dt + 2 * db + ((i >> 1) & 1)) ^ (4 * (key & 3))) << 4) + 8 * (i & 1);
  }

  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_run = kNoMax, l_run = 0.f;  // per query; l of this lane's keys only

  issue(0, 0);
  for (int kt = 0; kt < ntiles; ++kt) {
    // this wave's part of tile kt has landed, and after the barrier everybody's; everybody
    // is done reading the other stage
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) expcnt(7) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + 1 < ntiles) issue(kt + 1, (kt + 1) & 1);
    const char* stage = lds + (kt & 1) * kStage;
    const int key0 = kt * kBK + 32 * kh;
    if (key0 > a.p0 + q_lo + 31 || key0 >= kend) continue;  // no key of the half is visible to the wave

    f32x16 st;
#pragma unroll
    for (int r = 0; r < 16; ++r) st[r] = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const h8 kop = *reinterpret_cast<const h8*>(stage + ko[s]);
      st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kop, qop[s], st, 0, 0, 0);
    }
    // lane holds keys key0 + 8 (r / 4) + 4 half + r % 4 for query my_pos: causal / range mask
    // only where the half reaches past the wave's first query or past kend
    if (key0 + 31 > a.p0 + q_lo || key0 + 32 > kend) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = key0 + 8 * (r >> 2) + 4 * hf + (r & 3);
        if (key > my_pos || key >= kend) st[r] = -INFINITY;
      }
    }
    float tmax = st[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) tmax = fmaxf(tmax, st[r]);
    tmax = halves_reduce<false>(tmax);
    // Lazy rescaling: the running max moves only when a score exceeds it by more than
    // kRescale (log2 units), so P = 2^(s - m_run) stays below 2^kRescale (far inside fp16's
    // range) and the O / l rescale is skipped for the wave unless some query needs it.  The
    // first visible key always moves it.
    const bool move = tmax > m_run + kRescale;
    if (__builtin_amdgcn_ballot_w64(move)) {
      const float m_new = move ? tmax : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
    }
    h8 p[2];
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float e = __builtin_amdgcn_exp2f(st[r] - m_run);
      psum += e;
      p[r >> 3][r & 7] = (_Float16)e;
    }
    l_run += psum;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const h4 v0 = read_tr4(stage + vo[dt] + 16 * s * (kD * 2));
        const h4 v1 = read_tr4(stage + vo[dt] + (16 * s + 8) * (kD * 2));
        const h8 vop = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vop, p[s], o[dt], 0, 0, 0);
      }
  }

  // ---- merge the two key halves, normalise, store whole rows ------------------------------
  // lane holds O^T[d = 32 dt + 8 (r / 4) + 4 half + r % 4][query my_q]
  l_run = halves_reduce<true>(l_run);
  float* mo = reinterpret_cast<float*>(lds) + qg * (64 * 64 + 128);  // [64 registers][64 lanes], m, l
  __syncthreads();
  if (kh == 1) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) mo[(16 * dt + r) * 64 + lane] = o[dt][r];
    mo[64 * 64 + lane] = m_run;
    mo[64 * 64 + 64 + lane] = l_run;
  }
  __syncthreads();
  if (kh == 0) {
    const float m1 = mo[64 * 64 + lane], l1 = mo[64 * 64 + 64 + lane];
    const float mx = fmaxf(m_run, m1);
    const float a0 = __builtin_amdgcn_exp2f(m_run - mx), a1 = __builtin_amdgcn_exp2f(m1 - mx);
    const float inv = 1.0f / fmaf(l1, a1, l_run * a0);
    const float f0 = a0 * inv, f1 = a1 * inv;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = fmaf(mo[(16 * dt + r) * 64 + lane], f1, o[dt][r] * f0);
  }
  __syncthreads();
  float* T = reinterpret_cast<float*>(lds);  // [64 queries][kOld]
  if (kh == 0) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(T + (32 * qg + qc) * kOld + 32 * dt + 8 * q + 4 * hf) =
            f32x4{o[dt][4 * q], o[dt][4 * q + 1], o[dt][4 * q + 2], o[dt][4 * q + 3]};
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kBQ * kD / 4 / 256; ++i) {
    const int c = t + 256 * i, row = c >> 5, d = (c & 31) * 4, tok = i0 + row;
    if (tok >= a.n) continue;
    const f32x4 x = *reinterpret_cast<const f32x4*>(T + row * kOld + d);
    if constexpr (F32) {
      *reinterpret_cast<f32x4*>(a.o32 + (((size_t)bt * a.qh + h) * a.n + tok) * kD + d) = x;
    } else {
      h4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = (_Float16)x[e];
      *reinterpret_cast<h4*>(a.o16 + (size_t)tok * a.qh * kD + (size_t)h * kD + d) = y;
    }
  }
}

}  // namespace

int launch_prefill_attention(const PrefillArgs& a, hipStream_t st) {
  AttnFwd f;
  memset(&f, 0, sizeof(f));
  f.q16 = a.q16;
  f.k = a.kcache;
  f.v = a.vcache;
  f.o16 = a.out;
  f.n = a.n; f.p0 = a.p0; f.qh = a.qh; f.kvh = a.kvh; f.max_ctx = a.max_ctx;
  f.batch = 1;
  hipLaunchKernelGGL(prefill_attn_kernel<false>, dim3((a.n + kBQ - 1) / kBQ, a.qh), dim3(256), 0, st, f);
  return check_launch();
}

// ---- the causal-attention primitive (manual_causal_attention, common.py:201-216) -----
// k and v are rounded to fp16 planes of max_ctx = seq positions in one launch; the attention
// kernel reads the fp32 q itself (scaled by scaling * log2 e and rounded, as the prefill's
// q|k|v epilogue leaves it) and writes the fp32 output, for every sequence at once.
namespace {

__global__ __launch_bounds__(256) void kv_to_f16_kernel(const float* k, const float* v, _Float16* k16, _Float16* v16,
                                                        long long n8) {
  const float* x = blockIdx.y ? v : k;
  _Float16* y = blockIdx.y ? v16 : k16;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n8; i += (long long)gridDim.x * blockDim.x) {
    const f32x4 v0 = reinterpret_cast<const f32x4*>(x)[2 * i], v1 = reinterpret_cast<const f32x4*>(x)[2 * i + 1];
    h8 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = (_Float16)v0[e];
      h[e + 4] = (_Float16)v1[e];
    }
    reinterpret_cast<h8*>(y)[i] = h;
  }
}

}  // namespace

size_t causal_attention_ws_bytes(int batch, int kvh, int seq) {
  return 2 * align_up((size_t)batch * kvh * seq * kD * 2, 256);  // the fp16 k and v planes
}

int launch_causal_attention(const float* q, const float* k, const float* v, float* out, int batch, int qh,
                            int kvh, int seq, float scaling, void* ws, hipStream_t st) {
  const size_t kvn = (size_t)batch * kvh * seq * kD;
  _Float16* k16 = static_cast<_Float16*>(ws);
  _Float16* v16 = reinterpret_cast<_Float16*>(static_cast<char*>(ws) + causal_attention_ws_bytes(batch, kvh, seq) / 2);
  const long long n8 = (long long)(kvn / 8), blocks = (n8 + 255) / 256;
  hipLaunchKernelGGL(kv_to_f16_kernel, dim3((unsigned)(blocks < 8192 ? blocks : 8192), 2), dim3(256), 0, st, k, v, k16,
                     v16, n8);
  int rc = check_launch();
  if (rc) return rc;
  AttnFwd f;
  memset(&f, 0, sizeof(f));
  f.q32 = q;
  f.qmul = scaling * 1.4426950408889634f;
  f.k = reinterpret_cast<const uint16_t*>(k16);
  f.v = reinterpret_cast<const uint16_t*>(v16);
  f.o32 = out;
  f.n = seq; f.p0 = 0; f.qh = qh; f.kvh = kvh; f.max_ctx = seq;
  // as many sequences per launch as blockIdx.z and an int block number hold
  const long long tiles = (long long)((seq + kBQ - 1) / kBQ) * qh;
  const int most = (int)max(1LL, min(65535LL, (1LL << 30) / tiles));
  for (int b = 0; b < batch; b += most) {
    f.batch = min(most, batch - b);
    f.q32 = q + (size_t)b * qh * seq * kD;
    f.o32 = out + (size_t)b * qh * seq * kD;
    f.k = reinterpret_cast<const uint16_t*>(k16 + (size_t)b * kvh * seq * kD);
    f.v = reinterpret_cast<const uint16_t*>(v16 + (size_t)b * kvh * seq * kD);
    hipLaunchKernelGGL(prefill_attn_kernel<true>, dim3((seq + kBQ - 1) / kBQ, qh, f.batch), dim3(256), 0, st, f);
    if ((rc = check_launch())) return rc;
  }
  return Q4D_OK;
}

}  // namespace q4d
