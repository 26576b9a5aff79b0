"""A host shim over the library's internal launchers and rules (csrc/q4d_internal.h), for tests of
kernels and rules that no public call reaches by itself.  Compiled from the text below when first
asked for; it holds no device code."""

import ctypes
import subprocess
import tempfile
from functools import lru_cache
from pathlib import Path

from llm_accelerator_amd import _lib

ROOT = Path(__file__).resolve().parents[1]
ROCM = Path("/opt/rocm")

SOURCE = r"""
#include <string.h>
#include "q4d_internal.h"
using namespace q4d;
extern "C" {
// out: mt, nt, k12
void shim_rows_tile(int M, int N, int K, int count, int* out) {
  const RowsTile t = rows_tile(M, N, K, count);
  out[0] = t.mt; out[1] = t.nt; out[2] = t.k12;
}
// an output projection of a short prefill
int shim_chain_resid(int M, int N, int K, int ksplit) {
  alignas(16) static float memory[4];  // never read
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.M = M; a.N = N; a.K = K; a.ksplit = ksplit;
  a.nseg = 1;
  a.seg_end[0] = N;
  a.s[0] = reinterpret_cast<const uint16_t*>(memory);
  a.part = memory;
  a.part_cap = (size_t)1 << 40;
  return chain_applies(a, EP_RESID, false);
}
// q4d_linear's and q4d_gemm's choice of the rows kernel
int shim_rows_linear(int batch, int rows, int K, int xf32) { return rows_linear(batch, rows, K, xf32); }
int shim_rows_apply(int M, int N, int K, int ep) {
  alignas(16) static float memory[4];  // never read
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.M = M; a.N = a.ldy = a.seg_end[0] = N; a.K = K;
  a.nseg = a.rows = 1;
  a.s[0] = reinterpret_cast<const uint16_t*>(memory);
  return rows_apply(a, ep, false);
}
// launch_gemm as the batched decode step calls it (the skinny kernel at up to 64 rows)
int shim_skinny_gemm(const q4d_matrix_t* w, int nseg, const uint16_t* x, int M, void* y, int ep, const float* resid,
                     float* part, size_t part_floats, int x_tiled, int y_tiled, int* ksplit_used, void* stream) {
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  int rows = 0;
  for (int i = 0; i < nseg; ++i) {
    a.w[i] = w[i].w;
    a.s[i] = w[i].s;
    a.seg_end[i] = rows += w[i].rows;
  }
  a.nseg = nseg;
  a.N = ep == EP_SWIGLU ? w[0].rows : rows;
  a.K = w[0].cols;
  a.M = M;
  a.x = x;
  a.y = y;
  a.ldy = a.N;
  a.resid = resid;
  a.part = part;
  a.part_cap = part_floats;
  a.skinny = 1;
  a.x_tiled = x_tiled;
  a.y_tiled = y_tiled;
  a.ksplit_used = ksplit_used;
  return launch_gemm(a, ep, ep == EP_SWIGLU, static_cast<hipStream_t>(stream));
}
}
"""

EP_F16, EP_F32, EP_RESID, EP_SWIGLU = 0, 1, 2, 3


@lru_cache(maxsize=None)
def load() -> ctypes.CDLL:
    _lib.load()
    with tempfile.TemporaryDirectory() as d:
        src, so = Path(d) / "shim.cpp", Path(d) / "shim.so"
        src.write_text(SOURCE)
        subprocess.run([str(ROCM / "llvm/bin/clang++"), "-shared", "-fPIC", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
                        f"-I{ROOT / 'llm_accelerator_amd' / 'csrc'}", f"-I{ROCM / 'include'}", str(src),
                        str(_lib.LIB_PATH), "-o", str(so)], check=True)
        lib = ctypes.CDLL(str(so))
    i, p = ctypes.c_int, ctypes.c_void_p
    lib.shim_rows_tile.argtypes, lib.shim_rows_tile.restype = [i, i, i, i, p], None
    lib.shim_chain_resid.argtypes, lib.shim_chain_resid.restype = [i, i, i, i], i
    lib.shim_rows_linear.argtypes, lib.shim_rows_linear.restype = [i, i, i, i], i
    lib.shim_rows_apply.argtypes, lib.shim_rows_apply.restype = [i, i, i, i], i
    lib.shim_skinny_gemm.argtypes = [p, i, p, i, p, i, p, p, ctypes.c_size_t, i, i, p, p]
    lib.shim_skinny_gemm.restype = i
    return lib
