// Shared plumbing of the W4A16 linear kernels: argument bundle and variant registry.
#pragma once

#include "tf_common.h"

namespace tf {

// One W4A16 linear call (w4a16.py:178-232). Pointers are device pointers; x rows and the
// qweight_t rows are 16-byte aligned (checked by tf_w4a16_linear).
struct LinearArgs {
  const uint16_t* x;       // fp16 [m, k], row stride ldx
  int64_t ldx;
  const uint32_t* qw;      // qweight_t [n, k/8]
  const uint16_t* scales;  // fp16 [k/g, n]
  const uint32_t* qz;      // qzeros [k/g, n/8]
  const uint16_t* bias;    // fp16 [n] or nullptr
  uint16_t* out;           // fp16 [m, n], row stride ldo
  int64_t ldo;
  int m;
  int n;
  int k;
  int log2g;               // log2(group_size)
  // Epilogue (TF_EPILOGUE_*): NONE writes y; RESIDUAL writes fp16(residual + fp16(y)) (out may
  // be residual itself, element for element); SILU_MUL writes [m, n / 2]:
  // fp16(fp16(silu(fp16(y[:, j]))) * fp16(y[:, n / 2 + j])).
  int epilogue = TF_EPILOGUE_NONE;
  const uint16_t* residual = nullptr;  // fp16 [m, n], row stride ldr
  int64_t ldr = 0;
  // W4A8 input (tf_w4a8_linear_ex): e4m3fn codes [m, k] with row stride ldx8 bytes, read by
  // the kernels that stage x (others get x converted to fp16 in `x`), and the fp32 row scales
  // of x applied to each row's sum before the bias: y = xscale[m] * sum + bias.
  const uint8_t* x8 = nullptr;
  int64_t ldx8 = 0;
  const float* xscale = nullptr;  // [m] with stride xscale_stride (0: one scale for all rows)
  int64_t xscale_stride = 0;
  // RMSNorm + e4m3 prologue (tf_rmsnorm_fp8_w4a16_linear, decode GEMV stream form only): x holds
  // the rows before the norm; the kernel normalizes each with weight norm_w (fp16 [k], 16-byte
  // aligned) and norm_eps, quantizes it to e4m3 with its dynamic scale and multiplies with
  // fp16(code * scale), the activation rmsnorm_fp8_quant_dq writes for the row.
  const uint16_t* norm_w = nullptr;
  float norm_eps = 0.0f;
  double norm_inv_k = 0.0;  // fp64(1 / k)
};

// Row scale of row m (1 without a W4A8 input, and for rows past m, which are never stored).
__device__ __forceinline__ float row_scale(const LinearArgs& a, int m) {
  return (a.xscale != nullptr && m < a.m) ? a.xscale[(int64_t)m * a.xscale_stride] : 1.0f;
}

// Column mapping of the fused SiLU*mul epilogue for kernels that hold a 16-column group in
// one row of 16 lanes: local column l of the tile at n_base takes the gate row
// n_base / 2 + 8 (l / 16) + l % 8 when l % 16 < 8, else the up row n / 2 + that; lanes l and
// l ^ 8 then hold the gate and up values of one output column. Without the epilogue the
// mapping is the identity n_base + l.
__device__ __forceinline__ int phys_col(const LinearArgs& a, int n_base, int l) {
  if (a.epilogue != TF_EPILOGUE_SILU_MUL) return n_base + l;
  const int j = (n_base >> 1) + ((l >> 4) << 3) + (l & 7);
  return (l & 8) ? (a.n >> 1) + j : j;
}

// Output column of local column l under the SiLU*mul mapping (valid on the gate lanes).
__device__ __forceinline__ int silu_out_col(int n_base, int l) { return (n_base >> 1) + ((l >> 4) << 3) + (l & 7); }

// True when the physical column of local column l holds data (inside N; for SiLU*mul, its
// output column inside n / 2).
__device__ __forceinline__ bool col_valid(const LinearArgs& a, int n_base, int l) {
  if (a.epilogue != TF_EPILOGUE_SILU_MUL) return n_base + l < a.n;
  return silu_out_col(n_base, l) < (a.n >> 1);
}

// The same mapping for the kernels with an instance for it (SILU: a SiLU*mul call without a K
// split; with one they write physical columns and the reduce pairs them).
template <bool SILU>
__device__ __forceinline__ int tile_col(const LinearArgs& a, int n_base, int l) {
  if (!SILU) return n_base + l;
  return ((l & 8) ? a.n >> 1 : 0) + silu_out_col(n_base, l);
}
template <bool SILU>
__device__ __forceinline__ bool tile_col_valid(const LinearArgs& a, int n_base, int l) {
  return SILU ? silu_out_col(n_base, l) < (a.n >> 1) : n_base + l < a.n;
}

__device__ __forceinline__ uint16_t f16_bits(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }

// fp16(residual + fp16(v)): the unfused `residual + linear(x)` of two fp16 tensors.
__device__ __forceinline__ uint16_t finish_residual(float v, uint16_t r) {
  const float y = (float)(_Float16)v;
  return f16_bits(y + half_bits_to_float(r));
}

// fp16(fp16(silu(fp16(g))) * fp16(u)): torch's fp16 silu (x / (1 + exp(-x)) in fp32, one
// rounding) followed by its fp16 multiply, on the rounded linear outputs.
__device__ __forceinline__ uint16_t finish_silu_mul(float g, float u) {
  const float g16 = (float)(_Float16)g;
  const float u16 = (float)(_Float16)u;
  const float s16 = (float)(_Float16)(g16 / (1.0f + expf(-g16)));
  return f16_bits(s16 * u16);
}

// Write one output value v (= acc + bias, fp32) of row m, physical column n under the
// NONE / RESIDUAL epilogues.
__device__ __forceinline__ void store_out(const LinearArgs& a, int m, int n, float v) {
  uint16_t r = f16_bits(v);
  if (a.epilogue == TF_EPILOGUE_RESIDUAL) r = finish_residual(v, a.residual[(int64_t)m * a.ldr + n]);
  a.out[(int64_t)m * a.ldo + n] = r;
}

// Kernels whose accumulators hold runs of four consecutive output columns of one row (the
// MFMA with the weight fragment as its first operand) store each run as one 8-byte piece where
// N, the row strides and the pointers are in 4-element units.
__device__ __forceinline__ bool run_store_ok(const LinearArgs& a, const uint16_t* dst, int64_t ldd, bool residual) {
  return (a.n & 3) == 0 && (ldd & 3) == 0 && (reinterpret_cast<uintptr_t>(dst) & 7) == 0 &&
         (!residual || ((a.ldr & 3) == 0 && (reinterpret_cast<uintptr_t>(a.residual) & 7) == 0));
}

// Columns n .. n + 3 of row m (v: acc * row scale + bias in fp32) to dst (row stride ldd) as
// fp16, or as fp16(residual + fp16(v)) under the residual epilogue: the values store_out
// writes. vec: run_store_ok holds (then a run is inside N or past it); else per value, the
// columns past N skipped.
__device__ __forceinline__ void store_run4(const LinearArgs& a, uint16_t* dst, int64_t ldd, bool residual, int m,
                                           int n, const float (&v)[4], bool vec) {
  if (vec) {
    uint16_t h[4];
    if (residual) {
      const u2 res = *reinterpret_cast<const u2*>(a.residual + (int64_t)m * a.ldr + n);
#pragma unroll
      for (int j = 0; j < 4; ++j) h[j] = finish_residual(v[j], (uint16_t)(res[j >> 1] >> (16 * (j & 1))));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) h[j] = f16_bits(v[j]);
    }
    *reinterpret_cast<u2*>(dst + (int64_t)m * ldd + n) =
        u2{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (n + j >= a.n) break;
    uint16_t r = f16_bits(v[j]);
    if (residual) r = finish_residual(v[j], a.residual[(int64_t)m * a.ldr + n + j]);
    dst[(int64_t)m * ldd + n + j] = r;
  }
}

// Swaps the upper half wave of a with the lower half wave of b: afterwards lanes 0..31 hold their
// own a in a and the a of lane + 32 in b, lanes 32..63 the b of lane - 32 in a and their own b in b.
__device__ __forceinline__ void swap_halves(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(as_u32(a), as_u32(b), false, false);
  a = as_f32(r[0]);
  b = as_f32(r[1]);
}

// Columns n .. n + 3 of row m from the sums d of one run: fp32 to slice z of ws [split][M][N]
// (partials), else y with row scale rs, bias and the NONE / RESIDUAL epilogue to out. vec as in
// store_run4 (partials: 16-byte pieces of ws).
__device__ __forceinline__ void store_sums4(const LinearArgs& a, float* ws, bool partials, int z, int m, int n,
                                            float rs, const f4& d, bool residual, bool vec) {
  if (partials) {
    float* const p = ws + ((int64_t)z * a.m + m) * a.n + n;
    if (vec) {
      *reinterpret_cast<f4*>(p) = d;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < a.n) p[j] = d[j];
    }
    return;
  }
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float b = (a.bias && n + j < a.n) ? half_bits_to_float(a.bias[n + j]) : 0.0f;
    v[j] = d[j] * rs + b;
  }
  store_run4(a, a.out, a.ldo, residual, m, n, v, vec);
}

// Outputs j .. j + 3 of row m under SiLU*mul from the sums of their gate and up columns, one 8-byte
// piece where vec holds. N % 16 == 0, so a run lies inside N / 2 or past it.
__device__ __forceinline__ void store_silu4(const LinearArgs& a, int m, int j, float rs, const float (&gate)[4],
                                            const float (&up)[4], bool vec) {
  const int half = a.n >> 1;
  if (j >= half) return;
  uint16_t h[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float bg = a.bias ? half_bits_to_float(a.bias[j + q]) : 0.0f;
    const float bu = a.bias ? half_bits_to_float(a.bias[half + j + q]) : 0.0f;
    // y in fp32 before its fp16 rounding, as the plain epilogue computes it (the empty asm keeps the
    // compiler from fusing multiply, add and rounding into v_fma_mixlo_f16, which rounds once).
    float vg = gate[q] * rs + bg, vu = up[q] * rs + bu;
    __asm__ volatile("" : "+v"(vg), "+v"(vu));
    h[q] = finish_silu_mul(vg, vu);
  }
  uint16_t* const p = a.out + (int64_t)m * a.ldo + j;
  if (vec) {
    *reinterpret_cast<u2*>(p) = u2{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = h[q];
  }
}

// The results of a wave that holds TM x TN transposed 16x16 accumulator tiles (the MFMA with the
// weight fragment as its first operand): register q of lane l is row (m) l % 16 and column (n)
// 4 (l / 16) + q of its tile, so a lane holds runs of four consecutive columns of one row. Rows
// m_base + 16 tm, (virtual) columns n_base + 16 tn.
// SILU (SiLU*mul without partials): the wave's columns are mapped by phys_col (eight gate columns, then
// the eight up columns of the same outputs), so lanes l and l + 32 hold the gate and up values of
// one run. One half-wave swap between the two tiles of a pair gives the lower half wave both
// values of the first tile and the upper half wave both of the second, and every lane finishes
// four outputs of each pair. The alternative, fp16 y to a workspace and a second kernel that pairs
// it, writes and reads [M, N] once more: on MI355X the whole call took 1218 us against 1070 here at
// gate_up (N 37888, K 3584) M = 4096, 81.3 against 73.9 at M = 256, and 460 against 392 for the fp8
// GEMM with its norm at M = 2048. An instance of its own (SILU): as a runtime branch it cost the
// other epilogues 1% (down_proj M = 1000) and spilled the four-wave 32x32 tiles.
template <bool SILU, int TM, int TN>
__device__ __forceinline__ void store_tile16(const LinearArgs& a, float* ws, bool partials, int z, int m_base,
                                             int n_base, int lane, const f4 (&acc)[TM][TN]) {
  const int g = lane >> 4;
  if constexpr (SILU) {
    const int hw = lane >> 5;  // which tile of a pair this lane finishes
    const bool vec = (a.ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(a.out) & 7) == 0;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const int m = m_base + tm * 16 + (lane & 15);
      const float rs = row_scale(a, m);
#pragma unroll
      for (int tn = 0; tn < TN; tn += 2) {
        float gate[4], up[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // every lane takes part, rows past M too
          gate[q] = acc[tm][tn][q];
          up[q] = acc[tm][tn + 1 < TN ? tn + 1 : tn][q];
          swap_halves(gate[q], up[q]);
        }
        if (m < a.m && !(tn + 1 >= TN && hw))
          store_silu4(a, m, (n_base >> 1) + 8 * (tn + hw) + 4 * (g & 1), rs, gate, up, vec);
      }
    }
    return;
  }
  const bool residual = a.epilogue == TF_EPILOGUE_RESIDUAL;
  const bool vec = partials ? (a.n & 3) == 0 && (reinterpret_cast<uintptr_t>(ws) & 15) == 0
                            : run_store_ok(a, a.out, a.ldo, residual);
#pragma unroll
  for (int tm = 0; tm < TM; ++tm) {
    const int m = m_base + tm * 16 + (lane & 15);
    if (m >= a.m) continue;
    const float rs = row_scale(a, m);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int n = n_base + tn * 16 + 4 * g;
      if (n < a.n) store_sums4(a, ws, partials, z, m, n, rs, acc[tm][tn], residual, vec);
    }
  }
}

// store_tile16 for transposed 32x32 accumulator tiles: register 4 r + q of lane l is row l % 32 and
// column 8 r + 4 (l / 32) + q, so under the SiLU*mul mapping a lane holds the gate values of a run
// in registers 8 p .. 8 p + 3 and its up values in 8 p + 4 .. 8 p + 7.
template <bool SILU, int TM, int TN>
__device__ __forceinline__ void store_tile32(const LinearArgs& a, float* ws, bool partials, int z, int m_base,
                                             int n_base, int lane, const f16v (&acc)[TM][TN]) {
  const int h4 = 4 * (lane >> 5);
  const bool residual = a.epilogue == TF_EPILOGUE_RESIDUAL;
  const bool vec = partials ? (a.n & 3) == 0 && (reinterpret_cast<uintptr_t>(ws) & 15) == 0
                   : SILU   ? (a.ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(a.out) & 7) == 0
                            : run_store_ok(a, a.out, a.ldo, residual);
#pragma unroll
  for (int tm = 0; tm < TM; ++tm) {
    const int m = m_base + tm * 32 + (lane & 31);
    if (m >= a.m) continue;
    const float rs = row_scale(a, m);
    if constexpr (SILU) {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          float gate[4], up[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) gate[q] = acc[tm][tn][8 * p + q], up[q] = acc[tm][tn][8 * p + 4 + q];
          store_silu4(a, m, (n_base >> 1) + 16 * tn + 8 * p + h4, rs, gate, up, vec);
        }
      continue;
    }
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n_base + tn * 32 + 8 * r + h4;
        if (n >= a.n) continue;
        const f4 d = {acc[tm][tn][4 * r], acc[tm][tn][4 * r + 1], acc[tm][tn][4 * r + 2], acc[tm][tn][4 * r + 3]};
        store_sums4(a, ws, partials, z, m, n, rs, d, residual, vec);
      }
  }
}

// ------------------------------------------------------------------ launch helpers

// LDS bytes one workgroup may use on the current device (160 KiB on gfx950), queried once
// per device.
inline size_t device_max_lds() {
  static size_t cache[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 64 * 1024;
  if (cache[dev] == 0) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
      v = 64 * 1024;
    cache[dev] = (size_t)v;
  }
  return cache[dev];
}

// Dynamic LDS above 64 KiB must be enabled per kernel before the launch.
template <typename Kernel>
inline int reserve_lds(Kernel kernel, size_t bytes, const char* name) {
  if (bytes > 64 * 1024 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)bytes) != hipSuccess)
    return fail(TF_ELAUNCH, std::string("tf_w4a16_linear: cannot reserve LDS for ") + name);
  return TF_OK;
}

// Buffer offsets are 32-bit: every byte offset into qweight_t, scales, qzeros and x must fit
// (the streaming kernels address them through buffer resources).
inline int check_offsets(const LinearArgs& a) {
  const int64_t x_bytes = ((int64_t)(a.m - 1) * a.ldx + a.k) * 2;
  const int64_t w_bytes = (int64_t)a.n * (a.k / 2);
  if (x_bytes >= (int64_t)kOutOfRange || w_bytes >= (int64_t)kOutOfRange)
    return fail(TF_EINVAL, "tf_w4a16_linear: gemv kernels need x and qweight_t below 2 GiB");
  return TF_OK;
}

using LaunchFn = int (*)(const LinearArgs&, const tf_gemm_config&, float* workspace,
                         hipStream_t stream);
using WorkspaceFn = int64_t (*)(const LinearArgs&, const tf_gemm_config&);
// The checks a launch function makes before it launches anything (TF_OK or an error), for
// callers that must reject a call before they queue work of their own (tf_w4a8_linear_ex).
using CheckFn = int (*)(const LinearArgs&, const tf_gemm_config&);

// A compiled kernel variant: cfg holds (kernel, block_m, block_n, block_k, num_warps,
// num_stages) with split_k = 1. check may be null when the launch function rejects nothing
// beyond what tf_w4a16_linear_ex checks first.
struct Variant {
  tf_gemm_config cfg;
  LaunchFn launch;
  WorkspaceFn workspace;
  CheckFn check = nullptr;
};

const Variant* gemv_variants(int* count);
const Variant* gemv_stream_variants(int* count);
const Variant* gemm_variants(int* count);
const Variant* gemm2_variants(int* count);
const Variant* gemm3_variants(int* count);
const Variant* gemm4_variants(int* count);
const Variant* gemm5_variants(int* count);
const Variant* gemm8_variants(int* count);

int check_group_size(int32_t group_size, int64_t k, const char* name);
int log2_group(int32_t g);

// Upper bound on the split-K factor of any kernel.
constexpr int kMaxSplitK = 16;

}  // namespace tf
