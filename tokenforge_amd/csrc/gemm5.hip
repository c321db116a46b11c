// W4A16 GEMM for M from a handful of rows to 128, where the weight stream is the cost: eight waves
// split a tile's columns and its K.
//
// A workgroup of 8 = WN x WK waves computes 16 MT rows x BN = 16 RT WN columns. Wave (wn, kz) owns
// 16 RT columns and every WK-th 128-wide K step: it streams the packed weights, scales and zero
// words of its columns and steps into a register ring P steps deep, dequantizes each packed word
// (fp16(q - z) * s, one rounding) straight into the weight operand of v_mfma_f32_16x16x32_f16 and
// multiplies it with MT row fragments of x read from LDS. x streams into two LDS stages of WK steps
// ([WK][16 MT][128] fp16, buffer loads with the LDS destination), one stage ahead, with one barrier
// per WK steps. The WK partial sums of a tile meet in LDS at the end, added in kz order.
//
// Why this split. Weights pass from HBM to the MFMA without LDS, so LDS only carries x; an x fragment
// is read once per RT column tiles, and x is fetched from L2 once per workgroup, so a wide BN is what
// keeps both below the weight stream's time (at M = 48 the 64-column tiles of gemm3.hip fetch three
// times the bytes of the weights in x, and read 1 KB of LDS per MFMA). Splitting K over the waves
// instead of the columns lets BN be chosen for the grid (a whole round of tiles over the CUs) with
// eight waves in flight in any case, and needs no second kernel, unlike a K split over workgroups.
// Measured on MI355X against the fastest of the other forms (us, cold weights): gate_up (37888 x 3584)
// with SiLU*mul M = 16 23.3 / 26.8, M = 32 26.4 / 32.1, M = 64 32.7 / 46.9 (a pure read of the layer's
// loads takes 14.7); 3584 x 3584 M = 16 6.6 / 8.2; 4608 x 3584 M = 128 13.5 / 19.3, M = 512 27.9 / 36.7;
// 3584 x 18944 M = 64 22.8 / 27.2. Past M = 128 the LDS-tile GEMMs, which dequantize a weight once per 256
// rows, take over as soon as their tiles fill the CUs.
//
// LDS rows hold 16 chunks of 16 bytes (one 256-byte bank line); chunk c of row r sits in slot
// c ^ (r & 11), free of bank conflicts for the fragment reads (lane 16 g + c at row c, chunk
// 4 g + j), as in gemm4.hip. Steps past the workgroup's K range are loaded all the same, as zeros
// (weights through an empty buffer resource, x at an offset out of range), so every wave issues the
// same loads in every iteration and the barrier's vmcnt wait stays exact. Shapes: N % 16 == 0, K %
// 128 == 0.
//
// Split-K over workgroups (split_k > 1): K slices write fp32 partials [split][M][N] to the caller's
// workspace and splitk_reduce (gemm.hip) sums them in split order.
#include <type_traits>

#include "linear.h"

namespace tf {

int64_t split_workspace(const LinearArgs& a, int split);
int finish_split(const LinearArgs& a, const float* ws, int split, hipStream_t stream);

namespace {

constexpr int kStepK = 128;

template <int MT, int RT, int WN, int WK, int P>
struct G5 {
  static constexpr int kWaves = WN * WK;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int BM = 16 * MT;
  static constexpr int BN = 16 * RT * WN;
  static constexpr int kSub = BM * kStepK * 2;                     // bytes of one step of x
  static constexpr int kStage = WK * kSub;                         // bytes of one x stage
  static constexpr int kDma = kStage / 1024;                       // 1 KB LDS-load instructions per stage
  static constexpr int kDmaPerWave = kDma / kWaves;
  static constexpr int kSums = kWaves * MT * RT * 1024;  // the partial sums that meet in LDS
  static constexpr int kLds = kSums > 2 * kStage ? kSums : 2 * kStage;
  // VMEM issued after x stage t (an iteration back) when iteration t waits for it: the weights issued
  // at that iteration's end. (The first iterations may have more in flight; their wait is then longer,
  // never too short.)
  static constexpr int kAfterX = 3 * RT;
  static_assert(kWaves == 8 && WK >= 2, "eight waves, at least two of them along K");
  static_assert(kDma % kWaves == 0, "every wave loads the same share of a stage");
  static_assert(P >= 2 && P <= 4, "register ring of two to four steps");
  static_assert(kLds <= 160 * 1024, "x stages or sums exceed the LDS");
  static_assert(kAfterX < 64, "vmcnt range");
};

template <int N>
__device__ __forceinline__ void step_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (0x0 << 8) | ((N >> 4) << 14));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

template <int MT, int RT, int WN, int WK, int P, bool SILU>
__global__ __launch_bounds__(64 * WN * WK, 2) void gemm5_kernel(LinearArgs a, float* __restrict__ ws, int split_k,
                                                                int tiles_n, int tiles_m) {
  using C = G5<MT, RT, WN, WK, P>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15;
  const int g = lane >> 4;
  const int kz = wave / WN;
  const int wn = wave % WN;

  const int per_split = tiles_n * tiles_m;
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int z = t / per_split;
  const int r = t - z * per_split;
  const int m0 = (r % tiles_m) * C::BM;
  const int v0 = (r / tiles_m) * (C::BN / 16) + wn * RT;  // this wave's first (virtual) 16-column tile

  const int nsteps = a.k >> 7;
  const int s0 = (int)(((int64_t)z * nsteps) / split_k);
  const int s1 = (int)(((int64_t)(z + 1) * nsteps) / split_k);
  const int groups = a.k >> a.log2g;
  const uint32_t gps = (uint32_t)(kStepK >> a.log2g);  // groups per step

  const uint32_t x_bytes = (uint32_t)(((int64_t)(a.m - 1) * a.ldx + a.k) * 2);
  const uint32_t q_bytes = (uint32_t)a.n * (uint32_t)(a.k >> 1);
  const uint32_t s_bytes = (uint32_t)(groups * a.n * 2);
  const uint32_t z_bytes = (uint32_t)(groups * (a.n >> 3) * 4);

  // ---- x stage: instruction i = wave + 8 ii fills KB i of it: step i / (4 MT) of the stage, rows
  // 4 (i % (4 MT)) + g, lane l writing 16-byte slot l (chunk c ^ (row & 11) of its row).
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, x_bytes);
  uint32_t x_off[C::kDmaPerWave];  // byte offset of the lane's chunk for stage start s0, or out of range
  int x_sub[C::kDmaPerWave];       // wave-uniform
#pragma unroll
  for (int ii = 0; ii < C::kDmaPerWave; ++ii) {
    const int i = wave + C::kWaves * ii;
    const int sub = i / (4 * MT);
    const int row = 4 * (i - sub * 4 * MT) + g;
    x_sub[ii] = sub;
    x_off[ii] = m0 + row < a.m
                    ? (uint32_t)(((int64_t)(m0 + row) * a.ldx + (int64_t)sub * kStepK + (c ^ (row & 11)) * 8) * 2)
                    : kOutOfRange;
  }
  auto issue_x = [&](int s, int st) __attribute__((always_inline)) {  // the stage of steps s .. s + WK - 1
#pragma unroll
    for (int ii = 0; ii < C::kDmaPerWave; ++ii) {
      const int i = wave + C::kWaves * ii;
      const bool ok = s + x_sub[ii] < s1;  // wave-uniform
      const uint32_t off = ok ? x_off[ii] + (uint32_t)s * (kStepK * 2) : kOutOfRange;
      const uint32_t dst = (uint32_t)(st * C::kStage + i * 1024);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void*)(smem + dst), 16, off, 0, 0,
                                               0);
    }
  };

  // ---- weights of step s. Tile layout (N % 16 == 0: every 16-column tile is full): the lane's chunk
  // (column c, K block g) of step s of tile t sits at byte (t nsteps + s) 1024 + (16 g + c) 16, its
  // scale and zero word at (t P + grp) 32 + 2 c and (t P + grp) 8 + 4 (c / 8), grp = s gps + (32 g) / G.
  // SiLU*mul: virtual tile v covers outputs 8 v .. 8 v + 7: lanes c < 8 take half v % 2 of tile v / 2
  // (gate rows 8 v + c), lanes c >= 8 the up rows N / 2 + 8 v + c - 8, half-tile v + N / 16. Either
  // way a lane's part of an offset is a constant (one per parity of v: with N / 16 odd the up rows of
  // an even v are the second half of a tile) and the rest is wave-uniform.
  const uint32_t gl = (uint32_t)((g * 32) >> a.log2g);  // the lane's group inside a step
  const uint32_t cl = SILU ? (uint32_t)c & 7u : (uint32_t)c;
  constexpr int NP = SILU ? 2 : 1;
  uint32_t w_lane[NP], s_lane[NP], z_lane[NP];  // by the parity of the wave's local tile rt
#pragma unroll
  for (int par = 0; par < NP; ++par) {
    const int vpar = (v0 + par) & 1;
    const bool up = SILU && c >= 8;
    const int n16 = a.n >> 4;
    const uint32_t dt = up ? (uint32_t)((n16 + vpar) >> 1) : 0u;  // tiles from the gate row's
    const uint32_t dh = up && (n16 & 1) ? (vpar ? 0xFFFFFFFFu : 1u) : 0u;  // halves (added modulo 2^32)
    w_lane[par] = dt * (uint32_t)nsteps * 1024u + dh * 128u + (16u * g + cl) * 16u;
    s_lane[par] = (dt * (uint32_t)groups + gl) * 32u + dh * 16u + 2u * cl;
    z_lane[par] = (dt * (uint32_t)groups + gl) * 8u + dh * 4u + 4u * (cl >> 3);
  }
  const uint32_t zsh = 4u * awq_nibble_of((uint32_t)c & 7u);
  u4 raw[P][RT];
  uint32_t raw_s[P][RT], raw_z[P][RT];
  auto issue_w = [&](int s, int slot) __attribute__((always_inline)) {
    const bool ok = s < s1;
    const __amdgpu_buffer_rsrc_t rq = make_rsrc(a.qw, ok ? q_bytes : 0u);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.scales, ok ? s_bytes : 0u);
    const __amdgpu_buffer_rsrc_t rz = make_rsrc(a.qz, ok ? z_bytes : 0u);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const uint32_t v = (uint32_t)(v0 + rt);
      const uint32_t tt = SILU ? v >> 1 : v, h = SILU ? v & 1u : 0u;
      const uint32_t gi = tt * (uint32_t)groups + (uint32_t)s * gps;
      const int par = SILU ? rt & 1 : 0;
      // A tile past N lies past the end of its buffers (zeros), or under SiLU*mul in rows that
      // exist: its results are not stored.
      raw[slot][rt] = __builtin_amdgcn_raw_buffer_load_b128(
          rq, (int)(w_lane[par] + (tt * (uint32_t)nsteps + (uint32_t)s) * 1024u + h * 128u), 0, 0);
      raw_s[slot][rt] =
          (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rs, (int)(s_lane[par] + gi * 32u + h * 16u), 0, 0);
      raw_z[slot][rt] = __builtin_amdgcn_raw_buffer_load_b32(rz, (int)(z_lane[par] + gi * 8u + h * 4u), 0, 0);
    }
  };

  f4 acc[MT][RT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[mt][rt] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  // A fragment mt of K block j of this wave's step: row 16 mt + c, chunk 4 g + j.
  const uint32_t a_lane = (uint32_t)(kz * C::kSub + c * 256 + ((4 * g) ^ (c & 11)) * 16);
  const UnpackConsts uc = unpack_consts();
  auto compute = [&](int st, int slot) __attribute__((always_inline)) {
    const uint32_t base = a_lane + (uint32_t)(st * C::kStage);
    QuantParams qp[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) qp[rt] = make_params((raw_z[slot][rt] >> zsh) & 0xFu, raw_s[slot][rt]);
    h8 af[2][MT];
    auto read_a = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        af[j & 1][mt] = *reinterpret_cast<const h8*>(smem + (base ^ (uint32_t)(j * 16)) + mt * 4096);
    };
    read_a(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < 3) read_a(j + 1);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        h2 wd[4];
        dequant_word(raw[slot][rt][j], qp[rt], uc, wd);
        const h8 b = pack_h8(wd);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[mt][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, af[j & 1][mt], acc[mt][rt], 0, 0, 0);
      }
    }
  };

  // ---- prologue: the first x stage in flight, weights of this wave's first P steps in the ring
  issue_x(s0, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < P; ++i) {
    issue_w(s0 + kz + i * WK, i);
    __builtin_amdgcn_sched_barrier(0);
  }

  // Iteration at stage start s (ring slot a compile-time value): wait for its x stage, issue the next
  // one into the stage read in the previous iteration, multiply this wave's step, refill its ring slot. In the tail (fewer than P stages left) the weights an iteration issues are never
  // read, so the compiler drops those loads and the count after the stage is smaller than kAfterX:
  // the tail's barriers wait for every load instead.
  auto iteration = [&](int s, int st, auto slot_tag, auto tail_tag) __attribute__((always_inline)) {
    constexpr int slot = decltype(slot_tag)::value;
    step_barrier<decltype(tail_tag)::value ? 0 : C::kAfterX>();
    issue_x(s + WK, 1 - st);
    // The waits count the loads issued after each x stage: no later load may move above it.
    __builtin_amdgcn_sched_barrier(0);
    if (s + kz < s1) compute(st, slot);  // wave-uniform: no step left for this wave past the end
    issue_w(s + kz + P * WK, slot);
    __builtin_amdgcn_sched_barrier(0);
  };
  using Loop = std::false_type;
  using Tail = std::true_type;
  int s = s0, st = 0;
  for (; s + (P - 1) * WK < s1; s += P * WK) {
    iteration(s, st, std::integral_constant<int, 0>{}, Loop{});
    st = 1 - st;
    iteration(s + WK, st, std::integral_constant<int, 1>{}, Loop{});
    st = 1 - st;
    if constexpr (P > 2) {
      iteration(s + 2 * WK, st, std::integral_constant<int, 2>{}, Loop{});
      st = 1 - st;
    }
    if constexpr (P > 3) {
      iteration(s + 3 * WK, st, std::integral_constant<int, 3>{}, Loop{});
      st = 1 - st;
    }
  }
  // Fewer than P stages remain.
  if (s < s1) {
    iteration(s, st, std::integral_constant<int, 0>{}, Tail{});
    st = 1 - st;
  }
  if constexpr (P > 2) {
    if (s + WK < s1) {
      iteration(s + WK, st, std::integral_constant<int, 1>{}, Tail{});
      st = 1 - st;
    }
  }
  if constexpr (P > 3) {
    if (s + 2 * WK < s1) iteration(s + 2 * WK, st, std::integral_constant<int, 2>{}, Tail{});
  }

  // ---- the WK partial sums of each tile, through LDS (every x stage has been read; the loads
  // still in flight are of stages past the end: the barrier waits until they have landed, before
  // their LDS is reused): wave (wn, kz) takes row tiles kz, kz + WK, ... and adds them in kz order.
  step_barrier<0>();
  f4* const sums = reinterpret_cast<f4*>(smem);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) sums[((wave * MT + mt) * RT + rt) * 64 + lane] = acc[mt][rt];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (MT + WK - 1) / WK; ++i) {
    const int mt = kz + i * WK;
    if (mt >= MT) break;  // wave-uniform
    f4 out[1][RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      f4 v = sums[((wn * MT + mt) * RT + rt) * 64 + lane];
#pragma unroll
      for (int w = 1; w < WK; ++w) {
        const f4 p = sums[(((w * WN + wn) * MT + mt) * RT + rt) * 64 + lane];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] += p[q];
      }
      out[0][rt] = v;
    }
    store_tile16<SILU, 1, RT>(a, ws, split_k > 1, z, m0 + 16 * mt, 16 * v0, lane, out);
  }
}

int effective_split5(const LinearArgs& a, const tf_gemm_config& cfg) {
  const int nsteps = a.k >> 7;
  return cfg.split_k < nsteps ? cfg.split_k : (nsteps > 0 ? nsteps : 1);
}

int64_t gemm5_workspace(const LinearArgs& a, const tf_gemm_config& cfg) {
  return split_workspace(a, effective_split5(a, cfg));
}

template <int BM, int BN>
int check_gemm5(const LinearArgs& a, const tf_gemm_config& cfg) {
  if ((a.n & 15) || (a.k & 127))
    return fail(TF_EINVAL, "tf_w4a16_linear: this gemm_mfma variant needs N % 16 == 0 and K % 128 == 0");
  const int64_t x_bytes = ((int64_t)(a.m - 1) * a.ldx + a.k) * 2;
  const int64_t w_bytes = (int64_t)a.n * (a.k / 2);
  if (x_bytes >= (int64_t)kOutOfRange || w_bytes >= (int64_t)kOutOfRange)
    return fail(TF_EINVAL, "tf_w4a16_linear: this gemm_mfma variant needs x and qweight_t below 2 GiB");
  if (cdiv(a.n, BN) * cdiv(a.m, BM) * effective_split5(a, cfg) > 0x7FFFFFFF)
    return fail(TF_EINVAL, "tf_w4a16_linear: too many tiles");
  return TF_OK;
}

template <int MT, int RT, int WN, int WK, int P>
int launch_gemm5(const LinearArgs& a, const tf_gemm_config& cfg, float* ws, hipStream_t stream) {
  using C = G5<MT, RT, WN, WK, P>;
  if (int rc = check_gemm5<C::BM, C::BN>(a, cfg)) return rc;
  const int split = effective_split5(a, cfg);
  if (split > 1 && ws == nullptr) return fail(TF_EINVAL, "tf_w4a16_linear: split-K needs a workspace");
  const int tiles_n = (int)cdiv(a.n, C::BN);
  const int tiles_m = (int)cdiv(a.m, C::BM);
  const bool silu = split == 1 && a.epilogue == TF_EPILOGUE_SILU_MUL;
  auto kernel = silu ? gemm5_kernel<MT, RT, WN, WK, P, true> : gemm5_kernel<MT, RT, WN, WK, P, false>;
  if (int rc = reserve_lds(kernel, C::kLds, "gemm_mfma")) return rc;
  kernel<<<(unsigned)(tiles_n * tiles_m * split), C::kThreads, C::kLds, stream>>>(a, ws, split, tiles_n, tiles_m);
  if (int rc = check_launch("tf_w4a16_linear(gemm_mfma)")) return rc;
  return finish_split(a, ws, split, stream);
}

// block_k 128 with num_warps 8 marks these variants; block_m 16 MT, block_n 16 RT WN, num_stages 6, 7
// or 8 for WK = 2, 4 or 8 waves along K.
#define TF_GEMM5(MT, RT, WN, WK, P)                                                        \
  {{TF_KERNEL_GEMM_MFMA, 16 * MT, 16 * RT * WN, 128, 1, WN * WK, WK == 2 ? 6 : WK == 4 ? 7 : 8}, \
   (launch_gemm5<MT, RT, WN, WK, P>), gemm5_workspace, (check_gemm5<16 * MT, 16 * RT * WN>)}

const Variant kGemm5Variants[] = {
    // WK 8: narrow tiles, K split over all eight waves
    TF_GEMM5(1, 1, 1, 8, 4), TF_GEMM5(1, 2, 1, 8, 3), TF_GEMM5(1, 4, 1, 8, 2), TF_GEMM5(2, 1, 1, 8, 4),
    TF_GEMM5(2, 2, 1, 8, 3), TF_GEMM5(2, 4, 1, 8, 2),
    // WK 4
    TF_GEMM5(1, 2, 2, 4, 3), TF_GEMM5(1, 4, 2, 4, 2), TF_GEMM5(1, 5, 2, 4, 2), TF_GEMM5(2, 2, 2, 4, 3),
    TF_GEMM5(2, 4, 2, 4, 2), TF_GEMM5(2, 5, 2, 4, 2), TF_GEMM5(3, 2, 2, 4, 3), TF_GEMM5(3, 4, 2, 4, 2),
    TF_GEMM5(3, 5, 2, 4, 2), TF_GEMM5(4, 2, 2, 4, 3), TF_GEMM5(4, 4, 2, 4, 2), TF_GEMM5(4, 5, 2, 4, 2),
    // WK 2
    TF_GEMM5(2, 2, 4, 2, 3), TF_GEMM5(3, 3, 4, 2, 2), TF_GEMM5(4, 2, 4, 2, 3), TF_GEMM5(4, 3, 4, 2, 2), TF_GEMM5(5, 3, 4, 2, 2), TF_GEMM5(6, 2, 4, 2, 3),
    TF_GEMM5(6, 3, 4, 2, 2), TF_GEMM5(8, 1, 4, 2, 4), TF_GEMM5(8, 2, 4, 2, 2),
};

}  // namespace

const Variant* gemm5_variants(int* count) {
  *count = (int)(sizeof(kGemm5Variants) / sizeof(kGemm5Variants[0]));
  return kGemm5Variants;
}

}  // namespace tf
