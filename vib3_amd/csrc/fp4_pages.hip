// fp4_pages.hip — the reference's per-page NVFP4 launchers, the path execute_expert takes for
// NVFP4 experts that do not fit the fused table's one page per segment (engine.rs:5960-6226):
//
//   block-scaled GEMV (E2M1 weights x FP4-quantized activation, E8M0 scales):
//     vib3_launch_gemv_mma_nvfp4_preq[_fast]          kernels.cu:3752, :5229  row-major split-half
//     vib3_launch_fused_swiglu_mma_nvfp4_preq[_fast]  kernels.cu:3853, :5267  (SwiGLU of two)
//     vib3_launch_gemv_mma_nvfp4_tiled                kernels.cu:4359         tiled split-half
//     vib3_launch_gemv_scalar_nvfp4                   kernels.cu:4520         full bf16 scales
//     vib3_launch_gemv_mma_nvfp4, _fused_swiglu_mma_nvfp4  kernels.cu:3676, :3807  f32 input,
//                                                     quantized in the kernel; sequential codes
//   f32 GEMV over dequantized weights (the reference's scalar kernels, no activation rounding):
//     vib3_launch_partial_matmul_nvfp4[_f32out|_fp16in]  kernels.cu:1524, :2499, :1552
//     vib3_launch_fused_swiglu_nvfp4[_f32out]            kernels.cu:1537, :2483
//
// Layouts: a page is [rows][K/2] code bytes, then [rows][K/32] 2-byte scales (kernels.rs:
// 821-860: scales at page + K/2 * rows). "Sequential" bytes hold values 2j (low nibble) and
// 2j + 1; "split-half" 16-byte groups hold values j and j + 16 (after
// vib3_launch_repack_weights_inplace); "tiled" puts 16 rows x 64 values in 512-byte tiles
// (after vib3_launch_repack_row_to_tiled). The block-scaled kernels read a scale's exponent
// byte as E8M0, like the MMA instruction (kernels.cu:3355); the scalar ones its bf16 value.
//
// Arithmetic of the block-scaled kernels: as in fp4_fused.hip, each 32-value group's dot
// product is exact in f32, scaled by exact powers of two and summed in f64, the row rounded to
// f32 once: the result does not depend on the summation order and equals the oracle's. The
// scalar kernels accumulate x * w * s in f32 (an order of their own, as the reference's warp
// reductions have theirs).
#include "common.h"
#include "fp4.h"
#include "kernels.h"

namespace vib3 {
namespace {

enum { kLayRowSplit = 0, kLayTiled = 1, kLaySeq = 2 };

typedef float f32x2 __attribute__((ext_vector_type(2)));

struct PageGemvArgs {
  const uint8_t* act;     // split-half activation codes [K/32][16], or null: quantize x
  const uint8_t* act_sc;  // [K/32] E8M0
  const float* x;         // f32 activation when act is null
  const uint8_t* w[2];    // code bytes of one matrix, or up and gate
  const uint16_t* s[2];   // their scales [M][K/32]
  float* out;             // [M] f32
  int K, M;
};

// How k_fp4_page_rows and k_nvfp4_scalar_rows split a page (one launch reads at most a few megabytes, so they are bound by
// the round trips of a launch, not by bandwidth: every load a wave needs goes out at once, and the
// page is spread over as many waves as it has row groups).
//   * A row is read by L lanes, R = 64 / L rows by a wave; lane `sub` of a row takes the 32-value
//     groups sub, sub + L, ... (16 bytes each, so a load instruction reads 16 L contiguous bytes of
//     each row). L is the smallest of 16, 32 and 64 for which a row takes one pass of kJ groups per
//     lane (K <= 2048, 4096, 8192); above that L = 64 and the row takes several passes.
//   * The activation groups a lane multiplies are the same for every row, so they are decoded into
//     registers straight from memory: no staging, no barrier. (Decoding the whole activation into
//     LDS in 16-row workgroups used 33 of the 256 CUs for a 520-row page and waited for two barriers
//     and 56 dependent steps per lane.)
//   * Waves stride over the row groups, the next group's weights loading while one is reduced.
// Traced: 520-row gate/up page pair at K = 7168 (4.2 MB) 12.2 -> 5.1 us (f32 input quantized in the
// kernel: 36.7 -> 6.8), 1820-row down page at K = 2048 (2.1 MB) 4.9 -> 4.2 us.
constexpr int kJ = 4;

// Bytes of group g of row r in layout LAY.
template <int LAY>
__device__ __forceinline__ const uint8_t* group_ptr(const uint8_t* w, int r, int g, int K) {
  if (LAY == kLayTiled)
    return w + ((size_t)(r >> 4) * (K / 64) + (g >> 1)) * 512 + (r & 15) * 32 + (g & 1) * 16;
  return w + (size_t)r * (K / 2) + (size_t)g * 16;
}

// One pass's weights of a row group: code words and scales of NS matrices.
template <int NS>
struct PageStep {
  uint4 w[NS][kJ];
  uint16_t q[NS][kJ];
};

// Groups past the row end re-read its last group (no branch around the loads).
template <int LAY, int NS, int L>
__device__ __forceinline__ void page_issue(PageStep<NS>& b, const uint8_t* const (&w)[2],
                                           const uint16_t* const (&s)[2], int row, int pass, int K,
                                           int G, int sc_shift) {
  const int sub = lane_id() % L;
#pragma unroll
  for (int j = 0; j < kJ; j++) {
    if (pass * L * kJ + L * j >= G) break;  // (wave-uniform)
    const int g = min((pass * kJ + j) * L + sub, G - 1);
#pragma unroll
    for (int m = 0; m < NS; m++) {
      b.w[m][j] = ld_stream(group_ptr<LAY>(w[m], row, g, K));
      b.q[m][j] = ld_u16(s[m] + (size_t)row * (G >> sc_shift) + (g >> sc_shift));
    }
  }
}

template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (uint32_t)lo);
}

// Sum over a row's L lanes (every lane gets it).
template <int L>
__device__ __forceinline__ double row_sum(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0x141>(v);
  v += dpp_d<0x140>(v);
  if (L >= 32) v += shfl_xor_d(v, 16);
  if (L >= 64) v += shfl_xor_d(v, 32);
  return v;
}
template <int L>
__device__ __forceinline__ float row_sum(float v) {
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  v += dpp<0x141>(v);
  v += dpp<0x140>(v);
  if (L >= 32) v += __shfl_xor(v, 16);
  if (L >= 64) v += __shfl_xor(v, 32);
  return v;
}

// 32 consecutive f32 values (16-byte loads where `vec`).
__device__ __forceinline__ void load32(const float* x, bool vec, float (&v)[32]) {
  if (vec) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float4 t = ((const float4*)x)[i];
      v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 32; i++) v[i] = x[i];
  }
}

// The activation quantizer's rule (kernels.cu:3193-3240, inline at :3418-3470) for one group:
// E8M0 of the absolute maximum, codes rounded to nearest even, in sequential order.
__device__ __forceinline__ uint4 quantize_group_seq(const float (&v)[32], int& e_out) {
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; i++) amax = fmaxf(amax, fabsf(v[i]));
  const uint32_t e = e8m0_of_amax(amax);
  e_out = (int)e;
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float t[8] = {v[8 * i], v[8 * i + 1], v[8 * i + 2], v[8 * i + 3],
                        v[8 * i + 4], v[8 * i + 5], v[8 * i + 6], v[8 * i + 7]};
    o[i] = quantize8(t, e);
  }
  if (e == 0 && amax > 0.0f) {  // below the E8M0 range: v * inf, as k_fp4_quant_act
#pragma unroll
    for (int i = 0; i < 4; i++) {
      o[i] = 0;
#pragma unroll
      for (int j = 0; j < 8; j++) o[i] |= e2m1_rne(v[8 * i + j] * e8m0_inv(0)) << (4 * j);
    }
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// Block-scaled GEMV of NS matrices (NS = 2: up and gate, SwiGLU). ONE: a row is one pass.
// Sequential weights meet a sequential activation: with f32 input the workgroup quantizes it into
// LDS first (one group per thread), in the order the weights have.
template <int LAY, bool FULL, int NS, int L, bool ONE>
__global__ __launch_bounds__(256) void k_fp4_page_rows(PageGemvArgs a) {
  extern __shared__ uint4 lds[];
  constexpr int R = kWave / L;
  const int G = a.K / 32, M = a.M, lane = lane_id(), sub = lane % L, rr = lane / L;
  const int wpb = (int)(blockDim.x >> 6);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int groups = (M + R - 1) / R, stride = (int)gridDim.x * wpb;
  int rg = (int)blockIdx.x * wpb + wave;
  const uint8_t* const w[2] = {a.w[0], a.w[1]};
  const uint16_t* const s[2] = {a.s[0], a.s[1]};
  auto row_of = [&](int q) { return min(q * R + rr, M - 1); };
  PageStep<NS> A, B;
  const int passes = ONE ? 1 : (G + L * kJ - 1) / (L * kJ);
  if (LAY != kLaySeq) page_issue<LAY, NS, L>(A, w, s, row_of(rg), 0, a.K, G, 0);
  const uint8_t* codes = a.act;
  int* es = nullptr;
  if (LAY == kLaySeq) {
    es = (int*)(lds + G);
    const bool vec = ((uintptr_t)a.x & 15) == 0;
    for (int g = (int)threadIdx.x; g < G; g += (int)blockDim.x) {
      float v[32];
      load32(a.x + (size_t)g * 32, vec, v);
      int e;
      lds[g] = quantize_group_seq(v, e);
      es[g] = e;
    }
    __syncthreads();
    page_issue<LAY, NS, L>(A, w, s, row_of(rg), 0, a.K, G, 0);
  }
  f16x2 xp[kJ][16];
  int ex[kJ];
  auto load_act = [&](int pass) {
#pragma unroll
    for (int j = 0; j < kJ; j++) {
      if (pass * L * kJ + L * j >= G) break;
      const int g0 = (pass * kJ + j) * L + sub, g = min(g0, G - 1);
      const uint4 c = LAY == kLaySeq ? lds[g] : *(const uint4*)(codes + (size_t)g * 16);
      ex[j] = LAY == kLaySeq ? es[g] : (int)a.act_sc[g];
      // a group past the row end counts as zeros
      decode_group(g0 < G ? c : make_uint4(0u, 0u, 0u, 0u), xp[j]);
    }
  };
  double acc[NS];
  auto reduce = [&](const PageStep<NS>& b, int pass) {
#pragma unroll
    for (int j = 0; j < kJ; j++) {
      if (pass * L * kJ + L * j >= G) break;
#pragma unroll
      for (int m = 0; m < NS; m++) {
        f16x2 wp[16];
        decode_group(b.w[m][j], wp);
        float d = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) d = __builtin_amdgcn_fdot2(wp[i], xp[j][i], d, false);
        const int ew = (b.q[m][j] >> 7) & 0xff;
        const double sc = FULL ? (double)bf16_to_f32(b.q[m][j]) * pow2d(ex[j] - 127)
                               : pow2d(ew + ex[j] - 254);
        // a group past the row end: d = 0, and its scale may be anything
        const double t = fma((double)d, sc, acc[m]);
        acc[m] = (pass * kJ + j) * L + sub < G ? t : acc[m];
      }
    }
  };
  auto finish = [&](int q) {
    double t[NS];
#pragma unroll
    for (int m = 0; m < NS; m++) t[m] = row_sum<L>(acc[m]);
    const int row = q * R + rr;
    if (sub == 0 && row < M)
      a.out[row] = NS == 1 ? (float)t[0] : swiglu_fp4((float)t[NS - 1], (float)t[0]);
  };
  if (ONE) {
    load_act(0);
    for (;; ) {
      // the next row group (past the end: the last row again, dropped)
      page_issue<LAY, NS, L>(B, w, s, row_of(min(rg + stride, groups)), 0, a.K, G, 0);
#pragma unroll
      for (int m = 0; m < NS; m++) acc[m] = 0.0;
      reduce(A, 0);
      finish(rg);
      rg += stride;
      if (rg >= groups) break;
      A = B;
    }
  } else {
    for (; rg < groups; rg += stride) {
#pragma unroll
      for (int m = 0; m < NS; m++) acc[m] = 0.0;
      for (int p = 0; p < passes; p++) {
        if (p > 0 || rg >= stride) page_issue<LAY, NS, L>(A, w, s, row_of(rg), p, a.K, G, 0);
        load_act(p);
        reduce(A, p);
      }
      finish(rg);
    }
  }
}

// One group's 16 split-half bytes as the LDS pair layout group_dot reads.
__device__ __forceinline__ void put_group(uint4* pairs, int* ex, int g, uint4 w, int e) {
  f16x2 p[16];
  decode_group(w, p);
#pragma unroll
  for (int q = 0; q < 4; q++)
    pairs[(size_t)g * 4 + q] =
        make_uint4(__builtin_bit_cast(uint32_t, p[4 * q]), __builtin_bit_cast(uint32_t, p[4 * q + 1]),
                   __builtin_bit_cast(uint32_t, p[4 * q + 2]), __builtin_bit_cast(uint32_t, p[4 * q + 3]));
  ex[g] = e;
}

// The same GEMV with the activation staged: workgroup = 16 rows, 16 lanes per row (a lane takes
// groups l, l + 16, ...), the activation decoded once per workgroup into LDS pairs and exponents. One
// workgroup per 16 rows keeps every wave short and lets the hardware balance them, which wins where
// k_fp4_page_rows has too few groups per lane (short rows) or too many rows per wave (see page_staged).
template <int LAY, bool FULL, int NS>
__global__ __launch_bounds__(256) void k_fp4_page_staged(PageGemvArgs a) {
  extern __shared__ uint4 lds[];
  const int G = a.K / 32, tid = (int)threadIdx.x;
  // the arguments' two cache lines in one round trip (K lies in the second: fetching `act` behind it
  // cost 0.25 us of 2.5 to 4)
  asm volatile("" ::"s"(a.K), "s"(a.act));
  uint4* pairs = lds;                      // [G][4]
  int* ex = (int*)(lds + (size_t)G * 4);   // [G]
  for (int g = tid; g < G; g += 256)
    put_group(pairs, ex, g, *(const uint4*)(a.act + (size_t)g * 16), a.act_sc[g]);
  __syncthreads();
  const int gl = tid & 15, row = (int)blockIdx.x * 16 + (tid >> 4);
  const int rc = row < a.M ? row : a.M - 1;
  double acc[NS];
#pragma unroll
  for (int m = 0; m < NS; m++) acc[m] = 0.0;
  for (int g = gl; g < G; g += 16) {
    const double ea = pow2d(ex[g] - 127);
#pragma unroll
    for (int m = 0; m < NS; m++) {
      const uint4 w = *(const uint4*)group_ptr<LAY>(a.w[m], rc, g, a.K);
      const uint16_t sw = a.s[m][(size_t)rc * G + g];
      const double ws = FULL ? (double)bf16_to_f32(sw) : pow2d((int)((sw >> 7) & 0xff) - 127);
      acc[m] = fma((double)group_dot(w, pairs + (size_t)g * 4), ws * ea, acc[m]);
    }
  }
#pragma unroll
  for (int m = 0; m < NS; m++)
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) acc[m] += shfl_xor_d(acc[m], o);
  if (gl == 0 && row < a.M)
    a.out[row] = NS == 1 ? (float)acc[0] : swiglu_fp4((float)acc[NS - 1], (float)acc[0]);
}

struct ScalarArgs {
  const void* x;          // f32 or f16 [K]
  const uint8_t* w[2];    // sequential codes [M][K/2]
  const uint16_t* s[2];   // bf16 scales [M][K / bs]
  void* out;              // f16 or f32 [M]
  int K, M, bs_shift;     // block size 32 << bs_shift... as a shift of 32-value groups
};

// out[r] = sum_k x[k] * e2m1(W[r][k]) * bf16(s[r][k / bs]) in f32: per 32-value group the
// products x * e2m1 summed with fused multiply-adds, then times the block scale into the row
// sum; SwiGLU (NS = 2: up, gate) as the reference's epilogue silu(g) * u with
// silu(g) = g / (1 + e^-g) (kernels.cu:580-582, :2027-2028). The lane's x groups stay in registers
// as f32; split as above (a 520-row pair at K = 7168: 90 -> 8.0 us).
template <bool IN16, bool OUT16, int NS, int L, bool ONE>
__global__ __launch_bounds__(256) void k_nvfp4_scalar_rows(ScalarArgs a) {
  constexpr int R = kWave / L;
  const int G = a.K / 32, M = a.M, lane = lane_id(), sub = lane % L, rr = lane / L;
  const int wpb = (int)(blockDim.x >> 6);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int groups = (M + R - 1) / R, stride = (int)gridDim.x * wpb;
  const uint8_t* const w[2] = {a.w[0], a.w[1]};
  const uint16_t* const s[2] = {a.s[0], a.s[1]};
  const int passes = ONE ? 1 : (G + L * kJ - 1) / (L * kJ);
  const bool vec = ((uintptr_t)a.x & 15) == 0;
  PageStep<NS> A;
  float xv[kJ][32];
  auto load_x = [&](int pass) {
#pragma unroll
    for (int j = 0; j < kJ; j++) {
      if (pass * L * kJ + L * j >= G) break;
      const int g0 = (pass * kJ + j) * L + sub, g = min(g0, G - 1);
      if (!IN16) {
        load32((const float*)a.x + (size_t)g * 32, vec, xv[j]);
      } else {
        const uint16_t* p = (const uint16_t*)a.x + (size_t)g * 32;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          uint4 t;
          if (vec) t = ((const uint4*)p)[i];
          else __builtin_memcpy(&t, p + 8 * i, 16);
          const uint32_t tw[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
          for (int k = 0; k < 8; k++) xv[j][8 * i + k] = f16_to_f32((uint16_t)(tw[k >> 1] >> (16 * (k & 1))));
        }
      }
    }
  };
  float acc[NS];
  auto reduce = [&](const PageStep<NS>& b, int pass) {
#pragma unroll
    for (int j = 0; j < kJ; j++) {
      if (pass * L * kJ + L * j >= G) break;
#pragma unroll
      for (int m = 0; m < NS; m++) {
        const uint32_t wd[4] = {b.w[m][j].x, b.w[m][j].y, b.w[m][j].z, b.w[m][j].w};
        float p = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const f32x2 v0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wd[i], 1.0f, 0);
          const f32x2 v1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wd[i], 1.0f, 1);
          const f32x2 v2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wd[i], 1.0f, 2);
          const f32x2 v3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wd[i], 1.0f, 3);
          const float e[8] = {v0[0], v0[1], v1[0], v1[1], v2[0], v2[1], v3[0], v3[1]};
#pragma unroll
          for (int k = 0; k < 8; k++) p = __builtin_fmaf(xv[j][8 * i + k], e[k], p);
        }
        const float t = __builtin_fmaf(p, bf16_to_f32(b.q[m][j]), acc[m]);
        acc[m] = (pass * kJ + j) * L + sub < G ? t : acc[m];
      }
    }
  };
  for (int rg = (int)blockIdx.x * wpb + wave, first = rg; rg < groups; rg += stride) {
#pragma unroll
    for (int m = 0; m < NS; m++) acc[m] = 0.0f;
    for (int p = 0; p < passes; p++) {
      page_issue<kLaySeq, NS, L>(A, w, s, min(rg * R + rr, M - 1), p, a.K, G, a.bs_shift);
      if (!ONE || rg == first) load_x(p);
      reduce(A, p);
    }
    float t[NS];
#pragma unroll
    for (int m = 0; m < NS; m++) t[m] = row_sum<L>(acc[m]);
    const int row = rg * R + rr;
    if (sub == 0 && row < M) {
      const float v = NS == 1 ? t[0] : (t[NS - 1] / (1.0f + expf(-t[NS - 1]))) * t[0];
      if (OUT16) ((uint16_t*)a.out)[row] = f32_to_f16_bits(v);
      else ((float*)a.out)[row] = v;
    }
  }
}

// Launch shape for M rows of G groups: L lanes per row (see above), and one wave per row group up
// to eight per CU, two to a workgroup while that spreads a page over more CUs.
struct PageShape {
  int L;
  bool one;
  unsigned grid, block;
};
PageShape page_shape(int M, int G) {
  PageShape p{};
  p.L = G <= 16 * kJ ? 16 : G <= 32 * kJ ? 32 : 64;
  p.one = G <= p.L * kJ;
  const int groups = (M + kWave / p.L - 1) / (kWave / p.L);
  const int waves = groups < 8 * device_cus() ? groups : 8 * device_cus();
  const int wpb = waves <= 4 * device_cus() ? 2 : 4;
  p.block = 64u * wpb;
  p.grid = (unsigned)((waves + wpb - 1) / wpb);
  return p;
}

// Whether a page with quantized activations takes k_fp4_page_staged. us per launch, weights from HBM,
// staged / row kernel:
//   * short rows, where a launch's fixed chain decides: K = 1024 520 rows 3.2 / 3.4, pairs 3.8 / 3.9
//     (16 rows 3.2 / 2.6), K = 512 2.5 / 3.1;
//   * many rows, where the row kernel's waves walk several row groups: K = 2048 2064 rows 4.6 / 4.3,
//     8192 5.4 / 5.7, pairs 5.5 / 5.3 and 5.7 / 6.0 (3072 rows); K = 2560 7168 rows 5.9 / 5.9, 16384
//     7.8 / 9.3; K = 4096 12288 rows 10.2 / 9.2, 16384 10.8 / 11.4, pairs of 6144 9.9 / 9.0, 8192 10.6 / 10.8;
//     K = 7168 12288 rows 16.3 / 14.6, pairs of 8192 16.4 / 16.4, 10240 18.6 / 19.7; full scales K = 3072 10240
//     rows 7.1 / 7.1, 12288 7.4 / 8.1, K = 5120 12288 rows 10.8 / 12.3;
//   * tiled pages, whose 64 lanes per row (K > 4096) take 32 bytes of each 128-byte line, earlier:
//     K = 7168 6144 rows 12.2 / 12.0, 7168 12.8 / 13.2, 12288 16.4 / 21.6.
bool page_staged(int lay, bool full, int ns, int K, int M) {
  const int single = full ? 10240 : 12288;
  if (K <= 1024) return ns == 1 || M > 64;
  if (K <= 2048) return M > 2560;
  if (K <= 2560) return M > 6144;
  if (K <= 4096) return M > (ns == 2 ? 6144 : single);
  if (K >= 8192 && lay != kLayTiled) return ns == 1 && M > 14336;
  return M > (lay == kLayTiled ? 6144 : ns == 2 ? 8192 : single);
}

int page_gemv(int lay, bool full, int ns, const void* act, const void* act_sc, const float* x,
              const void* w0, const void* s0, const void* w1, const void* s1, void* out, int K,
              int M, void* stream) {
  if (K <= 0 || M < 0) return VIB3_ERR_BAD_COUNT;
  if (K % 32 || (lay == kLayTiled && (K % 64 || M % 16))) return VIB3_ERR_UNSUPPORTED;
  if ((!act && !x) || (act && !act_sc) || !w0 || !s0 || !out || (ns == 2 && (!w1 || !s1)))
    return VIB3_ERR_BAD_POINTER;
  if ((((uintptr_t)w0 | (uintptr_t)(ns == 2 ? w1 : w0) | (uintptr_t)(act ? act : w0)) & 15))
    return VIB3_ERR_BAD_POINTER;
  if (M == 0) return 0;
  const int G = K / 32;
  // K's limit (30816, or 23808 with f32 input): the whole decoded activation in 64 KB (what
  // k_fp4_page_staged holds)
  if ((size_t)G * 68 + (act ? 0 : (size_t)G * 20 + 32) > 65536) return VIB3_ERR_UNSUPPORTED;
  PageGemvArgs a{};
  a.act = (const uint8_t*)act; a.act_sc = (const uint8_t*)act_sc; a.x = x;
  a.w[0] = (const uint8_t*)w0; a.s[0] = (const uint16_t*)s0;
  a.w[1] = (const uint8_t*)w1; a.s[1] = (const uint16_t*)s1;
  a.out = (float*)out; a.K = K; a.M = M;
  hipStream_t st = (hipStream_t)stream;
  if (act && page_staged(lay, full, ns, K, M)) {
#define VIB3_PAGE_STAGED(LY, F, N)                                                              \
  hipLaunchKernelGGL((k_fp4_page_staged<LY, F, N>), dim3((unsigned)((M + 15) / 16)), dim3(256), \
                     (unsigned)G * 68u, st, a)
    if (lay == kLayTiled) VIB3_PAGE_STAGED(kLayTiled, false, 1);
    else if (full) VIB3_PAGE_STAGED(kLayRowSplit, true, 1);
    else if (ns == 2) VIB3_PAGE_STAGED(kLayRowSplit, false, 2);
    else VIB3_PAGE_STAGED(kLayRowSplit, false, 1);
#undef VIB3_PAGE_STAGED
    VIB3_RETURN_LAUNCH();
  }
  const PageShape p = page_shape(M, G);
  const unsigned lds = act ? 0u : (unsigned)G * 20u;
#define VIB3_PAGE_L(LY, F, N, LL, O) \
  hipLaunchKernelGGL((k_fp4_page_rows<LY, F, N, LL, O>), dim3(p.grid), dim3(p.block), lds, st, a)
#define VIB3_PAGE_GEMV(LY, F, N)                        \
  do {                                                  \
    if (p.L == 16) VIB3_PAGE_L(LY, F, N, 16, true);     \
    else if (p.L == 32) VIB3_PAGE_L(LY, F, N, 32, true); \
    else if (p.one) VIB3_PAGE_L(LY, F, N, 64, true);    \
    else VIB3_PAGE_L(LY, F, N, 64, false);              \
  } while (0)
  if (lay == kLayRowSplit && !full && ns == 1) VIB3_PAGE_GEMV(kLayRowSplit, false, 1);
  else if (lay == kLayRowSplit && !full && ns == 2) VIB3_PAGE_GEMV(kLayRowSplit, false, 2);
  else if (lay == kLayRowSplit && full && ns == 1) VIB3_PAGE_GEMV(kLayRowSplit, true, 1);
  else if (lay == kLayTiled && !full && ns == 1) VIB3_PAGE_GEMV(kLayTiled, false, 1);
  else if (lay == kLaySeq && !full && ns == 1) VIB3_PAGE_GEMV(kLaySeq, false, 1);
  else if (lay == kLaySeq && !full && ns == 2) VIB3_PAGE_GEMV(kLaySeq, false, 2);
  else return VIB3_ERR_UNSUPPORTED;
#undef VIB3_PAGE_GEMV
#undef VIB3_PAGE_L
  VIB3_RETURN_LAUNCH();
}

int scalar_gemv(bool in16, bool out16, int ns, const void* x, const void* w0, const void* s0,
                const void* w1, const void* s1, void* out, int K, int M, int bs, void* stream) {
  if (K <= 0 || M < 0 || bs <= 0) return VIB3_ERR_BAD_COUNT;
  if (K % 32 || bs % 32 || (bs & (bs - 1)) || (K / 32) % (bs / 32)) return VIB3_ERR_UNSUPPORTED;
  if ((size_t)K * 4 > 65536) return VIB3_ERR_UNSUPPORTED;
  if (!x || !w0 || !s0 || !out || (ns == 2 && (!w1 || !s1))) return VIB3_ERR_BAD_POINTER;
  if ((((uintptr_t)w0 | (uintptr_t)(ns == 2 ? w1 : w0)) & 15)) return VIB3_ERR_BAD_POINTER;
  if (M == 0) return 0;
  ScalarArgs a{};
  a.x = x; a.w[0] = (const uint8_t*)w0; a.s[0] = (const uint16_t*)s0;
  a.w[1] = (const uint8_t*)w1; a.s[1] = (const uint16_t*)s1;
  a.out = out; a.K = K; a.M = M; a.bs_shift = __builtin_ctz((unsigned)(bs / 32));
  const PageShape p = page_shape(M, K / 32);
  hipStream_t st = (hipStream_t)stream;
#define VIB3_SCALAR_L(I, O, N, LL, ONE) \
  hipLaunchKernelGGL((k_nvfp4_scalar_rows<I, O, N, LL, ONE>), dim3(p.grid), dim3(p.block), 0, st, a)
#define VIB3_SCALAR(I, O, N)                          \
  do {                                                \
    if (p.L == 16) VIB3_SCALAR_L(I, O, N, 16, true);  \
    else if (p.L == 32) VIB3_SCALAR_L(I, O, N, 32, true); \
    else if (p.one) VIB3_SCALAR_L(I, O, N, 64, true); \
    else VIB3_SCALAR_L(I, O, N, 64, false);           \
  } while (0)
  if (!in16 && out16 && ns == 1) VIB3_SCALAR(false, true, 1);
  else if (!in16 && !out16 && ns == 1) VIB3_SCALAR(false, false, 1);
  else if (in16 && out16 && ns == 1) VIB3_SCALAR(true, true, 1);
  else if (!in16 && out16 && ns == 2) VIB3_SCALAR(false, true, 2);
  else if (!in16 && !out16 && ns == 2) VIB3_SCALAR(false, false, 2);
  else return VIB3_ERR_UNSUPPORTED;
#undef VIB3_SCALAR
#undef VIB3_SCALAR_L
  VIB3_RETURN_LAUNCH();
}

}  // namespace
}  // namespace vib3

using namespace vib3;

extern "C" {

int vib3_launch_gemv_mma_nvfp4_preq(const void* act_fp4, const void* act_scales,
                                    const void* weight_packed, const void* scales, void* output,
                                    int K, int M_slice, void* stream) {
  return page_gemv(kLayRowSplit, false, 1, act_fp4, act_scales, nullptr, weight_packed, scales,
                   nullptr, nullptr, output, K, M_slice, stream);
}

int vib3_launch_gemv_mma_nvfp4_preq_fast(const void* act_fp4, const void* act_scales,
                                         const void* weight_packed, const void* scales,
                                         void* output, int K, int M_slice, void* stream) {
  return vib3_launch_gemv_mma_nvfp4_preq(act_fp4, act_scales, weight_packed, scales, output, K,
                                         M_slice, stream);
}

int vib3_launch_fused_swiglu_mma_nvfp4_preq(const void* act_fp4, const void* act_scales,
                                            const void* up_weight, const void* up_scales,
                                            const void* gate_weight, const void* gate_scales,
                                            void* output, int K, int M_slice, void* stream) {
  return page_gemv(kLayRowSplit, false, 2, act_fp4, act_scales, nullptr, up_weight, up_scales,
                   gate_weight, gate_scales, output, K, M_slice, stream);
}

int vib3_launch_fused_swiglu_mma_nvfp4_preq_fast(const void* act_fp4, const void* act_scales,
                                                 const void* up_weight, const void* up_scales,
                                                 const void* gate_weight, const void* gate_scales,
                                                 void* output, int K, int M_slice, void* stream) {
  return vib3_launch_fused_swiglu_mma_nvfp4_preq(act_fp4, act_scales, up_weight, up_scales,
                                                 gate_weight, gate_scales, output, K, M_slice,
                                                 stream);
}

int vib3_launch_gemv_mma_nvfp4_tiled(const void* act_fp4, const void* act_scales,
                                     const void* weight, const void* scales, void* output, int K,
                                     int M_slice, void* stream) {
  return page_gemv(kLayTiled, false, 1, act_fp4, act_scales, nullptr, weight, scales, nullptr,
                   nullptr, output, K, M_slice, stream);
}

int vib3_launch_gemv_scalar_nvfp4(const void* act_fp4, const void* act_scales,
                                  const void* weight_packed, const void* scales, void* output,
                                  int K, int M_slice, void* stream) {
  return page_gemv(kLayRowSplit, true, 1, act_fp4, act_scales, nullptr, weight_packed, scales,
                   nullptr, nullptr, output, K, M_slice, stream);
}

int vib3_launch_gemv_mma_nvfp4(const void* input, const void* weight_packed, const void* scales,
                               void* output, int K, int M_slice, void* stream) {
  return page_gemv(kLaySeq, false, 1, nullptr, nullptr, (const float*)input, weight_packed,
                   scales, nullptr, nullptr, output, K, M_slice, stream);
}

int vib3_launch_fused_swiglu_mma_nvfp4(const void* input, const void* up_weight,
                                       const void* up_scales, const void* gate_weight,
                                       const void* gate_scales, void* output, int K,
                                       int M_slice, void* stream) {
  return page_gemv(kLaySeq, false, 2, nullptr, nullptr, (const float*)input, up_weight,
                   up_scales, gate_weight, gate_scales, output, K, M_slice, stream);
}

int vib3_launch_partial_matmul_nvfp4(const void* input, const void* weight_packed,
                                     const void* scales, void* output, int K, int M_slice,
                                     int block_size, void* stream) {
  return scalar_gemv(false, true, 1, input, weight_packed, scales, nullptr, nullptr, output, K,
                     M_slice, block_size, stream);
}

int vib3_launch_partial_matmul_nvfp4_f32out(const void* input, const void* weight_packed,
                                            const void* scales, void* output, int K, int M_slice,
                                            int block_size, void* stream) {
  return scalar_gemv(false, false, 1, input, weight_packed, scales, nullptr, nullptr, output, K,
                     M_slice, block_size, stream);
}

int vib3_launch_partial_matmul_nvfp4_fp16in(const void* input, const void* weight_packed,
                                            const void* scales, void* output, int K, int M_slice,
                                            int block_size, void* stream) {
  return scalar_gemv(true, true, 1, input, weight_packed, scales, nullptr, nullptr, output, K,
                     M_slice, block_size, stream);
}

int vib3_launch_fused_swiglu_nvfp4(const void* input, const void* up_weight,
                                   const void* up_scales, const void* gate_weight,
                                   const void* gate_scales, void* output, int K, int M_slice,
                                   int block_size, void* stream) {
  return scalar_gemv(false, true, 2, input, up_weight, up_scales, gate_weight, gate_scales,
                     output, K, M_slice, block_size, stream);
}

int vib3_launch_fused_swiglu_nvfp4_f32out(const void* input, const void* up_weight,
                                          const void* up_scales, const void* gate_weight,
                                          const void* gate_scales, void* output, int K,
                                          int M_slice, int block_size, void* stream) {
  return scalar_gemv(false, false, 2, input, up_weight, up_scales, gate_weight, gate_scales,
                     output, K, M_slice, block_size, stream);
}

}  // extern "C"
