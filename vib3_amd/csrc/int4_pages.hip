// int4_pages.hip — INT4 pages one at a time (the launcher API) in the shapes that k_int4_rows
// (int4_gemv.hip) does not take at its rate: rows that are not 16-byte aligned, and k > 8192.
//
// k_int4_ragged — one page with unaligned rows of any k > 64 (odd k too); g a multiple of 32.
// k_down_rows   — (down_rows.h, FLAT) one page with k > 8192 and an f16 activation, where flat_down_ok.
#include "common.h"
#include "down_rows.h"
#include "kernels.h"

namespace vib3 {

// ------------------------------------------------------------------------- k_int4_ragged
//
// One page (or an up/gate pair) whose rows are not 16-byte aligned: odd k, k not a multiple of 32,
// unaligned bases. A row is ceil(k / 32) chunks of 16 bytes read where they lie (global memory takes
// unaligned 16-byte loads); the last chunk is the row's last 16 bytes, and its columns that the chunk
// before already covers meet a zero activation, as do the columns past k. So a chunk has one group
// scale (g a multiple of 32) and no load leaves the row. Activations stay f32, in registers.
//
// Bound by a launch's round trips for one page: L lanes read a row (64 / L rows per wave), each up to
// kRagJ chunks, every load of a row out at once. L is the smallest of 16, 32, 64 that takes a row in
// one pass, widened while a page gives fewer than two waves per CU. (One byte load per two columns and
// lane, as k_int4_generic: 520 x 1000 gate/up 6.9 -> 3.6 us, 520 x 1364 down 11.4 -> 3.3 us,
// 3283 x 4785 gate/up 53 -> 14.5 us. Staging the activation through LDS was slower on the small pages
// (4.2 and 4.9 us), a second set of weights in flight on all.)
constexpr int kRagJ = 4;

typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(1)));
typedef uint16_t u16_u __attribute__((aligned(1)));

__device__ __forceinline__ uint4 ld16_any(const uint8_t* p) {
  const u32x4_u v = *(__attribute__((address_space(1))) const u32x4_u*)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}

// Sum over q of x[q] * (code - 8) of the 32 codes of a chunk, in f32. Codes become f16 pairs
// exactly (0x6400 | code is 1024 + code, 0x6400 | code << 4 is 1024 + 16 code), which the mixed
// fused multiply-add takes beside the f32 activation.
__device__ __forceinline__ float ragged_dot(const uint4 w, const float (&x)[32]) {
  const uint32_t v[4] = {w.x, w.y, w.z, w.w};
  const h2 lo_off = {(half_t)-1032.0f, (half_t)-1032.0f};
  const h2 hi_mul = {(half_t)0.0625f, (half_t)0.0625f}, hi_off = {(half_t)-72.0f, (half_t)-72.0f};
  float p0 = 0.0f, p1 = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t u = v[i], t = v[i] >> 8;
    const h2 a = as_h2((u & 0x000F000Fu) | 0x64006400u) + lo_off;                              // 0, 4
    const h2 b = __builtin_elementwise_fma(as_h2((u & 0x00F000F0u) | 0x64006400u), hi_mul, hi_off);  // 1, 5
    const h2 c = as_h2((t & 0x000F000Fu) | 0x64006400u) + lo_off;                              // 2, 6
    const h2 d = __builtin_elementwise_fma(as_h2((t & 0x00F000F0u) | 0x64006400u), hi_mul, hi_off);  // 3, 7
    p0 = __builtin_fmaf(x[8 * i + 0], (float)a[0], p0);
    p1 = __builtin_fmaf(x[8 * i + 1], (float)b[0], p1);
    p0 = __builtin_fmaf(x[8 * i + 2], (float)c[0], p0);
    p1 = __builtin_fmaf(x[8 * i + 3], (float)d[0], p1);
    p0 = __builtin_fmaf(x[8 * i + 4], (float)a[1], p0);
    p1 = __builtin_fmaf(x[8 * i + 5], (float)b[1], p1);
    p0 = __builtin_fmaf(x[8 * i + 6], (float)c[1], p0);
    p1 = __builtin_fmaf(x[8 * i + 7], (float)d[1], p1);
  }
  return p0 + p1;
}

template <bool DUAL, int L, bool ONE>
__global__ __launch_bounds__(128) void k_int4_ragged(GenericArgs a) {
  constexpr int R = kWave / L, NS = DUAL ? 2 : 1;
  const int lane = lane_id(), sub = lane % L, rr = lane / L;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int K = a.K, M = a.M, pk = (K + 1) / 2, ng = (K + a.g - 1) / a.g, cpr = (K + 31) / 32;
  const int cpg = a.g / 32;  // chunks per scale group
  const int groups = (M + R - 1) / R, stride = (int)gridDim.x * 2;
  const int passes = ONE ? 1 : (cpr + L * kRagJ - 1) / (L * kRagJ);
  const uint8_t* const d[2] = {a.data0, DUAL ? a.data1 : a.data0};
  const uint8_t* const s[2] = {(const uint8_t*)a.scales0, (const uint8_t*)(DUAL ? a.scales1 : a.scales0)};
  float xv[kRagJ][32];
  uint4 w[NS][kRagJ];
  uint16_t q[NS][kRagJ];
  auto issue = [&](int row, int pass) {
#pragma unroll
    for (int j = 0; j < kRagJ; j++) {
      if ((pass * kRagJ + j) * L >= cpr) break;  // (wave-uniform)
      const int c = min((pass * kRagJ + j) * L + sub, cpr - 1);
#pragma unroll
      for (int m = 0; m < NS; m++) {
        w[m][j] = ld16_any(d[m] + (size_t)row * pk + min(16 * c, pk - 16));
        q[m][j] = *(__attribute__((address_space(1))) const u16_u*)(s[m] + 2 * ((size_t)row * ng + c / cpg));
      }
    }
  };
  // x of this lane's chunks: zero for a chunk past the row end, for columns the chunk before
  // covers and for columns past k. Regular chunks load columns 32 c ...; the row's last 16 bytes
  // are columns k - 32 ... (even k) or k - 31 ... (odd k: loaded from k - 32 and moved by one, so
  // that no load leaves x).
  auto load_x = [&](int pass) {
#pragma unroll
    for (int j = 0; j < kRagJ; j++) {
      if ((pass * kRagJ + j) * L >= cpr) break;
      const int c = (pass * kRagJ + j) * L + sub;
      const int base = min(32 * c, K - 32);
      float t[32];
      if (a.x_dt == VIB3_DT_F32) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const uint4 u = ld16_any((const uint8_t*)((const float*)a.x + base + 4 * i));
          t[4 * i] = __uint_as_float(u.x); t[4 * i + 1] = __uint_as_float(u.y);
          t[4 * i + 2] = __uint_as_float(u.z); t[4 * i + 3] = __uint_as_float(u.w);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const uint4 u = ld16_any((const uint8_t*)((const uint16_t*)a.x + base + 8 * i));
          const uint32_t v[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
          for (int k = 0; k < 8; k++) {
            const uint16_t h = (uint16_t)(v[k >> 1] >> (16 * (k & 1)));
            t[8 * i + k] = a.x_dt == VIB3_DT_F16 ? f16_to_f32(h) : bf16_to_f32(h);
          }
        }
      }
      const bool move = (K & 1) && 32 * c > K - 32;
      // first column of the chunk that is its own: 0, past the overlap, or 32 (no chunk)
      const int lo = c >= cpr ? 32 : max(32 * c - 2 * (pk - 16), 0);
#pragma unroll
      for (int i = 0; i < 32; i++) {
        const float v = move ? (i < 31 ? t[i < 31 ? i + 1 : i] : 0.0f) : t[i];
        xv[j][i] = i >= lo ? v : 0.0f;
      }
    }
  };
  auto store = [&](int row, const float (&t)[NS]) {
    const float v = DUAL ? (t[NS - 1] / (1.0f + expf(-t[NS - 1]))) * t[0] : t[0];
    if (a.out_dt == VIB3_DT_F16) ((uint16_t*)a.out)[row] = f32_to_f16_bits(v);
    else ((float*)a.out)[row] = v;
  };
  uint64_t again = 0;
  int rg = (int)blockIdx.x * 2 + wave;
  if (ONE) {
    issue(min(rg * R + rr, M - 1), 0);
    load_x(0);
  }
  for (int turn = 0; rg < groups; rg += stride, turn++) {
    const bool first = turn == 0;
    const int row = rg * R + rr;
    float acc[NS];
#pragma unroll
    for (int m = 0; m < NS; m++) acc[m] = 0.0f;
    for (int p = 0; p < passes; p++) {
      if (!ONE || !first) issue(min(row, M - 1), p);
      if (!ONE) load_x(p);
#pragma unroll
      for (int j = 0; j < kRagJ; j++) {
        if ((p * kRagJ + j) * L >= cpr) break;
#pragma unroll
        for (int m = 0; m < NS; m++)
          acc[m] = __builtin_fmaf(ragged_dot(w[m][j], xv[j]), decode_scale(q[m][j], a.sdt), acc[m]);
      }
    }
#pragma unroll
    for (int m = 0; m < NS; m++) {
      acc[m] = lanes_sum<L>(acc[m]);
      // (infinite or no number, which a sum stays once it is; a row's lanes agree)
      if (!(__builtin_fabsf(acc[m]) <= __FLT_MAX__)) again |= 1ull << (turn & 63);
    }
    if (sub == 0 && row < M) store(row, acc);
  }
  // Rows whose sums overflowed, or whose terms are no finite numbers, term by term: with |x| above
  // 2^120 a chunk's sum of x (q - 8) can overflow ahead of its scale where no x ((q - 8) scale) does.
  // (After the loop: a branch inside it cost 0.3 us per launch. A bit stands for every 64th turn.)
  if (__builtin_expect(again != 0, 0)) {
    rg = (int)blockIdx.x * 2 + wave;
    for (int turn = 0; rg < groups; rg += stride, turn++) {
      const int row = rg * R + rr;
      if (row >= M || !(again >> (turn & 63) & 1)) continue;
      float t[NS];
      for (int m = 0; m < NS; m++) {
        float v = 0.0f;
        for (int col = sub; col < K; col += L) {
          const uint8_t b = d[m][(size_t)row * pk + (col >> 1)];
          const int code = (col & 1) ? b >> 4 : b & 15;
          const uint16_t sc = *(__attribute__((address_space(1))) const u16_u*)(s[m] + 2 * ((size_t)row * ng + col / a.g));
          v = __builtin_fmaf(load_act(a.x, a.x_dt, col), (float)(code - 8) * decode_scale(sc, a.sdt), v);
        }
        t[m] = lanes_sum<L>(v);
      }
      if (sub == 0) store(row, t);
    }
  }
}

// ------------------------------------------------------------------------- host launchers

template <bool D>
static void launch_ragged_t(const GenericArgs& a, hipStream_t s) {
  const int cpr = (a.K + 31) / 32;
  int L = cpr <= 16 * kRagJ ? 16 : cpr <= 32 * kRagJ ? 32 : 64;
  while (L < 64 && L < cpr && a.M / (kWave / L) < 2 * device_cus()) L *= 2;
  const int groups = (a.M + kWave / L - 1) / (kWave / L);
  const int cap = 8 * device_cus();  // waves, two per workgroup
  const dim3 grid((unsigned)(((groups < cap ? groups : cap) + 1) / 2));
  if (L == 16) hipLaunchKernelGGL((k_int4_ragged<D, 16, true>), grid, dim3(128), 0, s, a);
  else if (L == 32) hipLaunchKernelGGL((k_int4_ragged<D, 32, true>), grid, dim3(128), 0, s, a);
  else if (cpr <= 64 * kRagJ) hipLaunchKernelGGL((k_int4_ragged<D, 64, true>), grid, dim3(128), 0, s, a);
  else hipLaunchKernelGGL((k_int4_ragged<D, 64, false>), grid, dim3(128), 0, s, a);
}

int launch_ragged(const GenericArgs& a, bool dual, hipStream_t s) {
  if (dual) launch_ragged_t<true>(a, s);
  else launch_ragged_t<false>(a, s);
  VIB3_RETURN_LAUNCH();
}

// One flat matrix of 8192 < k, f16 activation: k_down_rows with one slot. k_int4_rows would need more
// than four chunks per lane in registers, and k_int4_rows_ksplit, which splits k over two or four waves,
// reads and converts the activation once per wave: 1024 x 14336 9.4 us there, 5.1 here; 4096 x 14336 10.9 and
// 10.2; 512 x 8224 9.4 and 4.9 (pages from HBM). False where the rows and scales are not one page,
// the staged activation exceeds 64 KB, rows exceed page_magic's range, or the split kernel is faster
// (us there / here):
//   * more rows than one workgroup per CU takes, whose last workgroups run alone: 10240 x 8224 18.0 / 20.0,
//     8192 x 14336 15.6 / 16.4 (from two full rounds on the long rows' kernel wins again: 14336 x 8224
//     23.6 / 21.9, 12288 x 20480 32.6 / 30.0; 16384 x 16384 30.1 / 31.0 it does not);
//   * staging an activation that one or a few rows use: 1 x 20480 5.3 / 6.6, 4 x 28672 6.5 / 7.7;
//   * k > 20480, where two workgroups' LDS fill a CU: 5120 x 24576 18.5 / 19.4 (4096 15.7 / 14.2, 7168
//     25.3 / 21.4), 3584 x 28672 15.5 / 16.1 (1024 10.2 / 7.8), 5120 x 30816 21.6 / 26.3.
bool flat_down_ok(const RowsArgs& a) {
  const int cpr = a.K / 32, pk = a.K / 2, M = a.M;
  if (a.x_dt != VIB3_DT_F16 || cpr <= 4 * kWave || M >= 65536 || down_rows_lds(1, cpr) > 64 * 1024 ||
      (const uint8_t*)a.flat0.scales != a.flat0.data + (size_t)M * pk)
    return false;
  if (a.K <= 12288) return M <= 8192 || M >= 14336;
  if (a.K <= 16384) return M <= 7168;
  if (M <= 4) return false;
  if (a.K <= 20480) return M <= 8192 || M >= 12288;
  if (a.K <= 24576) return M <= 4096 || (M > 6144 && M <= 8192);
  return M <= 2048;
}

int launch_flat_down(const RowsArgs& a, hipStream_t s) {
  FlatDownArgs d{};
  d.h = a.x; d.h_dt = a.x_dt; d.K = a.K; d.M = a.M; d.g = a.g; d.sdt = a.sdt; d.nslots = 1;
  d.rpp = a.M; d.magic = page_magic(a.M); d.flat = a.flat0.data;
  d.out = (float*)a.out; d.out_dt = a.out_dt;
  // as few rows per wave as make one eight-wave workgroup per CU (5120 rows of k = 8224: two per wave,
  // 1.25 workgroups per CU, 13.9 us, four per wave 11.3)
  const int waves = 8 * device_cus();
  if (a.M <= waves) launch_down_rows_t<1, 4, false, true>(d, s, KTime{});
  else if (a.M <= 2 * waves) launch_down_rows_t<2, 4, false, true>(d, s, KTime{});
  else launch_down_rows_t<4, 4, false, true>(d, s, KTime{});
  VIB3_RETURN_LAUNCH();
}

}  // namespace vib3
