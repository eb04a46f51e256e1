// down_rows.h — k_down_rows, the down projection from activations staged in LDS, and its launch: the
// layer's (int4_gemv.hip) and, with FLAT, a single page's (int4_pages.hip). A header, so that each
// translation unit holds only its own instantiations: the layer's kernels are sensitive to what is
// placed beside them (with the page kernels in int4_gemv.hip the Kimi layer took about 0.5 us more).
#pragma once

#include "common.h"
#include "kernels.h"

namespace vib3 {

// Data and scale rows of row r of a paged matrix whose page (r's) starts at `base`.
__device__ __forceinline__ void page_row(const uint8_t* base, int r, int rpp, int rows,
                                         uint64_t magic, int pk, int ng, const uint8_t*& d,
                                         const uint16_t*& s) {
  const int p = (int)(((uint64_t)(uint32_t)r * magic) >> 32);
  const int rr = r - p * rpp;
  const int rows_here = min(rpp, rows - p * rpp);
  d = base + (size_t)rr * pk;
  s = (const uint16_t*)(base + (size_t)rows_here * pk) + (size_t)rr * ng;
}

// Sum over each 16-lane row of the wave; every lane gets its row's total.
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  v += dpp<0x141>(v);
  v += dpp<0x140>(v);
  return v;
}

// FLAT launches carry the page's address and the output type besides.
struct FlatDownArgs : DownArgs {
  const uint8_t* flat;
  int out_dt;
};
template <bool FLAT>
struct DownRowsArgsOf {
  typedef DownArgs type;
};
template <>
struct DownRowsArgsOf<true> {
  typedef FlatDownArgs type;
};
template <bool FLAT>
using DownRowsArgs = typename DownRowsArgsOf<FLAT>::type;

// ------------------------------------------------------------------------- k_down_rows
//
// Down projection + weighted combine with the activations of every slot staged once per
// workgroup in LDS, already in chunk_dot's pair layout (so a batch costs no conversion work).
// A wave owns a group of R output rows (64 / R lanes per row, J chunks per lane per pass) and
// walks the slots in router order, each slot in ceil(chunks / (64 / R * J)) passes over k, so
// the combine o = o + w_s * d_s happens in registers in the reference's order: no cross-wave
// reduction, no barrier in the loop. f16 intermediates whose staged form fits 64 KB of LDS;
// other shapes use k_down_combine.

template <int J>
struct DownRowsBatch {
  uint4 w[J];
  uint16_t q[J];
};

// Sum over each run of L lanes (L = 16, 32 or 64); every lane gets its run's total.
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
  v = row16_sum(v);
  if (L >= 32) v += __shfl_xor(v, 16);
  if (L >= 64) v += __shfl_xor(v, 32);
  return v;
}

#ifndef VIB3_DOWN_SCALAR_PAGES
#define VIB3_DOWN_SCALAR_PAGES 1  // (build-time switch of the scalar page-address path)
#endif
constexpr int kDownScalarSlots = 16;  // most slots whose page addresses k_down_rows keeps in SGPRs

// FLAT: one matrix at an address the host knows times one f16 vector (no tables, no weights; f16 or
// f32 output).
template <int R, int J, int NB, bool ONE, bool FLAT = false>  // ONE: the whole row in one pass (cpr <= CPP)
__global__ __launch_bounds__(512) void k_down_rows(DownRowsArgs<FLAT> a) {
  VIB3_TRACE_POINT(0);
  extern __shared__ uint4 lds[];
  constexpr int L = kWave / R;  // lanes per row
  constexpr int CPP = L * J;    // chunks per pass
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int grp = lane / L, sub = lane % L;
  const int cpr = a.K / 32, pk = a.K / 2, ng = (a.K + a.g - 1) / a.g;
  const int P = ONE ? 1 : (cpr + CPP - 1) / CPP;  // passes per slot
  const int ns = FLAT ? 1 : a.nslots, top_k = FLAT ? 0 : a.top_k;
  const int CT = ONE ? CPP : cpr;  // chunks per slot in LDS (one pass: zero past cpr)
  uint4* xq = lds;                                       // [ns][4][CT] pair words
  float* xsum = (float*)(lds + (size_t)ns * 4 * CT);     // [ns][CT] offset term

  const int G = (a.M + R - 1) / R;  // row groups
  const int g0 = (int)blockIdx.x * (int)(blockDim.x >> 6) + wave;
  // scale index of chunk c: (32 c) / g, a shift for the usual power-of-two group sizes
  const bool g_pow2 = (a.g & (a.g - 1)) == 0;
  const int g_shift = __builtin_ctz((unsigned)a.g);
  auto scale_of = [&](int c) { return g_pow2 ? (c * 32) >> g_shift : (c * 32) / a.g; };
  // lane s < nslots holds slot s's page-table row (down segment), router weight and, when
  // pages hold whole row groups, the address of the page holding this wave's rows: the loop
  // then reads no page table (a scalar table read per batch would delay every batch's loads
  // by its latency)
  const bool group_pages = FLAT || a.rpp % R == 0;
  // With the gate/up kernel's list of page addresses, whole row groups per page and few slots,
  // the page addresses come through scalar loads (one round trip, no ids), which leaves the
  // vector memory counter to the activations: those go out first, and waiting for the
  // addresses does not wait for them.
  const bool scalar_pages =
      !FLAT && VIB3_DOWN_SCALAR_PAGES && a.bases && group_pages && ns <= kDownScalarSlots;
  const int r0 = min(R * g0, a.M - 1);
  const int page0 = (int)(((uint64_t)(uint32_t)r0 * a.magic) >> 32);  // page of this wave's rows
  uint64_t my_t = 0, my_base = 0;
  if constexpr (FLAT) my_base = (uint64_t)(uintptr_t)a.flat;
  float my_w = 1.0f;
  if (!FLAT && lane < ns) {
    if (lane < top_k) my_w = a.wts[lane];
    else if (a.shared_w) my_w = a.shared_w[lane - top_k];  // sigmoid gate of a shared expert
  }
  if (!FLAT && !scalar_pages && lane < ns) {
    const uint64_t* t =
        lane < top_k ? a.routed_table + ((size_t)a.ids[lane] * 3 + 2) * a.max_pages
                     : a.shared_table + ((size_t)(lane - top_k) * 3 + 2) * a.max_pages;
    my_t = (uint64_t)(uintptr_t)t;
    if (group_pages) {
      typedef __attribute__((address_space(1))) const uint64_t gtab;
      my_base = *(gtab*)(t + page0);
    }
  }
  auto scalar_bases = [&]() {  // page addresses from the list the gate/up kernel wrote
    uint64_t bs[kDownScalarSlots];
#pragma unroll
    for (int s = 0; s < kDownScalarSlots; s++)  // slots past the last repeat it
      bs[s] = ld_table(a.bases + (size_t)min(s, ns - 1) * a.bases_stride + page0);
    __builtin_amdgcn_sched_barrier(0);  // (all loads issued before the first wait)
    uint64_t base = 0;
#pragma unroll
    for (int s = 0; s < kDownScalarSlots; s++) base = lane == s ? bs[s] : base;
    return base;
  };

  // one row group per wave (the launcher sizes the grid so); its batches are (slot, pass),
  // passes innermost
  const int n = g0 < G ? ns * P : 0;
  struct Pos { int s, p; };
  auto advance = [&](Pos q) {
    if (++q.p == P) {
      q.p = 0;
      q.s = min(q.s + 1, ns - 1);
    }
    return q;
  };
  auto rl64 = [&](uint64_t v, int l) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
  };
  // start() runs unconditionally; a batch past the end reads the intermediate (cached in
  // L2) instead of weights. Lanes past the last chunk re-read it (their x is taken as zero).
  auto start = [&](DownRowsBatch<J>& b, Pos q, bool past) {
    const uint8_t* d = nullptr;
    const uint16_t* sc = nullptr;
    if (group_pages) {  // every lane its own row of the group's page
      const uint64_t pb = rl64(my_base, q.s);
      past = past || pb == 0;  // (no address: a down stage launched before any gate/up stage)
      page_row((const uint8_t*)(uintptr_t)pb, min(R * g0 + grp, a.M - 1), a.rpp, a.M, a.magic,
               pk, ng, d, sc);
    } else {
      const MatRef m{(const uint64_t*)(uintptr_t)rl64(my_t, q.s), nullptr, nullptr, a.rpp, a.M,
                     a.magic};
#pragma unroll
      for (int r = 0; r < R; r++) {  // the rows are wave-uniform: scalar table reads
        const uint8_t* dq;
        const uint16_t* sq;
        mat_row<true>(m, min(R * g0 + r, a.M - 1), pk, ng, dq, sq);
        if (grp == r) { d = dq; sc = sq; }
      }
    }
    if (past) {
      d = (const uint8_t*)a.h;
      sc = (const uint16_t*)a.h;
    }
#pragma unroll
    for (int j = 0; j < J; j++) {
      const int c = min(q.p * CPP + sub + L * j, cpr - 1);
      b.w[j] = ld_stream(d + (uint32_t)c * 16u);
      b.q[j] = ld_u16(sc + scale_of(c));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  float o = 0.0f, acc = 0.0f;
  auto finish = [&](const DownRowsBatch<J>& b, Pos q, bool keep) {
#pragma unroll
    for (int j = 0; j < J; j++) {
      const int c0 = q.p * CPP + sub + L * j;
      const int c = ONE ? c0 : min(c0, cpr - 1);
      const uint4* xp = xq + (size_t)q.s * 4 * CT + c;
      XChunk x;
      const uint4 va = xp[0], vb = xp[CT], vc = xp[2 * CT], vd = xp[3 * CT];
      x.a[0] = as_h2(va.x); x.a[1] = as_h2(va.y); x.a[2] = as_h2(va.z); x.a[3] = as_h2(va.w);
      x.b[0] = as_h2(vb.x); x.b[1] = as_h2(vb.y); x.b[2] = as_h2(vb.z); x.b[3] = as_h2(vb.w);
      x.c[0] = as_h2(vc.x); x.c[1] = as_h2(vc.y); x.c[2] = as_h2(vc.z); x.c[3] = as_h2(vc.w);
      x.d[0] = as_h2(vd.x); x.d[1] = as_h2(vd.y); x.d[2] = as_h2(vd.z); x.d[3] = as_h2(vd.w);
      x.xs8 = xsum[q.s * CT + c];
      const float t = __builtin_fmaf(chunk_dot(b.w[j], x), decode_scale(b.q[j], a.sdt), acc);
      acc = (ONE || c0 < cpr) ? t : acc;  // one pass: x is zero past cpr
    }
    if (q.p == P - 1) {  // the slot's last pass: its row sums, rounded, into the combine
      float dsum = lanes_sum<L>(acc) * kTwo24;
      if (!FLAT && a.round_f16) dsum = (float)(half_t)dsum;
      const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_w), q.s));
      const float next = FLAT ? dsum : add_mul_rn(o, w, dsum);  // weighted_accumulate_f32 in slot order
      o = keep ? next : o;                         // (engine.rs:5262-5302)
      acc = 0.0f;
    }
  };

  // NB load buffers in a ring: while batch i is reduced, batch i+1 is loading
  DownRowsBatch<J> buf[NB];
  Pos pos[NB];
  pos[0] = Pos{0, 0};
#pragma unroll
  for (int b = 1; b < NB; b++) pos[b] = advance(pos[b - 1]);
  VIB3_TRACE_POINT(1);
  // stage the activations: each thread takes up to three chunks per pass and issues all of
  // their loads before converting any (one round trip per pass, not one per chunk)
  const char* hb = (const char*)a.h;
  const int nitem = ns * CT, bd = (int)blockDim.x;
  auto load_raw = [&](int i0, uint4 (&raw)[3][4]) {
#pragma unroll
    for (int u = 0; u < 3; u++) {
      const int i = min(i0 + u * bd, nitem - 1);
      const int sl = i / CT, c = min(i - sl * CT, cpr - 1);
      const uint4* src = (const uint4*)(hb + ((size_t)sl * a.K + (size_t)c * 32) * 2);
#pragma unroll
      for (int q = 0; q < 4; q++) raw[u][q] = src[q];
    }
  };
  auto stage = [&](int i0, const uint4 (&raw)[3][4]) {
    // Every lane takes delivery of its raw words here, outside the lane-masked region below:
    // a wait inside a region that the wave can skip would leave the compiler unsure whether
    // these loads are done, and it would then wait for every load in flight in the main loop.
#pragma unroll
    for (int u = 0; u < 3; u++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        asm volatile("" ::"v"(raw[u][q].x), "v"(raw[u][q].y), "v"(raw[u][q].z), "v"(raw[u][q].w));
#pragma unroll
    for (int u = 0; u < 3; u++) {
      const int i = i0 + u * bd;
      if (i >= nitem) break;
      const int sl = i / CT, c = i - sl * CT;
      // f16 intermediates are already f16 pairs: the pair layout is a permutation of the
      // words ((x0,x4) (x1,x5) (x2,x6) (x3,x7) of each 8), and the offset term the sum of
      // the 32 values in index order (make_chunk's numbers exactly, without its conversions)
      uint32_t A[4], B[4], C[4], D[4];
      float sum = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const uint32_t w[4] = {raw[u][q].x, raw[u][q].y, raw[u][q].z, raw[u][q].w};
        A[q] = (w[0] & 0xffffu) | (w[2] << 16);
        B[q] = (w[0] >> 16) | (w[2] & 0xffff0000u);
        C[q] = (w[1] & 0xffffu) | (w[3] << 16);
        D[q] = (w[1] >> 16) | (w[3] & 0xffff0000u);
#pragma unroll
        for (int j = 0; j < 4; j++) {
          sum += f16_to_f32((uint16_t)(w[j] & 0xffff));
          sum += f16_to_f32((uint16_t)(w[j] >> 16));
        }
      }
      const bool in = c < cpr;  // (selected word by word: a select of whole vectors went
                                // through scratch memory)
      auto word4 = [&](const uint32_t (&v)[4]) {
        return make_uint4(in ? v[0] : 0u, in ? v[1] : 0u, in ? v[2] : 0u, in ? v[3] : 0u);
      };
      uint4* xp = xq + (size_t)sl * 4 * CT + c;
      xp[0] = word4(A);
      xp[CT] = word4(B);
      xp[2 * CT] = word4(C);
      xp[3 * CT] = word4(D);
      xsum[sl * CT + c] = in ? 8.0f * kTwoM24 * sum : 0.0f;
    }
  };
  {
    // first pass, every thread (indices clamped): the first weight batches go out behind the
    // (cached) activations, so waiting for the activations does not wait for the weights
    uint4 raw[3][4];
    load_raw((int)threadIdx.x, raw);
    if (scalar_pages) {
      __builtin_amdgcn_sched_barrier(0);  // (the activation loads issue first)
      my_base = scalar_bases();
    }
    // (also for a wave with no batches: every position is valid, and a branch here would make
    // the waits below count for both cases, i.e. wait for the weights too)
#pragma unroll
    for (int b = 0; b + 1 < NB; b++) start(buf[b], pos[b], false);  // rows clamp to M - 1
#ifdef VIB3_TRACE
    VIB3_TRACE_POINT(7);  // first batches issued
#pragma unroll
    for (int u = 0; u < 3; u++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        asm volatile("" ::"v"(raw[u][q].x), "v"(raw[u][q].y), "v"(raw[u][q].z), "v"(raw[u][q].w));
    VIB3_TRACE_POINT(6);  // activations arrived
#endif
    stage((int)threadIdx.x, raw);
  }
  for (int i0 = (int)threadIdx.x + 3 * bd; i0 < nitem; i0 += 3 * bd) {
    uint4 raw[3][4];
    load_raw(i0, raw);
    stage(i0, raw);
  }
  __syncthreads();
  VIB3_TRACE_POINT(2);
  if (n == 0) return;
  // The loop always runs whole rounds of NB batches, and a batch past the end is reduced like
  // the others and then dropped (a select, not a branch): an exit between two batches would
  // give the loop head a path on which a buffer is still loading, and the compiler would then
  // wait there for every load in flight.
  for (int k = 0; k < n; k += NB) {
#pragma unroll
    for (int b = 0; b < NB; b++) {
      // refill the buffer consumed last with batch k + b + NB - 1
      const int nb = (b + NB - 1) % NB;
      pos[nb] = advance(pos[(nb + NB - 1) % NB]);
      // (the explicit wait: see k_int4_rows; here it keeps the compiler's count exact with
      // the past-the-end batches, which read the cached intermediate instead of weights)
      // (batch b's loads done: at most the NB - 2 batches issued after it still loading)
      VIB3_WAIT_VM((NB - 2) * 2 * J);
      start(buf[nb], pos[nb], k + b + NB - 1 >= n);
      finish(buf[b], pos[b], k + b < n);
#ifdef VIB3_TRACE
      if (k + b == 0) VIB3_TRACE_POINT(4);  // first batch reduced
#endif
    }
  }
  VIB3_TRACE_POINT(5);
  // stored after the loop: a store inside it would share the load counter with the weight
  // loads, and the compiler then waits for all of them at the loop head
  const int r = R * g0 + grp;
  if constexpr (FLAT) {
    if (sub == 0 && r < a.M) {
      if (a.out_dt == VIB3_DT_F16) ((uint16_t*)a.out)[r] = f32_to_f16_bits(o);
      else a.out[r] = o;
    }
    return;
  }
  if (sub == 0 && r < a.M) a.out[r] = a.residual ? a.residual[r] + o : o;  // engine.rs:5302
  advance_router_tag(a.gen_word);
  VIB3_TRACE_POINT(3);
}

// ------------------------------------------------------------------------- launch

#ifndef VIB3_DOWN_WAVES
#define VIB3_DOWN_WAVES 0
#endif
static int knob(int v, int dflt) { return v > 0 ? v : dflt; }
#ifndef VIB3_DOWN_ROWS_BUFFERS
#define VIB3_DOWN_ROWS_BUFFERS 2  // load buffers per wave (build-time tuning knob)
#endif
constexpr int kDownRowsBuffers = VIB3_DOWN_ROWS_BUFFERS;

// LDS bytes of k_down_rows: per slot, every chunk's 4 pair words and one offset term.
static size_t down_rows_lds(int nslots, int chunks) {
  return (size_t)nslots * chunks * (64 + 4);
}

template <int R, int J, bool ONE, bool FLAT = false>
static void launch_down_rows_t(DownRowsArgs<FLAT>& a, hipStream_t s, KTime t) {
  // One row group per wave, and as many waves per workgroup as make one workgroup per CU
  // (2..8): every CU streams the same share of the weights, and stages the activations once.
  // (Four-wave workgroups left some CUs two workgroups and others one.)
  const int groups = (a.M + R - 1) / R;
  int wpb = knob(VIB3_DOWN_WAVES, (groups + device_cus() - 1) / device_cus());
  wpb = wpb < 2 ? 2 : wpb > 8 ? 8 : wpb;
  const int blocks = (groups + wpb - 1) / wpb;
  const int chunks = ONE ? kWave / R * J : a.K / 32;
  hipExtLaunchKernelGGL((k_down_rows<R, J, kDownRowsBuffers, ONE, FLAT>), dim3((unsigned)blocks),
                        dim3(64 * wpb), (unsigned)down_rows_lds(a.nslots, chunks), s, t.start,
                        t.stop, 0, a);
}

}  // namespace vib3
