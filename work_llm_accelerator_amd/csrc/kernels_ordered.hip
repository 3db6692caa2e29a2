// ORDERED kernels: bit-exact restatement of the reference host arithmetic on gfx950.
//
// The reference evaluates every output with one serial fp32 chain (qwen_decode_attention_kernel.cpp
// :62-98 and its prefill twins), so these kernels parallelise only across independent outputs
// (rows, tokens, heads, head dims) and keep each chain serial, in the reference order, with no
// FMA contraction (this file is built with -ffp-contract=off).
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <type_traits>

#include "kernels.hpp"
#include "qwen_device_math.hpp"
#include "runtime.hpp"

namespace qwen {

// ---------------------------------------------------------------------------------------------
// Serial chains.  A chain of dependent adds costs 4.15 cycles per step on one wave (register operands),
// and every other instruction of that wave 4 more (a 16-byte LDS read about 8), so each kernel below
// gives its chains a wave that does nothing but add: the products are formed by other waves (or by the
// matrix cores) and reach it through LDS.  One read feeds as many adds as the lanes can hold: the lanes
// of a 16-lane row hold consecutive pieces of a chain, which the adds take through DPP lane moves.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ void schedule_fence() {
  asm volatile("" ::: "memory");  // no load moves across it
  __builtin_amdgcn_sched_barrier(0);
}
template <class T>
__device__ __forceinline__ void pin(T& v) {  // v is computed here, neither before nor after
  asm volatile("" : "+v"(v));
}

// 16 steps of four chains per row: lanes 0-3 of each 16-lane row hold the chains' sums and the first four
// values, lanes 4-7 the next four, and so on (the other lanes' sums mean nothing).  row_ror:12 gives a lane
// the value of the lane four on, and the four plain adds keep a DPP read clear of a register that the VALU
// has just written.
__device__ __forceinline__ void add16_rows(float& acc, const float4& v) {
#define QWEN_ADD4(OP, CTRL)                                                                             \
  OP " %0, %1, %0 " CTRL "\n\t" OP " %0, %2, %0 " CTRL "\n\t" OP " %0, %3, %0 " CTRL "\n\t" OP " %0, %4, %0 " CTRL "\n\t"
  asm volatile(QWEN_ADD4("v_add_f32", "") QWEN_ADD4("v_add_f32_dpp", "row_ror:12 row_mask:0xf bank_mask:0xf")
                   QWEN_ADD4("v_add_f32_dpp", "row_ror:8 row_mask:0xf bank_mask:0xf")
                       QWEN_ADD4("v_add_f32_dpp", "row_ror:4 row_mask:0xf bank_mask:0xf")
               : "+v"(acc)
               : "v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w));
#undef QWEN_ADD4
}

// One chain, replicated in every row: step n of a 16-lane row's values takes lane n's by row_newbcast.
// v_fmac by 1.0 is the add (f64 has no DPP add); a double pair per lane, 32 steps.
__device__ __forceinline__ void add32_bcast(double& acc, const double2& v, double one) {
#define QWEN_STEP(N)                                                                  \
  "v_fmac_f64_dpp %0, %1, %3 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"      \
  "v_fmac_f64_dpp %0, %2, %3 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"
  asm volatile("s_nop 1\n\t" QWEN_STEP(0) QWEN_STEP(1) QWEN_STEP(2) QWEN_STEP(3) QWEN_STEP(4) QWEN_STEP(5)
                   QWEN_STEP(6) QWEN_STEP(7) QWEN_STEP(8) QWEN_STEP(9) QWEN_STEP(10) QWEN_STEP(11) QWEN_STEP(12)
                       QWEN_STEP(13) QWEN_STEP(14) QWEN_STEP(15) "s_nop 0"
               : "+v"(acc)
               : "v"(v.x), "v"(v.y), "v"(one));
#undef QWEN_STEP
}
__device__ __forceinline__ void add64_bcast(float& acc, const float4& v) {
#define QWEN_STEP(N)                                                                  \
  "v_add_f32_dpp %0, %1, %0 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"       \
  "v_add_f32_dpp %0, %2, %0 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"       \
  "v_add_f32_dpp %0, %3, %0 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"       \
  "v_add_f32_dpp %0, %4, %0 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"
  asm volatile("s_nop 1\n\t" QWEN_STEP(0) QWEN_STEP(1) QWEN_STEP(2) QWEN_STEP(3) QWEN_STEP(4) QWEN_STEP(5)
                   QWEN_STEP(6) QWEN_STEP(7) QWEN_STEP(8) QWEN_STEP(9) QWEN_STEP(10) QWEN_STEP(11) QWEN_STEP(12)
                       QWEN_STEP(13) QWEN_STEP(14) QWEN_STEP(15) "s_nop 0"
               : "+v"(acc)
               : "v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w));
#undef QWEN_STEP
}

// acc + v[0] + v[1] + ... left to right, v in LDS (16-byte aligned), N values a multiple of 64 (32: double);
// a whole wave, every lane gets the sum.
template <int N>
__device__ __forceinline__ float chain_add(float acc, const float* v) {
  static_assert(N % 64 == 0, "whole row reads");
  const float4* p = reinterpret_cast<const float4*>(v) + (threadIdx.x & 15);
  constexpr int kReads = N / 64, kAhead = kReads < 2 ? kReads : 2;
  float4 a[kAhead];
#pragma unroll
  for (int j = 0; j < kAhead; ++j) a[j] = p[16 * j];
  schedule_fence();
#pragma unroll
  for (int q = 0; q < kReads; ++q) {
    const float4 c = a[q % kAhead];
    if (q + kAhead < kReads) a[q % kAhead] = p[16 * (q + kAhead)];
    add64_bcast(acc, c);
    schedule_fence();
  }
  return acc;
}

template <int N>
__device__ __forceinline__ double chain_add(double acc, const double* v) {
  static_assert(N % 32 == 0, "whole row reads");
  const double2* p = reinterpret_cast<const double2*>(v) + (threadIdx.x & 15);
  constexpr int kReads = N / 32, kAhead = 2;
  double2 a[kAhead];
#pragma unroll
  for (int j = 0; j < kAhead; ++j) a[j] = p[16 * j];
  schedule_fence();
#pragma unroll 8
  for (int q = 0; q < kReads; ++q) {
    const double2 c = a[q % kAhead];
    if (q + kAhead < kReads) a[q % kAhead] = p[16 * (q + kAhead)];
    add32_bcast(acc, c, 1.0);
    schedule_fence();
  }
  return acc;
}

// ---------------------------------------------------------------------------------------------
// RMSNorm.  decode: double serial sum (qwen_decode_attention_kernel.cpp:13-27);
// prefill: float serial sum + approx_sqrt (qwen_prefill_attention_kernel.cpp:112-126).
// All threads form the squares (the square of a float is exact in double, so adding the finished
// square is the reference's step); wave 0 adds them in order.  Bound by the 1536-step chain: 8.9 us
// for 7 decode rows (20.5 us when one thread also loaded and multiplied), 8.9 us for 128 prefill rows (15.3).
// grid.x = tokens, block = 256.
// ---------------------------------------------------------------------------------------------
struct RmsScratch {
  double sq[QWEN_HIDDEN];  // squares (decode), or floats in the same storage (prefill)
  double inv_d;
  float inv_f;
};

// The row x[1536] into xs (LDS) normalized with w, by every thread of the block (at least 64).
__device__ __forceinline__ void rms_row_ordered(const float* __restrict__ x, const float* __restrict__ w,
                                                float* __restrict__ xs, RmsScratch& sc, bool prefill) {
  const int n = blockDim.x;
  float* sqf = reinterpret_cast<float*>(sc.sq);
  for (int d = threadIdx.x; d < QWEN_HIDDEN; d += n) {
    const float v = x[d];
    xs[d] = v;
    if (prefill)
      sqf[d] = v * v;
    else
      sc.sq[d] = (double)v * (double)v;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    __builtin_amdgcn_s_setprio(3);
    if (prefill) {
      float ms = chain_add<QWEN_HIDDEN>(0.0f, sqf);
      ms /= (float)QWEN_HIDDEN;
      if (threadIdx.x == 0) sc.inv_f = 1.0f / approx_sqrt(ms + QWEN_RMS_EPS);
    } else {
      double ms = chain_add<QWEN_HIDDEN>(0.0, sc.sq);
      ms /= (double)QWEN_HIDDEN;
      if (threadIdx.x == 0) sc.inv_d = 1.0 / __dsqrt_rn(ms + (double)QWEN_RMS_EPS);
    }
    __builtin_amdgcn_s_setprio(0);
  }
  __syncthreads();
  if (prefill) {
    const float inv = sc.inv_f;
    for (int d = threadIdx.x; d < QWEN_HIDDEN; d += n) xs[d] = xs[d] * inv * w[d];
  } else {
    const double inv = sc.inv_d;
    for (int d = threadIdx.x; d < QWEN_HIDDEN; d += n) xs[d] = (float)((double)xs[d] * inv * (double)w[d]);
  }
  __syncthreads();
}

__global__ void __launch_bounds__(256) rmsnorm_ordered_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                              float* __restrict__ y, int prefill) {
  __shared__ __align__(16) RmsScratch sc;
  __shared__ __align__(16) float xs[QWEN_HIDDEN];
  const size_t row = (size_t)blockIdx.x * QWEN_HIDDEN;
  rms_row_ordered(x + row, w, xs, sc, prefill != 0);
  for (int d = threadIdx.x; d < QWEN_HIDDEN; d += 256) y[row + d] = xs[d];
}

// ---------------------------------------------------------------------------------------------
// Serial INT4 projection (project_tiled, qwen_decode_attention_kernel.cpp:62-98):
//   y[t][o] = (residual[t][o] +) ( bias[o] + x[t][0]*w(o,0) + x[t][1]*w(o,1) + ... )  left to right,
//   w(o,i) = (float)int4(o,i) * scale[o], each product rounded before it is added.
// The rows come in up to three matrices that share the input (q, k, v), or as the gate/up pair, whose
// SiLU(gate) * up is formed in the epilogue (decode: host-compatible expf, qwen_decode_mlp_kernel.cpp:
// 79-81, 113-115; prefill: approx_exp, qwen_prefill_mlp_kernel.cpp:256-258, 318-320).
// ---------------------------------------------------------------------------------------------

// The 8 weights (float)int4 * s of one packed word.  v_cvt_off_f32_i4 gives int4 / 16 of a byte's low
// nibble in one instruction, so the weight is one more multiplication, by 16 s: the same rounded value,
// as long as 16 s does not overflow where s does not (`plain`; otherwise the factor is put back first).
__device__ __forceinline__ bool plain_scale(float s) { return __all(fabsf(s) < 0x1p120f); }

__device__ __forceinline__ void dequant8(uint32_t word, float s, bool plain, float* __restrict__ w) {
  uint32_t high = word >> 4;
  asm("" : "+v"(high));  // one shift for the four odd nibbles, not one extraction each
  const float lo[4] = {__builtin_amdgcn_cvt_off_f32_i4(word), __builtin_amdgcn_cvt_off_f32_i4((word >> 8) & 0xff),
                       __builtin_amdgcn_cvt_off_f32_i4((word >> 16) & 0xff), __builtin_amdgcn_cvt_off_f32_i4(word >> 24)};
  const float hi[4] = {__builtin_amdgcn_cvt_off_f32_i4(high), __builtin_amdgcn_cvt_off_f32_i4((high >> 8) & 0xff),
                       __builtin_amdgcn_cvt_off_f32_i4((high >> 16) & 0xff), __builtin_amdgcn_cvt_off_f32_i4(high >> 24)};
  if (plain) {
    const float s16 = 16.0f * s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[2 * i] = lo[i] * s16;
      w[2 * i + 1] = hi[i] * s16;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[2 * i] = (lo[i] * 16.0f) * s;
      w[2 * i + 1] = (hi[i] * 16.0f) * s;
    }
  }
}

// Barriers of the product rings below: a wave that wrote products waits for its LDS writes, the adds'
// wave (whose reads ahead stay in flight) does not.
__device__ __forceinline__ void ring_publish() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void ring_wait() { asm volatile("s_barrier" ::: "memory"); }

// The matrix that holds row `row` of the concatenation seg[0] | seg[1] | seg[2] (by value: the choice is
// a few scalar selects).
__device__ __forceinline__ OrdSegment pick_segment(const OrdProject& a, int row) {
  const bool s0 = row < a.seg[1].row0, s1 = row < a.seg[2].row0;
  OrdSegment g;
  g.w = s0 ? a.seg[0].w : s1 ? a.seg[1].w : a.seg[2].w;
  g.scale = s0 ? a.seg[0].scale : s1 ? a.seg[1].scale : a.seg[2].scale;
  g.bias = s0 ? a.seg[0].bias : s1 ? a.seg[1].bias : a.seg[2].bias;
  g.y = s0 ? a.seg[0].y : s1 ? a.seg[1].y : a.seg[2].y;
  g.stride = s0 ? a.seg[0].stride : s1 ? a.seg[1].stride : a.seg[2].stride;
  g.row0 = s0 ? 0 : s1 ? a.seg[1].row0 : a.seg[2].row0;
  return g;
}

// One token (grid.y = 1) or tokens blockIdx.y, at most a few: bound by the chain, 4 cycles per input.
// A block owns R rows: R / 16 waves add, 16 chains each, and four waves form the products (weights
// prefetched PD chunks ahead in registers, the input row in LDS).  A ring of three product chunks: at
// barrier c the chunks up to c + 1 are finished, so the adding waves read ahead across the chunk
// boundary while chunk c + 2 is formed.
// R = 16: 96 to 128 blocks, 1120 for the gate/up pair (8 rows of each matrix a block, so that SiLU * up
// needs no further launch).  NORM: the input row is RMS-normalized (decode) by every block, a 1536-step
// f64 chain that a launch of its own would also take, plus the launch.
// One token, traced in a resident decode step, before (one thread per output row that also unpacked, scaled and
// multiplied; 6 blocks for 1536 rows) and now: q/k/v with the norm 121 -> 13.1 us (three launches and the norm's
// before), o 36 -> 7.8 us, gate/up with the norm 93 -> 20.2 us, down (8960 steps) 196 -> 31.4 us.
template <int R, int KC, int PD, int K, bool NORM, bool GU>
__global__ void __launch_bounds__(256 + 4 * R) project_chain_kernel(OrdProject a) {
  constexpr int kAdders = 4 * R;             // threads of the adding waves
  constexpr int kPitch = KC + 4;
  constexpr int kWords = KC / 8;             // packed words of one row and chunk
  constexpr int NW = R * KC / 8 / 256;       // words per producer thread and chunk
  constexpr int kRowStep = 256 / kWords;     // rows between a thread's words
  constexpr int nc = K / KC;
  static_assert(NW * 256 * 8 == R * KC && kRowStep * NW == R, "producer split");
  static_assert(!NORM || K == QWEN_HIDDEN, "the norm covers a 1536-wide row");
  constexpr size_t kRing = 3 * R * kPitch * sizeof(float);
  // the norm's scratch is dead before the ring is first written
  __shared__ __align__(16) char lds[NORM && sizeof(RmsScratch) > kRing ? sizeof(RmsScratch) : kRing];
  __shared__ __align__(16) float xs[K];
  __shared__ float ups[GU ? R / 2 : 1];
  float* prod = reinterpret_cast<float*>(lds);
  const int tid = threadIdx.x;
  const int t = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool adder = wave < R / 16;
  const int pt = tid - kAdders;
  constexpr size_t row_bytes = (size_t)K / 2;
  // producers: word pt % kWords of rows pt / kWords + kRowStep * j
  const uint32_t* wptr[NW];
  float sc[NW];
  uint32_t wr[PD][NW];
  bool plain = true;
  if (!adder) {
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      const int r = pt / kWords + kRowStep * j;
      // gate/up: rows 0..R/2-1 are gate's, the others up's
      const OrdSegment g = GU ? (r < R / 2 ? a.seg[0] : a.seg[1]) : pick_segment(a, (int)blockIdx.x * R);
      const int row = GU ? (int)blockIdx.x * (R / 2) + r % (R / 2) : (int)blockIdx.x * R + r - g.row0;
      wptr[j] = reinterpret_cast<const uint32_t*>(g.w + (size_t)row * row_bytes) + pt % kWords;
      sc[j] = g.scale[row];
#pragma unroll
      for (int d = 0; d < PD; ++d) wr[d][j] = d < nc ? wptr[j][d * kWords] : 0u;
    }
  }
  if (NORM) {
    rms_row_ordered(a.x + (size_t)t * K, a.norm_w, xs, *reinterpret_cast<RmsScratch*>(lds), false);
  } else {
    for (int d = tid; d < K; d += 256 + kAdders) xs[d] = a.x[(size_t)t * K + d];
    __syncthreads();
  }
  if (!adder) {
#pragma unroll
    for (int j = 0; j < NW; ++j) plain = plain && plain_scale(sc[j]);
    float* buf = prod;
    for (int c0 = 0; c0 < nc; c0 += PD) {
#pragma unroll
      for (int d = 0; d < PD; ++d) {
        const int c = c0 + d;
        if (c < nc) {
          const float4* xp = reinterpret_cast<const float4*>(xs + c * KC + (pt % kWords) * 8);
          const float4 x0 = xp[0], x1 = xp[1];
#pragma unroll
          for (int j = 0; j < NW; ++j) {
            float w[8];
            dequant8(wr[d][j], sc[j], plain, w);
            float4* o = reinterpret_cast<float4*>(buf + (pt / kWords + kRowStep * j) * kPitch + (pt % kWords) * 8);
            o[0] = make_float4(x0.x * w[0], x0.y * w[1], x0.z * w[2], x0.w * w[3]);
            o[1] = make_float4(x1.x * w[4], x1.y * w[5], x1.z * w[6], x1.w * w[7]);
            if (c + PD < nc) wr[d][j] = wptr[j][(c + PD) * kWords];
          }
          buf = buf == prod + 2 * R * kPitch ? prod : buf + R * kPitch;
          if (c > 0) ring_publish();  // barrier c - 1
        }
      }
    }
    ring_publish();  // barrier nc - 1
    if (GU) ring_publish();
    return;
  }
  // chain 4 * (lane / 16) + lane % 4 of this wave, its values 4 * (lane % 16 / 4) on of each 16
  const int lane = tid & 63, chain = wave * 16 + (lane >> 4) * 4 + (lane & 3);
  float acc = 0.0f;
  __builtin_amdgcn_s_setprio(3);
  const OrdSegment g = GU ? a.seg[0] : pick_segment(a, (int)blockIdx.x * R);
  const int row = GU ? (int)blockIdx.x * (R / 2) + chain : (int)blockIdx.x * R + chain - g.row0;
  if (!GU && g.bias) acc = g.bias[row];
  constexpr int kAhead = 4, kReads = KC / 16;
  const float* mine = prod + chain * kPitch + (lane & 12);
  const float* cur = mine;
  float4 q[kAhead];
  ring_wait();  // barrier 0
#pragma unroll
  for (int j = 0; j < kAhead; ++j) q[j] = *reinterpret_cast<const float4*>(cur + 16 * j);
  int next_buf = 1;
  for (int c = 0; c < nc; ++c) {
    const float* next = mine + next_buf * R * kPitch;
#pragma unroll
    for (int i = 0; i < kReads; ++i) {
      const float4 v = q[i % kAhead];
      // (after the last chunk: a stale chunk of the ring, not added)
      q[i % kAhead] =
          *reinterpret_cast<const float4*>(i + kAhead < kReads ? cur + 16 * (i + kAhead) : next + 16 * (i + kAhead - kReads));
      add16_rows(acc, v);
      schedule_fence();
    }
    cur = next;
    next_buf = next_buf == 2 ? 0 : next_buf + 1;
    if (c + 1 < nc) ring_wait();  // barrier c + 1
  }
  const bool owner = (lane & 12) == 0;
  if (GU) {
    if (owner && chain >= R / 2) ups[chain - R / 2] = acc;
    ring_publish();
    if (owner && chain < R / 2)
      a.seg[0].y[(size_t)t * a.seg[0].stride + row] = (a.prefill ? silu_prefill(acc) : silu_decode(acc)) * ups[chain];
  } else if (owner) {
    const size_t idx = (size_t)t * g.stride + row;
    g.y[idx] = a.residual ? a.residual[idx] + acc : acc;
  }
}

// Several tokens: bound by the VALU, one add per product.  The products come from the matrix cores:
// v_mfma_f32_4x4x1 (16x16x1) is an outer product, whose fma with -0 is the rounded product itself, sign
// of zero and denormals included (checked bit for bit against v_mul_f32 on gfx950), so the VALU is left
// with the ordered adds: one per product instead of two and the unpacking.
// A block of four waves owns 64 rows (lane = row in the 4x4x1 form) and 4 * TT tokens, TT per wave.
// Chunks of 64 inputs: all threads dequantize the block's weights into LDS once for the four waves; a
// wave's own inputs stay in its registers (16 bytes per lane hold 64 inputs of 4 tokens, or 16 of 16, and
// the products' broadcast control picks the lanes of one input), both prefetched PD chunks ahead.  A ring
// of three chunks and one barrier per chunk, as above: while chunk c is consumed chunk c + 1 is finished,
// so that weight reads run kAhead groups of four inputs ahead, and each group's products one group ahead
// of their adds, across the chunk boundary.  STAGERS: four more waves do the dequantization, for launches
// of one block per CU, where it would stand in the way of the only wave on each SIMD.  TT = 1, 2, 4, 8 (4x4x1) or 16 (16x16x1): launch_mfma.
// The products cost the SIMD 2 cycles per token and input for 64 rows beside the add's 4 (a matrix
// instruction of 8 cycles makes 4 tokens' products; it does not overlap the VALU), against 4 + 4 and the
// weight's unpacking on the VALU.  One layer of 128 tokens, traced: q/k/v 405 -> 26 us, o 138 -> 26, gate/up
// 319 -> 152, down 784 -> 128 us.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kMmRows = 64;

template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// At least two waves per SIMD keeps the products in VGPRs (in AGPRs each would cost a move).
template <int TT, bool GU, bool STAGERS>
__global__ void __launch_bounds__(STAGERS ? 512 : 256) __attribute__((amdgpu_waves_per_eu(2)))
project_mfma_kernel(OrdProject a) {
  constexpr int C = 64, kPitch = C + 4;
  constexpr int kTokens = 4 * TT;                 // tokens of a block
  constexpr int PD = 4;                           // chunks in flight (1536 and 8960 hold a multiple of 4)
  constexpr int kWords = C / 32;                  // packed words of a chunk that a thread stages (4 threads per row)
  constexpr int H = TT == 16 ? 1 : (TT + 3) / 4;  // 4x4x1 token groups of a wave
  constexpr int NX = TT == 16 ? C / 16 : H;       // a lane's 16-byte pieces of a chunk's inputs
  constexpr int kAhead = TT == 16 ? 2 : 4;        // groups of four inputs read ahead
  __shared__ __align__(16) float wt[3][kMmRows * kPitch];
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  const bool stager = !STAGERS || __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) == 1;
  const int K = a.in_dim, nc = K / C;
  const size_t row_bytes = (size_t)K / 2;
  const int t0 = (int)blockIdx.y * kTokens + wave * TT;  // this wave's tokens
  // the matrix of the row this thread stages, and (not GU) of the whole block
  const OrdSegment g = GU ? (tid >= 128 ? a.seg[1] : a.seg[0]) : pick_segment(a, (int)blockIdx.x * kMmRows);
  const int wrow = GU ? (int)blockIdx.x * (kMmRows / 2) + ((tid >> 2) & 31)
                      : (int)blockIdx.x * kMmRows - g.row0 + (tid >> 2);
  // this thread's C / 4 weights of a chunk: part tid % 4 of row tid / 4
  const uint32_t* wptr = reinterpret_cast<const uint32_t*>(g.w + (size_t)wrow * row_bytes) + (tid & 3) * kWords;
  const float s = g.scale[wrow];
  // 4x4x1: lane l holds inputs 4 * (l / 4) + 0..3 of token l % 4 of each group; 16x16x1: inputs 16 j + 4 * (l / 16)
  // + 0..3 of token l % 16.  Tokens past the last repeat it (not stored).
  const float4* xptr[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const int t = t0 + (TT == 16 ? (lane & 15) : 4 * h + (lane & (TT < 4 ? TT - 1 : 3)));
    xptr[h] = reinterpret_cast<const float4*>(a.x + (size_t)min(t, a.tokens - 1) * K) + (TT == 16 ? lane >> 4 : lane >> 2);
  }
  uint32_t wr[PD][kWords];
  float4 xr[PD][NX];
  auto load_w = [&](int c, int d) {
#pragma unroll
    for (int i = 0; i < kWords; ++i) wr[d][i] = wptr[c * 4 * kWords + i];
  };
  auto load_x = [&](int c, int d) {
#pragma unroll
    for (int j = 0; j < NX; ++j) xr[d][j] = TT == 16 ? xptr[0][c * (C / 4) + 4 * j] : xptr[j % H][c * (C / 4)];
  };
#pragma unroll
  for (int d = 0; d < PD; ++d) {
    if (stager) load_w(d, d);
    if (!STAGERS || !stager) load_x(d, d);
  }
  float acc[TT];
  if (TT == 16) {
    // register i: row 16 * (i / 4) + lane % 16, token 4 * (lane / 16) + i % 4
#pragma unroll
    for (int i = 0; i < TT; ++i) acc[i] = (!GU && g.bias) ? g.bias[wrow - (tid >> 2) + 16 * (i / 4) + (lane & 15)] : 0.0f;
  } else {
    const float b0 = (!GU && g.bias) ? g.bias[wrow - (tid >> 2) + lane] : 0.0f;
#pragma unroll
    for (int i = 0; i < TT; ++i) acc[i] = b0;
  }
  const bool plain = plain_scale(s);
  // chunk c's weights from register slot d into ring buffer `ring`, and the slot's next load
  auto stage = [&](int c, int d, int ring) {
    float4* o = reinterpret_cast<float4*>(wt[ring] + (tid >> 2) * kPitch + (tid & 3) * (C / 4));
#pragma unroll
    for (int i = 0; i < kWords; ++i) {
      float q[8];
      dequant8(wr[d][i], s, plain, q);
      o[2 * i] = make_float4(q[0], q[1], q[2], q[3]);
      o[2 * i + 1] = make_float4(q[4], q[5], q[6], q[7]);
    }
    if (c + PD < nc) load_w(c + PD, d);
  };
  if (stager) {
    stage(0, 0, 0);
    stage(1, 1, 1);
  }
  __syncthreads();
  if (STAGERS && stager) {
    int ring2 = 2;  // of chunk c + 2
    for (int c0 = 0; c0 < nc; c0 += PD) {
#pragma unroll
      for (int d = 0; d < PD; ++d) {
        if (c0 + d + 2 < nc) stage(c0 + d + 2, (d + 2) % PD, ring2);
        ring2 = ring2 == 2 ? 0 : ring2 + 1;
        ring_publish();
      }
    }
    return;
  }
  const int woff = lane * kPitch;
  float4 wv[kAhead];
  auto read = [&](int slot, int ring, int k4) { wv[slot] = reinterpret_cast<const float4*>(wt[ring] + woff)[k4]; };
  constexpr int kGroups = C / 4;
#pragma unroll
  for (int i = 0; i < kAhead; ++i) read(i, 0, i);
  // products of one group (4x4x1) or one input (16x16x1)
  f32x4 p4[2][H][4];
  f32x16 p16[2];
  const f32x4 zero4 = {-0.0f, -0.0f, -0.0f, -0.0f};
  f32x16 zero16;
#pragma unroll
  for (int i = 0; i < 16; ++i) zero16[i] = -0.0f;
  auto part = [](const float4& v, int k) { return k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w; };
  // group GR of a chunk whose inputs are x: 4x4x1 input 4 GR + k sits in component k of lane block GR
  auto multiply = [&](auto gr, const float4* x, int parity, int slot) {
    constexpr int GR = decltype(gr)::value;
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        p4[parity][h][k] = __builtin_amdgcn_mfma_f32_4x4x1f32(part(x[h], k), part(wv[slot], k), zero4, 4, GR, 0);
  };
  // 16x16x1 input N of a chunk: component N % 4 of piece N / 16, lane block N / 4 % 4
  auto multiply16 = [&](auto in, const float4* x, int slot) {
    constexpr int N = decltype(in)::value;
    return __builtin_amdgcn_mfma_f32_16x16x1f32(part(x[TT == 16 ? N / 16 : 0], N % 4), part(wv[slot], N % 4), zero16, 2,
                                                N / 4 % 4, 0);
  };
  if constexpr (TT == 16)
    p16[0] = multiply16(std::integral_constant<int, 0>{}, xr[0], 0);
  else
    multiply(std::integral_constant<int, 0>{}, xr[0], 0, 0);
  int ring = 0;  // of chunk c
  for (int c0 = 0; c0 < nc; c0 += PD) {
#pragma unroll
    for (int d = 0; d < PD; ++d) {
      const int c = c0 + d;
      const int ring1 = ring == 2 ? 0 : ring + 1, ring2 = ring1 == 2 ? 0 : ring1 + 1;
      if (!STAGERS && c + 2 < nc) stage(c + 2, (d + 2) % PD, ring2);
      schedule_fence();
      static_for<kGroups>([&](auto gr) {
        constexpr int GR = decltype(gr)::value, slot = GR % kAhead, next = (GR + 1) % kAhead;
        constexpr bool last = GR + 1 == kGroups;
        const float4* xn = last ? xr[(d + 1) % PD] : xr[d];  // (after the last chunk: old inputs, not added)
        if constexpr (TT == 16) {
          static_for<4>([&](auto kk) {
            constexpr int k = decltype(kk)::value, N = (4 * GR + k + 1) % C;
            p16[(k + 1) & 1] = multiply16(std::integral_constant<int, N>{}, N == 0 ? xn : xr[d], k < 3 ? slot : next);
            if (k == 3) read(slot, GR + kAhead < kGroups ? ring : ring1, (GR + kAhead) % kGroups);
#pragma unroll
            for (int i = 0; i < TT; ++i) acc[i] += p16[k & 1][i];
#pragma unroll
            for (int i = 0; i < TT; ++i) pin(acc[i]);
            schedule_fence();
          });
        } else {
          multiply(std::integral_constant<int, (GR + 1) % kGroups>{}, xn, (GR + 1) & 1, next);
          read(slot, GR + kAhead < kGroups ? ring : ring1, (GR + kAhead) % kGroups);
#pragma unroll
          for (int h = 0; h < H; ++h)
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (4 * h + i < TT) acc[4 * h + i] += p4[GR & 1][h][k][i];
#pragma unroll
          for (int i = 0; i < TT; ++i) pin(acc[i]);
          schedule_fence();
        }
      });
      if (c + PD < nc) load_x(c + PD, d);
      // LDS operations of a wave finish in order: all but the last reads ahead are done, this wave's writes of
      // chunk c + 2 among them
      asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" ::"n"(kAhead) : "memory");
      ring = ring1;
    }
  }
  if constexpr (TT == 16) {
#pragma unroll
    for (int i = 0; i < (GU ? 8 : 16); ++i) {
      const int t = t0 + 4 * (lane >> 4) + (i & 3);
      if (t >= a.tokens) continue;
      if (GU) {
        const int row = (int)blockIdx.x * (kMmRows / 2) + 16 * (i / 4) + (lane & 15);
        a.seg[0].y[(size_t)t * a.seg[0].stride + row] =
            (a.prefill ? silu_prefill(acc[i]) : silu_decode(acc[i])) * acc[i + 8 < TT ? i + 8 : 0];
      } else {
        const size_t idx = (size_t)t * g.stride + (wrow - (tid >> 2) + 16 * (i / 4) + (lane & 15));
        g.y[idx] = a.residual ? a.residual[idx] + acc[i] : acc[i];
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < TT; ++i) {
      const int t = t0 + i;
      const float up = GU ? __shfl_xor(acc[i], 32) : 0.0f;
      if (t >= a.tokens) continue;
      if (GU) {
        const int row = (int)blockIdx.x * (kMmRows / 2) + lane;
        if (lane < 32)
          a.seg[0].y[(size_t)t * a.seg[0].stride + row] =
              (a.prefill ? silu_prefill(acc[i]) : silu_decode(acc[i])) * up;
      } else {
        const size_t idx = (size_t)t * g.stride + (wrow - (tid >> 2) + lane);
        g.y[idx] = a.residual ? a.residual[idx] + acc[i] : acc[i];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// RoPE + KV append for decode (qwen_decode_attention_kernel.cpp:29-42, 100-111, 206-213).
// One block of 64 threads per token b: pair p of every Q head and both K heads rotated with the
// host-computed (cos, sin) row of position pos[b]; K (rotated) and V rows written to row pos[b]
// of that token's cache.  rope: [positions][2][64] (cos row then sin row).  Positions outside
// [0, max_keys) are skipped (max_keys = the cache rows the caller sized).
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(64) rope_append_decode_kernel(float* __restrict__ q, const float* __restrict__ k,
                                                                const float* __restrict__ v, const int* __restrict__ pos,
                                                                const float* __restrict__ rope, int rope_rows_are_tokens,
                                                                float* __restrict__ k_cache, float* __restrict__ v_cache,
                                                                size_t cache_stride, int max_keys) {
  const int b = blockIdx.x;
  const int p = threadIdx.x;
  const int P = pos[b];
  if (P < 0 || P >= max_keys) return;  // position outside the cache rows the caller sized
  const float* cs = rope + (size_t)(rope_rows_are_tokens ? b : P) * 128;
  const float c = cs[p];
  const float sn = cs[64 + p];
  float* qb = q + (size_t)b * QWEN_HIDDEN;
  for (int h = 0; h < QWEN_Q_HEADS; ++h) {
    float* hp = qb + h * QWEN_HEAD_DIM;
    const float e = hp[p], od = hp[p + 64];
    hp[p] = e * c - od * sn;
    hp[p + 64] = od * c + e * sn;
  }
  float* kr = k_cache + (size_t)b * cache_stride + (size_t)P * QWEN_KV_WIDTH;
  float* vr = v_cache + (size_t)b * cache_stride + (size_t)P * QWEN_KV_WIDTH;
  const float* kb = k + (size_t)b * QWEN_KV_WIDTH;
  const float* vb = v + (size_t)b * QWEN_KV_WIDTH;
  for (int h = 0; h < QWEN_KV_HEADS; ++h) {
    const int base = h * QWEN_HEAD_DIM;
    const float e = kb[base + p], od = kb[base + p + 64];
    kr[base + p] = e * c - od * sn;
    kr[base + p + 64] = od * c + e * sn;
    vr[base + p] = vb[base + p];
    vr[base + p + 64] = vb[base + p + 64];
  }
}

// ---------------------------------------------------------------------------------------------
// RoPE for prefill, in place on the Q rows and the K cache rows of every token
// (qwen_prefill_attention_kernel.cpp:2304-2309, 2332-2337).  rope: [positions][2][64].
// grid.x = tokens, block = 64.  Token t has position t.
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(64) rope_prefill_kernel(float* __restrict__ q, float* __restrict__ k_rows,
                                                          const float* __restrict__ rope) {
  const int t = blockIdx.x;
  const int p = threadIdx.x;
  const float c = rope[(size_t)t * 128 + p];
  const float sn = rope[(size_t)t * 128 + 64 + p];
  float* qt = q + (size_t)t * QWEN_HIDDEN;
  for (int h = 0; h < QWEN_Q_HEADS; ++h) {
    float* hp = qt + h * QWEN_HEAD_DIM;
    const float e = hp[p], od = hp[p + 64];
    hp[p] = e * c - od * sn;
    hp[p + 64] = od * c + e * sn;
  }
  float* kt = k_rows + (size_t)t * QWEN_KV_WIDTH;
  for (int h = 0; h < QWEN_KV_HEADS; ++h) {
    float* hp = kt + h * QWEN_HEAD_DIM;
    const float e = hp[p], od = hp[p + 64];
    hp[p] = e * c - od * sn;
    hp[p + 64] = od * c + e * sn;
  }
}

// Prefill RoPE table (qwen_prefill_attention_kernel.cpp:128-143): inv_freq chain in float,
// angle = (float)pos * inv_freq, approx_sincos.  grid covers positions x 64 pairs.
__global__ void rope_table_prefill_kernel(float* __restrict__ rope, int first, int count) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= count * 64) return;
  const int pos = first + idx / 64;
  const int p = idx % 64;
  float inv_freq = 1.0f;
  for (int j = 0; j < p; ++j) inv_freq *= 0.8058421877614801f;
  const float angle = (float)pos * inv_freq;
  float s, c;
  approx_sincos(angle, &s, &c);
  rope[(size_t)pos * 128 + p] = c;
  rope[(size_t)pos * 128 + 64 + p] = s;
}

// ---------------------------------------------------------------------------------------------
// Two-pass softmax attention of decode tokens, one block of 128 threads per (head, token): the form without
// memory for the scores (the allocation-free dispatch).  decode_attention_context
// (qwen_decode_attention_kernel.cpp:113-162), keys 0..pos[b], scaling (float)(1/sqrt(128)), host-compatible expf.
// Pass 1 takes the max with the reference's `new > old` rule (any order gives the same value).
// Pass 2 walks the keys in ascending order in chunks of 128: lane j computes e for key base+j,
// lane 0 adds the denominators serially and lane d adds e*v[d] serially, so every sum keeps the
// reference order.  The score is recomputed in pass 2 exactly as the reference does.
// q: [tokens][1536]; cache of token b at k_cache + b*cache_stride.  Key counts are clamped to max_keys (the
// cache rows the caller sized).
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(128) attention_ordered_kernel(const float* __restrict__ q,
                                                                const float* __restrict__ k_cache,
                                                                const float* __restrict__ v_cache, size_t cache_stride,
                                                                const int* __restrict__ pos, int max_keys,
                                                                float* __restrict__ ctx) {
  __shared__ float qs[QWEN_HEAD_DIM];
  __shared__ float es[128];
  __shared__ float red[128];
  __shared__ float den_s;
  const int h = blockIdx.x;
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int kvh = h / QWEN_GROUPS;
  const int n = min(max(pos[b], 0) + 1, max_keys);
  // (float)(1.0/sqrt(128.0)) is this float, prefill's literal (bits 0x3db504f3; checked by
  // tests/test_oracle_math.py).
  const float scaling = 0.08838834764831845f;
  const float* kc = k_cache + (size_t)b * cache_stride + kvh * QWEN_HEAD_DIM;
  const float* vc = v_cache + (size_t)b * cache_stride + kvh * QWEN_HEAD_DIM;
  qs[tid] = q[(size_t)b * QWEN_HIDDEN + h * QWEN_HEAD_DIM + tid];
  __syncthreads();

  float m = -1.0e30f;
  for (int t = tid; t < n; t += 128) {
    const float* kr = kc + (size_t)t * QWEN_KV_WIDTH;
    float score = 0.0f;
    for (int d = 0; d < QWEN_HEAD_DIM; ++d) score += qs[d] * kr[d];
    const float sc = score * scaling;
    m = sc > m ? sc : m;
  }
  red[tid] = m;
  __syncthreads();
  for (int stride = 64; stride > 0; stride >>= 1) {
    if (tid < stride) {
      const float o = red[tid + stride];
      red[tid] = o > red[tid] ? o : red[tid];
    }
    __syncthreads();
  }
  m = red[0];

  float den = 0.0f;
  float acc = 0.0f;
  for (int base = 0; base < n; base += 128) {
    const int t = base + tid;
    if (t < n) {
      const float* kr = kc + (size_t)t * QWEN_KV_WIDTH;
      float score = 0.0f;
      for (int d = 0; d < QWEN_HEAD_DIM; ++d) score += qs[d] * kr[d];
      const float arg = score * scaling - m;
      es[tid] = glibc_expf(arg);
    }
    __syncthreads();
    const int cnt = min(128, n - base);
    if (tid == 0)
      for (int j = 0; j < cnt; ++j) den += es[j];
    for (int j = 0; j < cnt; ++j) acc += es[j] * vc[(size_t)(base + j) * QWEN_KV_WIDTH + tid];
    __syncthreads();
  }
  if (tid == 0) den_s = den;
  __syncthreads();
  const float dv = den_s;
  const float inv = dv > 0.0f ? 1.0f / dv : 0.0f;
  ctx[(size_t)b * QWEN_HIDDEN + h * QWEN_HEAD_DIM + tid] = acc * inv;
}

// ---------------------------------------------------------------------------------------------
// The same attention, and the prefill's (prefill_attention_context_block, qwen_prefill_attention_kernel.cpp:
// 204-289: keys 0..t, approx_exp), in two launches, with the scores of all keys kept in between (the reference
// evaluates each score twice with the same operations, so keeping it gives the same bits).
// scores: a block owns 64 keys of one KV head for QT query tokens; its key rows go through LDS once for
// the six query heads (one wave each, lane = key, the 128 products of a score added in order).  578 keys of
// one token: 5.7 + 13.1 us for the two launches (traced in a resident step), where one block per head that
// walked its keys alone took 55 us.  ROPE (one decode token): q is rotated on the way in, and the block that
// holds the new key's tile rotates that key and appends the K and V rows, instead of a launch of its own.
// scores[(token * 12 + head) * ld + key] = (q . k) * 1/sqrt(128).
// grid = (ceil(tokens / QT), 2, key tiles), block = 384.  vec: the cache rows are 16-byte aligned.
// ---------------------------------------------------------------------------------------------
struct OrdAttention {
  const float* q;
  float *k_cache, *v_cache;
  size_t cache_stride;  // floats between the sequences' caches (decode)
  const int* pos;       // decode
  int tokens, first, max_keys, prefill, past, vec;  // tokens first.. of the call
  const float *k_new, *v_new, *rope;                // ROPE
  int rope_rows_are_tokens;
  float* scores;        // of token `first` on
  int ld;
  float* ctx;
};

__device__ __forceinline__ int ord_keys(const OrdAttention& a, int b) {
  return a.prefill ? a.past + b + 1 : min(max(a.pos[b], 0) + 1, a.max_keys);
}

__device__ __forceinline__ float4 load4(const float* p, int vec) {
  return vec ? *reinterpret_cast<const float4*>(p) : make_float4(p[0], p[1], p[2], p[3]);
}

constexpr int kScoreKeys = 64, kScorePitch = QWEN_HEAD_DIM + 4;

template <int QT, bool ROPE>
__global__ void __launch_bounds__(384) scores_ordered_kernel(OrdAttention a) {
  __shared__ __align__(16) float kt[kScoreKeys * kScorePitch];
  __shared__ __align__(16) float qs[QT][QWEN_GROUPS * QWEN_HEAD_DIM];
  const int tid = threadIdx.x, lane = tid & 63, h = tid >> 6;
  const int b0 = a.first + (int)blockIdx.x * QT;
  const int kvh = blockIdx.y, key0 = (int)blockIdx.z * kScoreKeys;
  const int nq = min(QT, a.first + a.tokens - b0);
  const int nmax = ord_keys(a, b0 + nq - 1);  // the group's last token has the most keys (QT > 1: prefill)
  if (key0 >= nmax) return;
  const size_t seq = a.prefill ? 0 : (size_t)b0 * a.cache_stride;
  float* kc = a.k_cache + seq + kvh * QWEN_HEAD_DIM;
  const int P = ROPE ? a.pos[b0] : -1;
  const bool rot = ROPE && P >= 0 && P < a.max_keys;  // a position outside the cache rows: nothing rotated or written
  const float* cs = a.rope + (ROPE && rot ? (size_t)(a.rope_rows_are_tokens ? b0 : P) * QWEN_HEAD_DIM : 0);
  const int own = rot ? P - key0 : -1;  // the new key's row of this tile
  for (int e = tid; e < kScoreKeys * 32; e += 384) {
    const int r = e >> 5, part = e & 31;
    if (key0 + r < nmax && r != own)
      *reinterpret_cast<float4*>(kt + r * kScorePitch + part * 4) =
          load4(kc + (size_t)(key0 + r) * QWEN_KV_WIDTH + part * 4, a.vec);
  }
  for (int e = tid; e < nq * QWEN_GROUPS * 64; e += 384) {
    const int t = e / (QWEN_GROUPS * 64), i = e % (QWEN_GROUPS * 64), p = i & 63, hd = (i >> 6) * QWEN_HEAD_DIM;
    const float* src = a.q + (size_t)(b0 + t) * QWEN_HIDDEN + kvh * QWEN_GROUPS * QWEN_HEAD_DIM + hd;
    const float ev = src[p], od = src[p + 64];
    qs[t][hd + p] = rot ? ev * cs[p] - od * cs[64 + p] : ev;
    qs[t][hd + p + 64] = rot ? od * cs[p] + ev * cs[64 + p] : od;
  }
  if (ROPE && own >= 0 && own < kScoreKeys && tid < 64) {
    const float* kb = a.k_new + (size_t)b0 * QWEN_KV_WIDTH + kvh * QWEN_HEAD_DIM;
    const float* vb = a.v_new + (size_t)b0 * QWEN_KV_WIDTH + kvh * QWEN_HEAD_DIM;
    const float ev = kb[tid], od = kb[tid + 64], c = cs[tid], sn = cs[64 + tid];
    const float k0 = ev * c - od * sn, k1 = od * c + ev * sn;
    kt[own * kScorePitch + tid] = k0;
    kt[own * kScorePitch + tid + 64] = k1;
    float* kr = kc + (size_t)P * QWEN_KV_WIDTH;
    float* vr = a.v_cache + seq + kvh * QWEN_HEAD_DIM + (size_t)P * QWEN_KV_WIDTH;
    kr[tid] = k0;
    kr[tid + 64] = k1;
    vr[tid] = vb[tid];
    vr[tid + 64] = vb[tid + 64];
  }
  __syncthreads();
  float sc[QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) sc[t] = 0.0f;
  const float4* kl = reinterpret_cast<const float4*>(kt + lane * kScorePitch);
#pragma unroll 4
  for (int d = 0; d < QWEN_HEAD_DIM / 4; ++d) {
    const float4 k = kl[d];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const float4 q = *reinterpret_cast<const float4*>(&qs[t][h * QWEN_HEAD_DIM + d * 4]);
      sc[t] += q.x * k.x;
      sc[t] += q.y * k.y;
      sc[t] += q.z * k.z;
      sc[t] += q.w * k.w;
    }
  }
  const int key = key0 + lane;
#pragma unroll
  for (int t = 0; t < QT; ++t)
    if (t < nq && key < ord_keys(a, b0 + t))
      a.scores[((size_t)(b0 - a.first + t) * QWEN_Q_HEADS + kvh * QWEN_GROUPS + h) * a.ld + key] =
          sc[t] * 0.08838834764831845f;
}

// Softmax and P.V over kept scores, one block per (head, token).  Tiles of 64 keys: waves 4-7 form the
// products e_j * v_j[d] of tile i (V rows prefetched DEPTH tiles ahead in registers) and wave 3 the
// exponentials of tile i + 2, while waves 0-1 (lane = dim) and wave 2 (the denominator) add tile i - 1
// in key order from LDS: bound by that chain of one add per key, and by the V rows' latency where a
// history has few tiles.  DEPTH 4 for decode (12 blocks per token, their CUs to themselves), 2 for prefill
// (two blocks per CU).  grid = (12, tokens), block = 512.
constexpr int kPvTile = 64;

template <int DEPTH>
__global__ void __launch_bounds__(512) softmax_pv_ordered_kernel(OrdAttention a) {
  __shared__ __align__(16) float prod[2][kPvTile * QWEN_HEAD_DIM];  // [key][dim]
  __shared__ __align__(16) float es[4][kPvTile];
  __shared__ float red[8];
  __shared__ float den_s;
  const int h = blockIdx.x, b = a.first + (int)blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = ord_keys(a, b);
  const int nt = (n + kPvTile - 1) / kPvTile;
  const float* sc = a.scores + ((size_t)(b - a.first) * QWEN_Q_HEADS + h) * a.ld;
  const float* vc = a.v_cache + (a.prefill ? 0 : (size_t)b * a.cache_stride) + (h / QWEN_GROUPS) * QWEN_HEAD_DIM;
  constexpr int NV = kPvTile * 32 / 256;  // float4 of a tile per producer thread
  float4 v[DEPTH][NV];
  const int vrow = (tid & 255) >> 5, vpart = (tid & 31) * 4;
  auto fetch = [&](float4* r, int tile) {
#pragma unroll
    for (int j = 0; j < NV; ++j)  // rows past the last key re-read it; their products are not added
      r[j] = load4(vc + (size_t)min(tile * kPvTile + j * 8 + vrow, n - 1) * QWEN_KV_WIDTH + vpart, a.vec);
  };
  if (wave >= 4) {
#pragma unroll
    for (int i = 0; i < DEPTH; ++i)
      if (i < nt) fetch(v[i], i);
  }
  float m = -1.0e30f;
  for (int t = tid; t < n; t += 512) m = sc[t] > m ? sc[t] : m;
#pragma unroll
  for (int i = 32; i > 0; i >>= 1) {
    const float o = __shfl_xor(m, i);
    m = o > m ? o : m;
  }
  if (lane == 0) red[wave] = m;
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) m = red[i] > m ? red[i] : m;
  auto exps = [&](int tile) {
    const int t = tile * kPvTile + lane;
    if (t < n) {
      const float arg = sc[t] - m;
      es[tile & 3][lane] = a.prefill ? approx_exp(arg) : glibc_expf(arg);
    }
  };
  if (wave == 3) {
    if (nt > 0) exps(0);
    if (nt > 1) exps(1);
  }
  __syncthreads();
  float acc = 0.0f;
  if (wave < 3) __builtin_amdgcn_s_setprio(3);
  for (int i0 = 0; i0 < nt; i0 += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      const int i = i0 + u;
      if (i < nt) {
        float* p = prod[u & 1];
        if (wave >= 4) {
#pragma unroll
          for (int j = 0; j < NV; ++j) {
            const float e = es[i & 3][j * 8 + vrow];
            *reinterpret_cast<float4*>(p + (j * 8 + vrow) * QWEN_HEAD_DIM + vpart) =
                make_float4(e * v[u][j].x, e * v[u][j].y, e * v[u][j].z, e * v[u][j].w);
          }
          if (i + DEPTH < nt) fetch(v[u], i + DEPTH);
        } else if (wave == 3 && i + 2 < nt) {
          exps(i + 2);
        }
        __syncthreads();
        const int cnt = min(kPvTile, n - i * kPvTile);
        if (wave < 2) {
          const float* pd = p + wave * 64 + lane;
          if (cnt == kPvTile) {
#pragma unroll
            for (int j = 0; j < kPvTile; ++j) acc += pd[j * QWEN_HEAD_DIM];
          } else {
            for (int j = 0; j < cnt; ++j) acc += pd[j * QWEN_HEAD_DIM];
          }
        } else if (wave == 2) {
          if (cnt == kPvTile) {
            acc = chain_add<kPvTile>(acc, es[i & 3]);
          } else {
            for (int j = 0; j < cnt; ++j) acc += es[i & 3][j];
          }
        }
      }
    }
  }
  if (tid == 128) den_s = acc;
  __syncthreads();
  const float inv = den_s > 0.0f ? 1.0f / den_s : 0.0f;
  if (wave < 2) a.ctx[(size_t)b * QWEN_HIDDEN + h * QWEN_HEAD_DIM + tid] = acc * inv;
}

// ---------------------------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------------------------
void launch_rmsnorm_ordered(const float* x, const float* w, float* y, int tokens, bool prefill, hipStream_t st) {
  hipLaunchKernelGGL(rmsnorm_ordered_kernel, dim3(tokens), dim3(256), 0, st, x, w, y, prefill ? 1 : 0);
}

namespace {

int ceil_div(int a, int b) { return (a + b - 1) / b; }

template <int R, int KC, int PD, int K, bool NORM, bool GU>
void launch_chain(const OrdProject& a, int rows, hipStream_t st) {
  hipLaunchKernelGGL((project_chain_kernel<R, KC, PD, K, NORM, GU>), dim3(rows / R, a.tokens), dim3(256 + 4 * R), 0, st, a);
}

// Stagers up to TT = 4 (their registers leave four waves per SIMD).  At TT = 8 and 16 they would cost the CU's
// second block, and launch_mfma takes those forms for more blocks than CUs only.
template <int TT, bool GU>
void launch_mfma_tt(const OrdProject& a, int rows, hipStream_t st) {
  constexpr bool kStagers = TT <= 4;
  hipLaunchKernelGGL((project_mfma_kernel<TT, GU, kStagers>), dim3(rows / kMmRows, ceil_div(a.tokens, 4 * TT)),
                     dim3(kStagers ? 512 : 256), 0, st, a);
}

template <bool GU>
void launch_mfma(const OrdProject& a, int rows, hipStream_t st) {
  // Tokens per wave: the least of the measured cycles per input of one round of blocks (one per CU), or of each
  // round of several, times the rounds.  128 tokens: 131 us for 1536 rows of 8960 inputs at TT = 4 (222 at 8,
  // 434 at 16), 150 us for the gate/up pair at 4 or 8 (173 at 16).
  static constexpr int kTT[5] = {1, 2, 4, 8, 16};
  static constexpr int kOneRound[5] = {26, 31, 38, 59, 116}, kRound[5] = {20, 22, 26, 47, 88};
  int best = 0;
  long cost = -1;
  for (int i = 0; i < 5; ++i) {
    const long rounds = ((long)(rows / kMmRows) * ceil_div(a.tokens, 4 * kTT[i]) + 255) / 256;
    const long c = rounds == 1 ? kOneRound[i] : rounds * kRound[i];
    if (cost < 0 || c < cost) {
      cost = c;
      best = i;
    }
  }
  switch (kTT[best]) {
    case 1: launch_mfma_tt<1, GU>(a, rows, st); break;
    case 2: launch_mfma_tt<2, GU>(a, rows, st); break;
    case 4: launch_mfma_tt<4, GU>(a, rows, st); break;
    case 8: launch_mfma_tt<8, GU>(a, rows, st); break;
    default: launch_mfma_tt<16, GU>(a, rows, st); break;
  }
}

}  // namespace

// The chain kernel up to five tokens of 1536 rows and four of 2048, mfma beyond.  A decode layer, chain against
// mfma: o at 5 tokens 152 and 156 us, at 7 180 and 179, at 10 190 and 184; down at 3 tokens 136 and 163, at 5 151
// and 174, at 6 182 and 179, at 10 220 and 184 (its 86 KB of LDS leave a CU one block, so three tokens and
// more, 288 blocks and more, take a second round).
bool ordered_chain_shape(int rows, int tokens) { return (long)rows / 16 * tokens <= 512; }

void launch_project_ordered(const OrdProject& p, hipStream_t st) {
  OrdProject a = p;
  int rows = 0;
  for (int i = 0; i < 3; ++i) {
    a.seg[i].row0 = rows;
    rows += a.seg[i].rows;
  }
  if (ordered_chain_shape(rows, a.tokens)) {
    if (a.norm_w)
      launch_chain<16, 256, 6, QWEN_HIDDEN, true, false>(a, rows, st);
    else if (a.in_dim == QWEN_HIDDEN)
      launch_chain<16, 256, 6, QWEN_HIDDEN, false, false>(a, rows, st);
    else
      launch_chain<16, 256, 5, QWEN_INTERMEDIATE, false, false>(a, rows, st);
    return;
  }
  if (a.norm_w) throw std::runtime_error("the norm is fused for the chain kernel's shapes only");
  launch_mfma<false>(a, rows, st);
}

void launch_gate_up_ordered(const OrdProject& a, hipStream_t st) {
  if (a.tokens == 1) {
    if (a.norm_w)
      launch_chain<16, 128, 6, QWEN_HIDDEN, true, true>(a, 2 * QWEN_INTERMEDIATE, st);
    else
      launch_chain<16, 128, 6, QWEN_HIDDEN, false, true>(a, 2 * QWEN_INTERMEDIATE, st);
    return;
  }
  if (a.norm_w) throw std::runtime_error("the norm is fused for one token only");
  launch_mfma<true>(a, 2 * QWEN_INTERMEDIATE, st);
}

void launch_rope_append_decode(float* q, const float* k, const float* v, const int* pos, const float* rope,
                               bool rope_rows_are_tokens, float* k_cache, float* v_cache, size_t cache_stride,
                               int max_keys, int tokens, hipStream_t st) {
  hipLaunchKernelGGL(rope_append_decode_kernel, dim3(tokens), dim3(64), 0, st, q, k, v, pos, rope,
                     rope_rows_are_tokens ? 1 : 0, k_cache, v_cache, cache_stride, max_keys);
}

void launch_rope_prefill(float* q, float* k_rows, const float* rope, int tokens, hipStream_t st) {
  hipLaunchKernelGGL(rope_prefill_kernel, dim3(tokens), dim3(64), 0, st, q, k_rows, rope);
}

void launch_rope_table_prefill(float* rope, int first, int count, hipStream_t st) {
  const int n = count * 64;
  hipLaunchKernelGGL(rope_table_prefill_kernel, dim3((n + 255) / 256), dim3(256), 0, st, rope, first, count);
}

void launch_attention_ordered(const float* q, const float* k_cache, const float* v_cache, size_t cache_stride,
                              const int* pos, int max_keys, int tokens, float* ctx, hipStream_t st) {
  hipLaunchKernelGGL(attention_ordered_kernel, dim3(QWEN_Q_HEADS, tokens), dim3(128), 0, st, q, k_cache, v_cache,
                     cache_stride, pos, max_keys, ctx);
}

namespace {
constexpr size_t kScoreFloats = size_t(16) << 20;  // 64 MB of kept scores per pair of launches
int score_ld(int max_keys) { return ceil_div(max_keys, 64) * 64; }
// Tokens whose scores are kept at once: at least one query group of 4.
int score_tokens(int tokens, int max_keys) {
  const size_t fit = kScoreFloats / ((size_t)QWEN_Q_HEADS * score_ld(max_keys));
  const int most = (int)(fit < 4 ? 4 : fit > 65532 ? 65532 : fit & ~size_t(3));
  return tokens < most ? tokens : most;
}
}  // namespace

size_t attention_ordered_scores(int tokens, int max_keys) {
  return (size_t)score_tokens(tokens, max_keys) * QWEN_Q_HEADS * score_ld(max_keys);
}

void launch_attention_ordered_split(const OrdAttentionArgs& c, int tokens, float* scores, hipStream_t st) {
  OrdAttention a{};
  a.q = c.q;
  a.k_cache = c.k_cache;
  a.v_cache = c.v_cache;
  a.cache_stride = c.cache_stride;
  a.pos = c.pos;
  a.max_keys = c.max_keys;
  a.prefill = c.prefill ? 1 : 0;
  a.past = c.past;
  a.vec = ((reinterpret_cast<uintptr_t>(c.k_cache) | reinterpret_cast<uintptr_t>(c.v_cache)) & 15u) == 0 &&
          c.cache_stride % 4 == 0;
  a.k_new = c.k_new;
  a.v_new = c.v_new;
  a.rope = c.rope;
  a.rope_rows_are_tokens = c.rope_rows_are_tokens ? 1 : 0;
  a.scores = scores;
  a.ld = score_ld(c.max_keys);
  a.ctx = c.ctx;
  const int step = score_tokens(tokens, c.max_keys);
  for (int first = 0; first < tokens; first += step) {
    a.first = first;
    a.tokens = tokens - first < step ? tokens - first : step;
    const int keys = c.prefill ? c.past + first + a.tokens : c.max_keys;
    const int tiles = ceil_div(keys, kScoreKeys);
    if (c.k_new)
      hipLaunchKernelGGL((scores_ordered_kernel<1, true>), dim3(a.tokens, QWEN_KV_HEADS, tiles), dim3(384), 0, st, a);
    else if (c.prefill)
      hipLaunchKernelGGL((scores_ordered_kernel<4, false>), dim3(ceil_div(a.tokens, 4), QWEN_KV_HEADS, tiles),
                         dim3(384), 0, st, a);
    else
      hipLaunchKernelGGL((scores_ordered_kernel<1, false>), dim3(a.tokens, QWEN_KV_HEADS, tiles), dim3(384), 0, st, a);
    if (c.prefill)
      hipLaunchKernelGGL(softmax_pv_ordered_kernel<2>, dim3(QWEN_Q_HEADS, a.tokens), dim3(512), 0, st, a);
    else
      hipLaunchKernelGGL(softmax_pv_ordered_kernel<4>, dim3(QWEN_Q_HEADS, a.tokens), dim3(512), 0, st, a);
  }
}

}  // namespace qwen
