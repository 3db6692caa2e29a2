// Device-resident multi-layer model: weights uploaded once, every step queued on one stream.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <mutex>
#include <string>
#include <vector>

#include "kernels.hpp"
#include "qwen_hip_model.h"
#include "runtime.hpp"

using namespace qwen;

namespace {

// Repacked (FAST) weights and parameter pointers of one layer.  Scales, biases and norm weights
// point into the uploaded scale image (q/k/v scales and biases are contiguous there, so the
// fused QKV projection reads them in place).
struct FastLayer {
  uint8_t *qkv, *o, *gate, *up, *down;
  const float *sw_qkv, *b_qkv, *sw_o, *sw_gate, *sw_up, *sw_down, *ln, *post_ln;
};

constexpr size_t kQkvRows = QWEN_QKV_ROWS;  // 2048
constexpr size_t kMaxDecodeBatch = 65535;    // most sequences of one FAST decode call (attention grid z)
constexpr size_t kRepackedLayerBytes = QWEN_PACKED_WEIGHT_BYTES;

// Device buffer that only grows (freed after a device synchronize); `generation` counts the
// allocations, so users can re-initialize state kept in the buffer after a move.
struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
  unsigned generation = 0;
  void* get(size_t bytes) {
    if (bytes <= cap) return p;
    ++generation;
    if (p) {
      QWEN_HIP(hipDeviceSynchronize());
      QWEN_HIP(hipFree(p));
      p = nullptr;
      cap = 0;
    }
    const size_t want = bytes + (bytes >> 3) + (1u << 20);
    QWEN_HIP(hipMalloc(&p, want));
    cap = want;
    return p;
  }
};

struct LastCall {
  int kind = 0;  // 0 none, 1 decode, 2 prefill
  int mode = 0, batch = 0, seq_len = 0, max_keys = 0, past = 0;
  int first = 0, count = 0;  // layers first..first+count-1; their caches start at k_cache / v_cache
  const int* positions = nullptr;
  float *k_cache = nullptr, *v_cache = nullptr;
  uint64_t seq_stride = 0, layer_stride = 0;
};

}  // namespace

struct qwen_hip_model {
  int layers = 0;
  std::mutex mu;
  hipStream_t stream = nullptr;
  uint8_t* raw_w = nullptr;  // layers x QWEN_LAYER_BYTES (weight images)
  float* raw_s = nullptr;    // layers x QWEN_LAYER_BYTES/4 words (scale images)
  uint8_t* wp = nullptr;     // layers x repacked weights
  std::vector<FastLayer> fast;
  float* rope_decode = nullptr;   // [QWEN_MAX_SEQ][128]
  float* rope_prefill = nullptr;  // [QWEN_MAX_SEQ][128]
  uint16_t* embed = nullptr;      // tied embedding / lm_head table [vocab][1536] bf16
  uint16_t* head_norm = nullptr;  // final RMSNorm weight [1536] bf16
  int vocab = 0;                  // rows of `embed` (0: no head)
  DevBuf head_ws;                 // head: normalized rows and per-block argmax candidates
  Arena arena;                    // ORDERED per-layer intermediates
  DevBuf ws;                      // FAST workspace and ORDERED attention output
  unsigned zero_sums_ready = 0;   // ws generation whose zero limb sums were written
  LastCall last;

  // FAST workspace carve-up for `tokens` rows and `batch` x `nsplit` decode-attention partials.
  struct Ws {
    int8_t* xq;
    float* sx;
    int* sums;
    float *qkv, *ctx, *att, *s, *tmp, *part;
    float2* pml;
    float* splitk;  // K-split partials of the non-dual projections (out <= 2048)
    uint8_t* kvt;   // prefill attention: bf16 hi/lo K/V tiles of one layer
    int8_t* gxq;    // grouped code of the SiLU·up rows (2..64 tokens): limbs, per-(token, 64-row group)
    float* gsx;     //   scales and offset terms
    int* gcorr;
    const int* zero_sums;  // kSkinnyTokens x (0, 0): the limb sums of code whose offsets are applied per group
    int* budget;           // ragged decode attention: keys per block
    float* gmax;           // one token: max |SiLU.up| of each 16-row block of the gate/up projection
  };
  // Fixed region at the start of the workspace: the zero limb sums, zeroed once per workspace buffer
  // and never written otherwise.
  static constexpr size_t kFixedBytes = (kSkinnyTokens * 8u + 255u) & ~size_t(255u);
  Ws carve(size_t tokens, size_t batch, size_t nsplit, size_t kvt_bytes = 0) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
      const size_t o = off;
      off = (off + bytes + 255u) & ~size_t(255u);
      return o;
    };
    const size_t o_zs = take(kSkinnyTokens * 8u);  // fixed offset: never overlaps the parts below
    const size_t o_xq = take(xq_bytes(tokens, QWEN_INTERMEDIATE));
    const size_t o_sx = take(tokens * 4u);
    const size_t o_sums = take(tokens * 8u);
    const size_t o_qkv = take(tokens * kQkvRows * 4u);
    const size_t o_ctx = take(tokens * QWEN_HIDDEN * 4u);
    const size_t o_att = take(tokens * QWEN_HIDDEN * 4u);
    const size_t o_s = take(tokens * QWEN_INTERMEDIATE * 4u);
    const size_t o_tmp = take(tokens * QWEN_INTERMEDIATE * 4u);
    const size_t o_part = take(batch * QWEN_Q_HEADS * nsplit * QWEN_HEAD_DIM * 4u);
    const size_t o_pml = take(batch * QWEN_Q_HEADS * nsplit * 8u);
    const size_t o_splitk = take(splitk_bytes(kQkvRows, tokens));
    const size_t o_kvt = take(kvt_bytes);
    const size_t gtok = tokens < (size_t)kSkinnyTokens ? tokens : (size_t)kSkinnyTokens;
    const size_t o_gxq = take(xq_bytes(gtok, QWEN_INTERMEDIATE));
    const size_t o_gsx = take(gtok * (QWEN_INTERMEDIATE / 64) * 4u);
    const size_t o_gcorr = take(gtok * (QWEN_INTERMEDIATE / 64) * 4u);
    const size_t o_gmax = take((QWEN_INTERMEDIATE / 16) * 4u);
    const size_t o_budget = take(4u);
    char* b = static_cast<char*>(ws.get(off));
    if (ws.generation != zero_sums_ready) {  // fresh buffer: zero the sums once
      launch_zero_u32(reinterpret_cast<unsigned*>(b + o_zs), (int)(2 * kSkinnyTokens), stream);
      zero_sums_ready = ws.generation;
    }
    return Ws{reinterpret_cast<int8_t*>(b + o_xq), reinterpret_cast<float*>(b + o_sx),
              reinterpret_cast<int*>(b + o_sums), reinterpret_cast<float*>(b + o_qkv),
              reinterpret_cast<float*>(b + o_ctx), reinterpret_cast<float*>(b + o_att),
              reinterpret_cast<float*>(b + o_s), reinterpret_cast<float*>(b + o_tmp),
              reinterpret_cast<float*>(b + o_part), reinterpret_cast<float2*>(b + o_pml),
              reinterpret_cast<float*>(b + o_splitk), reinterpret_cast<uint8_t*>(b + o_kvt),
              reinterpret_cast<int8_t*>(b + o_gxq), reinterpret_cast<float*>(b + o_gsx), reinterpret_cast<int*>(b + o_gcorr),
              reinterpret_cast<const int*>(b + o_zs), reinterpret_cast<int*>(b + o_budget),
              reinterpret_cast<float*>(b + o_gmax)};
  }

  Ws carve_prefill(size_t tokens, int nseq, int keys, const AttnPrefillPlan& plan) {
    return carve(tokens, plan.nsplit > 1 ? tokens : 1, plan.nsplit, attn_prefill_workspace_bytes(keys, nseq));
  }

  // Plain scratch of `bytes` in the workspace, past the fixed region.
  float* scratch(size_t bytes) {
    const size_t off = kFixedBytes;
    return reinterpret_cast<float*>(static_cast<char*>(ws.get(off + bytes)) + off);
  }

  DevLayer dev_layer(int l) const {
    const uint8_t* w = raw_w + (size_t)l * QWEN_LAYER_BYTES;
    const float* s = raw_s + (size_t)l * (QWEN_LAYER_BYTES / 4);
    DevLayer d;
    d.ln = s + QWEN_OFF_INPUT_LN / 4;
    d.post_ln = s + QWEN_OFF_POST_LN / 4;
    d.qw = w + QWEN_OFF_Q_W;
    d.kw = w + QWEN_OFF_K_W;
    d.vw = w + QWEN_OFF_V_W;
    d.ow = w + QWEN_OFF_O_W;
    d.gw = w + QWEN_OFF_GATE_W;
    d.uw = w + QWEN_OFF_UP_W;
    d.dw = w + QWEN_OFF_DOWN_W;
    d.qb = s + QWEN_OFF_Q_B / 4;
    d.kb = s + QWEN_OFF_K_B / 4;
    d.vb = s + QWEN_OFF_V_B / 4;
    d.qs = s + QWEN_OFF_Q_S / 4;
    d.ks = s + QWEN_OFF_K_S / 4;
    d.vs = s + QWEN_OFF_V_S / 4;
    d.os = s + QWEN_OFF_O_S / 4;
    d.gs = s + QWEN_OFF_GATE_S / 4;
    d.us = s + QWEN_OFF_UP_S / 4;
    d.ds = s + QWEN_OFF_DOWN_S / 4;
    return d;
  }

  // Allocates images, tables and the repacked weights; raw images are filled by the caller.
  void allocate(int n) {
    layers = n;
    QWEN_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&raw_w), (size_t)n * QWEN_LAYER_BYTES));
    QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&raw_s), (size_t)n * QWEN_LAYER_BYTES));
    QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&wp), (size_t)n * kRepackedLayerBytes));
    // RoPE tables for every position: decode from host libm (qwen_decode_attention_kernel.cpp:29-42),
    // prefill on the device (qwen_prefill_attention_kernel.cpp:128-143).
    std::vector<float> host((size_t)QWEN_MAX_SEQ * 128u);
    for (int r = 0; r < QWEN_MAX_SEQ; ++r) decode_rope_row_host(r, &host[(size_t)r * 128u]);
    QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&rope_decode), host.size() * 4u));
    QWEN_HIP(hipMemcpy(rope_decode, host.data(), host.size() * 4u, hipMemcpyHostToDevice));
    QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&rope_prefill), host.size() * 4u));
    launch_rope_table_prefill(rope_prefill, 0, QWEN_MAX_SEQ, stream);
    QWEN_HIP(hipGetLastError());
  }

  // Repacks every layer's INT4 matrices from the raw images into the MFMA tile layout.
  void build_fast() {
    fast.resize(layers);
    for (int l = 0; l < layers; ++l) {
      const DevLayer d = dev_layer(l);
      uint8_t* base = wp + (size_t)l * kRepackedLayerBytes;
      FastLayer& f = fast[l];
      f.qkv = base;
      f.o = f.qkv + kQkvRows * QWEN_HIDDEN / 2;
      f.gate = f.o + (size_t)QWEN_HIDDEN * QWEN_HIDDEN / 2;
      f.up = f.gate + (size_t)QWEN_INTERMEDIATE * QWEN_HIDDEN / 2;
      f.down = f.up + (size_t)QWEN_INTERMEDIATE * QWEN_HIDDEN / 2;
      // q, k and v rows are contiguous in the layer image, so one repack covers all 2048 rows.
      launch_repack_int4(d.qw, (int)kQkvRows, QWEN_HIDDEN, f.qkv, stream);
      launch_repack_int4(d.ow, QWEN_HIDDEN, QWEN_HIDDEN, f.o, stream);
      launch_repack_int4(d.gw, QWEN_INTERMEDIATE, QWEN_HIDDEN, f.gate, stream);
      launch_repack_int4(d.uw, QWEN_INTERMEDIATE, QWEN_HIDDEN, f.up, stream);
      launch_repack_int4(d.dw, QWEN_HIDDEN, QWEN_INTERMEDIATE, f.down, stream);
      f.sw_qkv = d.qs;  // q_s, k_s, v_s contiguous
      f.b_qkv = d.qb;   // q_b, k_b, v_b contiguous
      f.sw_o = d.os;
      f.sw_gate = d.gs;
      f.sw_up = d.us;
      f.sw_down = d.ds;
      f.ln = d.ln;
      f.post_ln = d.post_ln;
    }
    QWEN_HIP(hipGetLastError());
    QWEN_HIP(hipStreamSynchronize(stream));
  }

  ~qwen_hip_model() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (void* p : {static_cast<void*>(raw_w), static_cast<void*>(raw_s), static_cast<void*>(wp),
                    static_cast<void*>(rope_decode), static_cast<void*>(rope_prefill), static_cast<void*>(embed),
                    static_cast<void*>(head_norm), head_ws.p,
                    ws.p})
      if (p) (void)hipFree(p);
    if (stream) (void)hipStreamDestroy(stream);
  }

  // ---- one step -------------------------------------------------------------------------
  // A FAST projection of the activations quantized in w (xq, sx, sums).  `fuse` (optional) selects an
  // epilogue fused into the split-K reduce step and carries its extra arguments.
  void gemm(const Ws& w, int tokens, int in, int out, const uint8_t* wpm, const float* sw, const float* bias,
            float* y, size_t ys, int epi, const uint8_t* wp2 = nullptr, const float* sw2 = nullptr,
            const float* resid = nullptr, int round = 0, int prefill_silu = 0, const GemmArgs* fuse = nullptr) {
    launch_gemm_i8(args(w, tokens, in, out, wpm, sw, bias, y, ys, wp2, sw2, resid, round, prefill_silu, fuse), epi,
                   stream);
  }
  GemmArgs args(const Ws& w, int tokens, int in, int out, const uint8_t* wpm, const float* sw, const float* bias,
                float* y, size_t ys, const uint8_t* wp2 = nullptr, const float* sw2 = nullptr,
                const float* resid = nullptr, int round = 0, int prefill_silu = 0,
                const GemmArgs* fuse = nullptr) const {
    GemmArgs g = fuse ? *fuse : GemmArgs{};
    g.wp = wpm;
    g.wp2 = wp2;
    g.sw = sw;
    g.sw2 = sw2;
    g.bias = bias;
    g.xq = w.xq;
    g.sx = w.sx;
    g.sums = w.sums;
    g.tokens = tokens;
    g.in_dim = in;
    g.out_dim = out;
    g.y = y;
    g.y_stride = ys;
    g.resid = resid;
    g.resid_stride = QWEN_HIDDEN;
    g.y_raw = nullptr;
    g.round_bf16 = round;
    g.prefill_silu = prefill_silu;
    g.part = wp2 ? nullptr : w.splitk;
    return g;
  }

  // Layers first..first+count-1; the caches of layer first+i start at kc0/vc0 + i*ls.
  void decode_fast(int first, int count, int B, float* hidden, const int* pos, int max_keys, float* kc0, float* vc0,
                   uint64_t ss, uint64_t ls, int round, bool pre_reduce = true, bool sep_attn = false) {
    const AttnDecodePlan plan = plan_attn_decode(B, max_keys);
    const Ws w = carve(B, B, plan.nsplit);
    const bool fused = B <= kSplitTokens;
    const bool one = fused && B == 1 && pre_reduce;  // one sequence: reduce steps in the next projection
    // one sequence with 64-key splits (at most 1536 keys): the attention over the history keys runs in
    // the Q/K/V projection's blocks, and the O projection's merge adds the new key's term
    const bool fuse_attn =
        one && !sep_attn && plan.chunk == kFusedAttnChunk && plan.nsplit <= kFusedAttnMaxSplits;
    AttnFuseArgs af{};
    af.part = w.part;
    af.pml = w.pml;
    af.nsplit = plan.nsplit;
    af.chunk = plan.chunk;
    af.max_keys = max_keys;
    // 2..64 sequences: the gate/up projection quantizes its SiLU·up rows per 64-row group for the down
    // projection (no separate quantization launch).  One sequence keeps the row code in both forms
    // (its prologue-fused form and the separate-launch form stay bit-identical).
    const bool grouped = B >= 2 && B <= kSkinnyTokens;
    GemmArgs down_pending{};                         // the previous layer's deferred down projection
    for (int i = 0; i < count; ++i) {
      const int l = first + i;
      const FastLayer& f = fast[l];
      float* kc = kc0 + (size_t)i * ls;
      float* vc = vc0 + (size_t)i * ls;
      // RoPE + KV append run inside the Q/K/V projection; with at most kSplitTokens sequences the two
      // RMSNorm + quantize steps run inside the split-K reduce kernels of the O and down projections.
      // (one sequence with the attention fused: the first layer's RMSNorm and quantization run in the
      // Q/K/V blocks' prologue instead)
      if ((i == 0 && !fuse_attn) || !fused)
        launch_norm_quant(hidden, QWEN_HIDDEN, B, QWEN_HIDDEN, f.ln, kNormDecode, w.xq, w.sx, w.sums, nullptr,
                          stream);
      {
        GemmArgs fq{};
        fq.fuse = kFuseQkvRope;
        fq.pos = pos;
        fq.rope = rope_decode;
        fq.k_cache = kc;
        fq.v_cache = vc;
        fq.seq_stride = ss;
        fq.limit = max_keys;
        if (one && i > 0) {
          // the previous layer's down projection left its K-split partials: every block of this
          // projection finishes that row (residual, bf16 rounding, this layer's RMSNorm, quantization)
          const GemmArgs qa = args(w, B, QWEN_HIDDEN, (int)kQkvRows, f.qkv, f.sw_qkv, f.b_qkv, w.qkv, kQkvRows,
                                   nullptr, nullptr, nullptr, 0, 0, &fq);
          if (fuse_attn ? !launch_gemm_i8_pre_attn(qa, down_pending, kPreResidualSplits, af, stream)
                        : !launch_gemm_i8_pre(qa, down_pending, kEpiResidual, kPreResidualSplits, stream))
            throw std::runtime_error("Q/K/V with the down reduce: bad shape");
        } else if (fuse_attn) {
          // the range's first layer: every block normalizes and quantizes the input row itself (a
          // reduce step with no partials: the row is the "residual", the correction terms zero)
          const GemmArgs qa = args(w, B, QWEN_HIDDEN, (int)kQkvRows, f.qkv, f.sw_qkv, f.b_qkv, w.qkv, kQkvRows,
                                   nullptr, nullptr, nullptr, 0, 0, &fq);
          GemmArgs in{};
          in.fuse = kFuseNormQuant;
          in.norm = kNormDecode;
          in.norm_w = f.ln;
          in.tokens = 1;
          in.in_dim = QWEN_HIDDEN;
          in.out_dim = QWEN_HIDDEN;
          in.resid = hidden;
          in.resid_stride = QWEN_HIDDEN;
          in.sw = f.ln;  // read, times a zero correction
          in.sums = w.zero_sums;
          in.sx = reinterpret_cast<const float*>(w.zero_sums);
          if (!launch_gemm_i8_pre_attn(qa, in, 0, af, stream))
            throw std::runtime_error("Q/K/V with the attention: bad shape");
        } else {
          gemm(w, B, QWEN_HIDDEN, (int)kQkvRows, f.qkv, f.sw_qkv, f.b_qkv, w.qkv, kQkvRows, kEpiStore, nullptr,
               nullptr, nullptr, 0, 0, &fq);
        }
      }
      // one sequence: the attention leaves its split partials, merged by every block of the O projection
      if (!fuse_attn)
        launch_attn_decode(w.qkv, (int)kQkvRows, kc, vc, ss, pos, B, max_keys, plan, w.part, w.pml, w.budget,
                           nullptr, one ? nullptr : w.xq, w.sx, w.sums, stream);
      GemmArgs fn{};
      fn.fuse = kFuseNormQuant;
      fn.norm = kNormDecode;
      fn.xq_out = w.xq;
      fn.sx_out = w.sx;
      fn.sums_out = w.sums;
      if (one) {
        // one sequence: the O projection leaves its fp32 partials, and every block of the gate/up
        // projection finishes that row (residual, RMSNorm, quantization) into its own activation
        // slice: one launch fewer per layer
        fn.norm_w = f.post_ln;
        fn.defer_reduce = 1;
        const GemmArgs oa = args(w, B, QWEN_HIDDEN, QWEN_HIDDEN, f.o, f.sw_o, nullptr, w.att, QWEN_HIDDEN, nullptr,
                                 nullptr, nullptr, 0, 0, &fn);
        fn.defer_reduce = 0;
        const AttnMergeArgs am{w.part, w.pml, pos, plan.nsplit, plan.chunk, max_keys, w.sx, w.sums,
                               fuse_attn ? w.qkv : nullptr};
        if (!launch_gemm_i8_prea(oa, am, stream)) throw std::runtime_error("O with the attention merge: bad shape");
        GemmArgs ga = args(w, B, QWEN_HIDDEN, QWEN_INTERMEDIATE, f.gate, f.sw_gate, nullptr, w.s, QWEN_INTERMEDIATE,
                           f.up, f.sw_up);
        ga.amax_out = w.gmax;  // the down projection's blocks take the row's maximum from these
        // the O partials of the head ranges carry their own offset corrections: a zero correction here
        GemmArgs op = oa;
        op.sums = w.zero_sums;
        op.sx = reinterpret_cast<const float*>(w.zero_sums);
        if (!launch_gemm_i8_pre(ga, op, kEpiStore, kOneTokenOSplits, stream))
          throw std::runtime_error("gate/up with the O reduce: bad shape");
      } else {
        if (fused) {
          fn.norm_w = f.post_ln;
          gemm(w, B, QWEN_HIDDEN, QWEN_HIDDEN, f.o, f.sw_o, nullptr, w.att, QWEN_HIDDEN, kEpiStore, nullptr, nullptr,
               nullptr, 0, 0, &fn);
        } else {
          gemm(w, B, QWEN_HIDDEN, QWEN_HIDDEN, f.o, f.sw_o, nullptr, w.att, QWEN_HIDDEN, kEpiStore);
          launch_norm_quant(w.att, QWEN_HIDDEN, B, QWEN_HIDDEN, f.post_ln, kNormDecode, w.xq, w.sx, w.sums, nullptr,
                            stream);
        }
        GemmArgs gq{};
        gq.xq_out = w.gxq;
        gq.gsx_out = w.gsx;
        gq.gcorr_out = w.gcorr;
        gemm(w, B, QWEN_HIDDEN, QWEN_INTERMEDIATE, f.gate, f.sw_gate, nullptr, w.s, QWEN_INTERMEDIATE, kEpiSiluMul,
             f.up, f.sw_up, nullptr, 0, 0, grouped ? &gq : nullptr);
      }
      const bool fuse_next = fused && i + 1 < count;  // the next layer's input RMSNorm + quantize
      fn.norm_w = fuse_next ? fast[l + 1].ln : nullptr;
      if (one) {
        // the SiLU·up row is quantized by every block of the down projection for its own K chunks;
        // the reduce step runs in the next layer's Q/K/V blocks (its own launch after the last layer)
        GemmArgs sq{};
        sq.y = w.s;
        sq.in_dim = QWEN_INTERMEDIATE;
        sq.sx_out = w.sx;
        sq.sums_out = w.sums;
        sq.amax_in = w.gmax;
        sq.amax_n = gate_up_maxima_count(QWEN_INTERMEDIATE);
        fn.defer_reduce = fuse_next ? 1 : 0;
        const GemmArgs da = args(w, B, QWEN_INTERMEDIATE, QWEN_HIDDEN, f.down, f.sw_down, nullptr, hidden,
                                 QWEN_HIDDEN, nullptr, nullptr, w.att, round, 0, fuse_next ? &fn : nullptr);
        fn.defer_reduce = 0;
        if (!launch_gemm_i8_preq(da, sq, stream)) throw std::runtime_error("down with the quantization: bad shape");
        if (fuse_next) down_pending = da;
      } else {
        if (!grouped)
          launch_norm_quant(w.s, QWEN_INTERMEDIATE, B, QWEN_INTERMEDIATE, nullptr, kNormNone, w.xq, w.sx, w.sums,
                            nullptr, stream);
        GemmArgs da = args(w, B, QWEN_INTERMEDIATE, QWEN_HIDDEN, f.down, f.sw_down, nullptr, hidden, QWEN_HIDDEN,
                           nullptr, nullptr, w.att, round, 0, fuse_next ? &fn : nullptr);
        if (grouped) {  // the down partials carry the per-group offsets: the reduce step gets zero sums
          da.xq = w.gxq;
          da.gsx = w.gsx;
          da.gcorr = w.gcorr;
          da.sums = w.zero_sums;
        }
        launch_gemm_i8(da, kEpiResidual, stream);
      }
    }
    QWEN_HIP(hipGetLastError());
  }

  // FAST prefill of S new tokens per sequence at positions past..past+S-1 (cache rows 0..past-1 hold
  // the earlier tokens of each sequence).
  void prefill_fast(int first, int count, int B, int S, int past, float* hidden, float* kc0, float* vc0, uint64_t ss,
                    uint64_t ls, int round) {
    const int T = B * S;
    const AttnPrefillPlan plan = plan_attn_prefill(S, past, B);
    const Ws w = carve_prefill(T, B, past + S, plan);
    // Up to kPrefillFuseTokens tokens the RMSNorm + quantization that follow the O and down projections run in
    // the step that adds those projections' K splits (their 64-token tiles alone fill a fraction of the CUs).
    // Up to kSkinnyTokens the SiLU·up rows go to the down projection in the grouped code, as a decode batch's.
    const bool fused = T <= kPrefillFuseTokens;
    const bool grouped = T <= kSkinnyTokens;
    GemmArgs gq{};
    gq.xq_out = w.gxq;
    gq.gsx_out = w.gsx;
    gq.gcorr_out = w.gcorr;
    GemmArgs fn{};
    fn.fuse = kFuseNormQuant;
    fn.norm = kNormPrefill;
    fn.xq_out = w.xq;
    fn.sx_out = w.sx;
    fn.sums_out = w.sums;
    for (int i = 0; i < count; ++i) {
      const FastLayer& f = fast[first + i];
      float* kc = kc0 + (size_t)i * ls;
      float* vc = vc0 + (size_t)i * ls;
      if (!fused || i == 0)
        launch_norm_quant(hidden, QWEN_HIDDEN, T, QWEN_HIDDEN, f.ln, kNormPrefill, w.xq, w.sx, w.sums, nullptr,
                          stream);
      // RoPE of q and k and the K/V cache append in the Q/K/V projection's epilogue
      GemmArgs fr{};
      fr.fuse = kFuseRopePrefill;
      fr.rope = rope_prefill;
      fr.k_cache = kc;
      fr.v_cache = vc;
      fr.seq_stride = ss;
      fr.seq_len = S;
      fr.past = past;
      fr.limit = past + S;
      gemm(w, T, QWEN_HIDDEN, (int)kQkvRows, f.qkv, f.sw_qkv, f.b_qkv, w.qkv, kQkvRows, kEpiStore, nullptr, nullptr,
           nullptr, 0, 0, &fr);
      launch_attn_prefill(w.qkv, (int)kQkvRows, kc, vc, ss, S, past, B, w.kvt, plan, w.part, w.pml, w.ctx, w.xq, w.sx,
                          w.sums, stream);
      if (plan.nsplit == 1)
        launch_norm_quant(w.ctx, QWEN_HIDDEN, T, QWEN_HIDDEN, nullptr, kNormNone, w.xq, w.sx, w.sums, nullptr, stream);
      fn.norm_w = f.post_ln;
      gemm(w, T, QWEN_HIDDEN, QWEN_HIDDEN, f.o, f.sw_o, nullptr, w.att, QWEN_HIDDEN, kEpiStore, nullptr, nullptr,
           nullptr, 0, 0, fused ? &fn : nullptr);
      if (!fused)
        launch_norm_quant(w.att, QWEN_HIDDEN, T, QWEN_HIDDEN, f.post_ln, kNormPrefill, w.xq, w.sx, w.sums, nullptr,
                          stream);
      gemm(w, T, QWEN_HIDDEN, QWEN_INTERMEDIATE, f.gate, f.sw_gate, nullptr, w.s, QWEN_INTERMEDIATE, kEpiSiluMul,
           f.up, f.sw_up, nullptr, 0, 1, grouped ? &gq : nullptr);
      if (!grouped)
        launch_norm_quant(w.s, QWEN_INTERMEDIATE, T, QWEN_INTERMEDIATE, nullptr, kNormNone, w.xq, w.sx, w.sums,
                          nullptr, stream);
      const bool fuse_next = fused && i + 1 < count;  // the next layer's input RMSNorm + quantize
      fn.norm_w = fuse_next ? fast[first + i + 1].ln : nullptr;
      GemmArgs da = args(w, T, QWEN_INTERMEDIATE, QWEN_HIDDEN, f.down, f.sw_down, nullptr, hidden, QWEN_HIDDEN,
                         nullptr, nullptr, w.att, round, 0, fuse_next ? &fn : nullptr);
      if (grouped) {  // the down partials carry the per-group offsets: the reduce step gets zero sums
        da.xq = w.gxq;
        da.gsx = w.gsx;
        da.gcorr = w.gcorr;
        da.sums = w.zero_sums;
      }
      launch_gemm_i8(da, kEpiResidual, stream);
    }
    QWEN_HIP(hipGetLastError());
  }

  void decode_ordered(int first, int count, int B, float* hidden, const int* pos, int max_keys, float* kc0,
                      float* vc0, uint64_t ss, uint64_t ls, int round) {
    float* att = scratch((size_t)B * QWEN_HIDDEN * 4u);
    for (int i = 0; i < count; ++i) {
      const DevLayer d = dev_layer(first + i);
      arena.reset();
      arena.reserve(decode_workspace_bytes(B, max_keys));
      DecodeBatch b{B, pos, rope_decode, false, kc0 + (size_t)i * ls, vc0 + (size_t)i * ls, (size_t)ss, max_keys};
      run_decode_attention(d, hidden, b, att, arena, stream);
      run_decode_mlp(d, att, B, hidden, arena, stream);
      if (round) launch_round_bf16(hidden, (size_t)B * QWEN_HIDDEN, stream);
    }
    arena.reset();
    QWEN_HIP(hipGetLastError());
  }

  void prefill_ordered(int first, int count, int B, int S, int past, float* hidden, float* kc0, float* vc0,
                       uint64_t ss, uint64_t ls, int round) {
    float* att = scratch((size_t)S * QWEN_HIDDEN * 4u);
    for (int i = 0; i < count; ++i) {
      const DevLayer d = dev_layer(first + i);
      for (int b = 0; b < B; ++b) {
        float* x = hidden + (size_t)b * S * QWEN_HIDDEN;
        arena.reset();
        arena.reserve(prefill_workspace_bytes(S, past));
        run_prefill_attention(d, x, S, past, rope_prefill, kc0 + (size_t)i * ls + (size_t)b * ss,
                              vc0 + (size_t)i * ls + (size_t)b * ss, att, arena, stream);
        run_prefill_mlp(d, att, S, x, arena, stream);
      }
      if (round) launch_round_bf16(hidden, (size_t)B * S * QWEN_HIDDEN, stream);
    }
    arena.reset();
    QWEN_HIP(hipGetLastError());
  }
};

namespace {

template <class Fn>
int guarded_model(Fn&& fn) {
  try {
    return fn();
  } catch (const HipError& e) {
    set_last_error(std::string(e.what) + ": " + hipGetErrorString(e.code));
  } catch (const std::exception& e) {
    set_last_error(e.what());
  }
  if (std::getenv("QWEN_HIP_VERBOSE")) std::fprintf(stderr, "qwen-mi355x: %s\n", last_error_cstr());
  return QWEN_ERR_DEVICE;
}

int invalid(const char* why) {
  set_last_error(why);
  return QWEN_ERR_KERNEL;
}

// Tensor keys of the synthetic generator: 16 per layer, then the embedding table.
enum : uint64_t { kTQ = 0, kTK, kTV, kTO, kTGate, kTUp, kTDown, kTQb, kTKb, kTVb };
constexpr uint64_t kEmbedKey = 1u << 20;

}  // namespace

extern "C" {

int qwen_hip_model_create(int layers, const uint8_t* weight_ddr, const float* scale_ddr, qwen_hip_model** out) {
  if (!out || !weight_ddr || !scale_ddr || layers <= 0 || layers > 1024) return invalid("invalid model arguments");
  *out = nullptr;
  return guarded_model([&]() -> int {
    qwen_hip_model* m = new qwen_hip_model();
    try {
      m->allocate(layers);
      QWEN_HIP(hipMemcpy(m->raw_w, weight_ddr, (size_t)layers * QWEN_LAYER_BYTES, hipMemcpyHostToDevice));
      QWEN_HIP(hipMemcpy(m->raw_s, scale_ddr, (size_t)layers * QWEN_LAYER_BYTES, hipMemcpyHostToDevice));
      m->build_fast();
    } catch (...) {
      delete m;
      throw;
    }
    *out = m;
    return QWEN_OK;
  });
}

int qwen_hip_model_create_synthetic(int layers, uint64_t seed, qwen_hip_model** out) {
  if (!out || layers <= 0 || layers > 1024) return invalid("invalid model arguments");
  *out = nullptr;
  return guarded_model([&]() -> int {
    qwen_hip_model* m = new qwen_hip_model();
    try {
      m->allocate(layers);
      const hipStream_t st = m->stream;
      QWEN_HIP(hipMemsetAsync(m->raw_w, 0, (size_t)layers * QWEN_LAYER_BYTES, st));
      QWEN_HIP(hipMemsetAsync(m->raw_s, 0, (size_t)layers * QWEN_LAYER_BYTES, st));
      struct Mat {
        uint64_t key;
        uint64_t w_off, s_off;
        int out, in;
      };
      const Mat mats[] = {{kTQ, QWEN_OFF_Q_W, QWEN_OFF_Q_S, QWEN_HIDDEN, QWEN_HIDDEN},
                          {kTK, QWEN_OFF_K_W, QWEN_OFF_K_S, QWEN_KV_WIDTH, QWEN_HIDDEN},
                          {kTV, QWEN_OFF_V_W, QWEN_OFF_V_S, QWEN_KV_WIDTH, QWEN_HIDDEN},
                          {kTO, QWEN_OFF_O_W, QWEN_OFF_O_S, QWEN_HIDDEN, QWEN_HIDDEN},
                          {kTGate, QWEN_OFF_GATE_W, QWEN_OFF_GATE_S, QWEN_INTERMEDIATE, QWEN_HIDDEN},
                          {kTUp, QWEN_OFF_UP_W, QWEN_OFF_UP_S, QWEN_INTERMEDIATE, QWEN_HIDDEN},
                          {kTDown, QWEN_OFF_DOWN_W, QWEN_OFF_DOWN_S, QWEN_HIDDEN, QWEN_INTERMEDIATE}};
      for (int l = 0; l < layers; ++l) {
        uint8_t* w = m->raw_w + (size_t)l * QWEN_LAYER_BYTES;
        float* s = m->raw_s + (size_t)l * (QWEN_LAYER_BYTES / 4);
        for (const Mat& mt : mats)
          launch_quantize_rows(nullptr, mt.out, mt.in, synth_stream_host(seed, (uint64_t)l * 16u + mt.key), 0.02f,
                               w + mt.w_off, s + mt.s_off / 4, st);
        launch_fill_vector(s + QWEN_OFF_Q_B / 4, QWEN_HIDDEN, synth_stream_host(seed, (uint64_t)l * 16u + kTQb),
                           0.02f, 1, 0.0f, st);
        launch_fill_vector(s + QWEN_OFF_K_B / 4, QWEN_KV_WIDTH, synth_stream_host(seed, (uint64_t)l * 16u + kTKb),
                           0.02f, 1, 0.0f, st);
        launch_fill_vector(s + QWEN_OFF_V_B / 4, QWEN_KV_WIDTH, synth_stream_host(seed, (uint64_t)l * 16u + kTVb),
                           0.02f, 1, 0.0f, st);
        launch_fill_vector(s + QWEN_OFF_INPUT_LN / 4, QWEN_HIDDEN, 0, 0.0f, 0, 1.0f, st);
        launch_fill_vector(s + QWEN_OFF_POST_LN / 4, QWEN_HIDDEN, 0, 0.0f, 0, 1.0f, st);
      }
      const size_t table = (size_t)QWEN_VOCAB * QWEN_HIDDEN;
      QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&m->embed), table * 2u));
      launch_fill_bf16_table(m->embed, table, synth_stream_host(seed, kEmbedKey), 0.02f, st);
      m->vocab = QWEN_VOCAB;
      const std::vector<uint16_t> ones(QWEN_HIDDEN, 0x3F80u);  // final norm weight 1.0 (HF init)
      QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&m->head_norm), QWEN_HIDDEN * 2u));
      QWEN_HIP(hipMemcpyAsync(m->head_norm, ones.data(), QWEN_HIDDEN * 2u, hipMemcpyHostToDevice, st));
      QWEN_HIP(hipStreamSynchronize(st));
      QWEN_HIP(hipGetLastError());
      m->build_fast();
    } catch (...) {
      delete m;
      throw;
    }
    *out = m;
    return QWEN_OK;
  });
}

int qwen_hip_model_destroy(qwen_hip_model* m) {
  delete m;
  return QWEN_OK;
}

int qwen_hip_model_layers(const qwen_hip_model* m) { return m ? m->layers : 0; }

int qwen_hip_model_layer_images(qwen_hip_model* m, int layer, uint8_t* weight_ddr, float* scale_ddr) {
  if (!m || !weight_ddr || !scale_ddr || layer < 0 || layer >= m->layers) return invalid("invalid readback arguments");
  std::lock_guard<std::mutex> lock(m->mu);
  return guarded_model([&]() -> int {
    QWEN_HIP(hipStreamSynchronize(m->stream));
    QWEN_HIP(hipMemcpy(weight_ddr, m->raw_w + (size_t)layer * QWEN_LAYER_BYTES, QWEN_LAYER_BYTES,
                       hipMemcpyDeviceToHost));
    QWEN_HIP(hipMemcpy(scale_ddr, m->raw_s + (size_t)layer * (QWEN_LAYER_BYTES / 4), QWEN_LAYER_BYTES,
                       hipMemcpyDeviceToHost));
    return QWEN_OK;
  });
}

int qwen_hip_model_head_tables(qwen_hip_model* m, uint16_t* embed_bf16, uint16_t* norm_bf16) {
  if (!m || !embed_bf16 || !norm_bf16) return invalid("invalid readback arguments");
  if (!m->embed || !m->head_norm) return invalid("model has no head (synthetic models, or qwen_hip_model_set_head)");
  std::lock_guard<std::mutex> lock(m->mu);
  return guarded_model([&]() -> int {
    QWEN_HIP(hipStreamSynchronize(m->stream));
    QWEN_HIP(hipMemcpy(embed_bf16, m->embed, (size_t)m->vocab * QWEN_HIDDEN * 2u, hipMemcpyDeviceToHost));
    QWEN_HIP(hipMemcpy(norm_bf16, m->head_norm, QWEN_HIDDEN * 2u, hipMemcpyDeviceToHost));
    return QWEN_OK;
  });
}

void* qwen_hip_model_stream(qwen_hip_model* m) { return m ? static_cast<void*>(m->stream) : nullptr; }

int qwen_hip_model_synchronize(qwen_hip_model* m) {
  if (!m) return invalid("null model");
  return guarded_model([&]() -> int {
    QWEN_HIP(hipStreamSynchronize(m->stream));
    return QWEN_OK;
  });
}

int qwen_hip_model_decode_layers(qwen_hip_model* m, int mode, int first_layer, int layer_count, int batch,
                                 float* hidden, const int* positions, int max_keys, float* k_cache, float* v_cache,
                                 uint64_t seq_stride, uint64_t layer_stride) {
  if (!m || !hidden || !positions || !k_cache || !v_cache) return invalid("null argument");
  if (first_layer < 0 || layer_count <= 0 || first_layer > m->layers - layer_count) return invalid("invalid layer range");
  const int round = (mode & QWEN_FLAG_NO_BF16_ROUND) ? 0 : 1;
  const bool pre_reduce = (mode & QWEN_FLAG_SEPARATE_REDUCE) == 0;
  const bool sep_attn = (mode & QWEN_FLAG_SEPARATE_ATTN) != 0;
  mode &= ~(QWEN_FLAG_NO_BF16_ROUND | QWEN_FLAG_SEPARATE_REDUCE | QWEN_FLAG_SEPARATE_ATTN);
  if (batch <= 0 || max_keys <= 0 || max_keys > QWEN_MAX_SEQ || (mode != QWEN_MODE_ORDERED && mode != QWEN_MODE_FAST))
    return invalid("invalid decode shape or mode");
  if (mode == QWEN_MODE_FAST && (size_t)batch > kMaxDecodeBatch) return invalid("FAST decode batch above 65535 sequences");
  if (seq_stride < (uint64_t)max_keys * QWEN_KV_WIDTH || (batch > 1 && layer_stride < (uint64_t)batch * seq_stride) ||
      (layer_count > 1 && layer_stride == 0))
    return invalid("KV strides too small for max_keys / batch");
  std::lock_guard<std::mutex> lock(m->mu);
  return guarded_model([&]() -> int {
    // QWEN_SPLIT_CUS asked for a two-halves decode on CU-masked streams.  That path was removed: on
    // MI355X its results matched the oracle, but the process then hung while the model (and with it
    // the CU-masked streams) was torn down, for a cause not found.
    const char* sp = std::getenv("QWEN_SPLIT_CUS");
    if (mode == QWEN_MODE_FAST && sp && std::atoi(sp) > 0)
      throw std::runtime_error("QWEN_SPLIT_CUS: the CU-masked split decode was removed");
    if (mode == QWEN_MODE_FAST)
      m->decode_fast(first_layer, layer_count, batch, hidden, positions, max_keys, k_cache, v_cache, seq_stride,
                     layer_stride, round, pre_reduce, sep_attn);
    else
      m->decode_ordered(first_layer, layer_count, batch, hidden, positions, max_keys, k_cache, v_cache, seq_stride,
                        layer_stride, round);
    m->last = LastCall{1, mode, batch, 1, max_keys, 0, first_layer, layer_count, positions, k_cache, v_cache,
                       seq_stride, layer_stride};
    return QWEN_OK;
  });
}

int qwen_hip_model_decode(qwen_hip_model* m, int mode, int batch, float* hidden, const int* positions, int max_keys,
                          float* k_cache, float* v_cache, uint64_t seq_stride, uint64_t layer_stride) {
  if (!m) return invalid("null argument");
  return qwen_hip_model_decode_layers(m, mode, 0, m->layers, batch, hidden, positions, max_keys, k_cache, v_cache,
                                      seq_stride, layer_stride);
}

int qwen_hip_model_prefill_layers(qwen_hip_model* m, int mode, int first_layer, int layer_count, int batch,
                                  int seq_len, int past, float* hidden, float* k_cache, float* v_cache,
                                  uint64_t seq_stride, uint64_t layer_stride) {
  if (!m || !hidden || !k_cache || !v_cache) return invalid("null argument");
  if (first_layer < 0 || layer_count <= 0 || first_layer > m->layers - layer_count) return invalid("invalid layer range");
  const int round = (mode & QWEN_FLAG_NO_BF16_ROUND) ? 0 : 1;
  mode &= ~QWEN_FLAG_NO_BF16_ROUND;
  if (batch <= 0 || seq_len <= 0 || past < 0 || past > QWEN_MAX_SEQ - seq_len || seq_len > QWEN_MAX_SEQ ||
      (mode != QWEN_MODE_ORDERED && mode != QWEN_MODE_FAST))
    return invalid("invalid prefill shape, past length or mode");
  const uint64_t rows = (uint64_t)past + (uint64_t)seq_len;
  if (seq_stride < rows * QWEN_KV_WIDTH || (batch > 1 && layer_stride < (uint64_t)batch * seq_stride) ||
      (layer_count > 1 && layer_stride == 0))
    return invalid("KV strides too small for past + seq_len / batch");
  std::lock_guard<std::mutex> lock(m->mu);
  return guarded_model([&]() -> int {
    if (mode == QWEN_MODE_FAST)
      m->prefill_fast(first_layer, layer_count, batch, seq_len, past, hidden, k_cache, v_cache, seq_stride,
                      layer_stride, round);
    else
      m->prefill_ordered(first_layer, layer_count, batch, seq_len, past, hidden, k_cache, v_cache, seq_stride,
                         layer_stride, round);
    m->last = LastCall{2, mode, batch, seq_len, past + seq_len, past, first_layer, layer_count, nullptr, k_cache,
                       v_cache, seq_stride, layer_stride};
    return QWEN_OK;
  });
}

int qwen_hip_model_prefill_chunk(qwen_hip_model* m, int mode, int batch, int seq_len, int past, float* hidden,
                                 float* k_cache, float* v_cache, uint64_t seq_stride, uint64_t layer_stride) {
  if (!m) return invalid("null argument");
  return qwen_hip_model_prefill_layers(m, mode, 0, m->layers, batch, seq_len, past, hidden, k_cache, v_cache,
                                       seq_stride, layer_stride);
}

int qwen_hip_model_prefill(qwen_hip_model* m, int mode, int batch, int seq_len, float* hidden, float* k_cache,
                           float* v_cache, uint64_t seq_stride, uint64_t layer_stride) {
  return qwen_hip_model_prefill_chunk(m, mode, batch, seq_len, 0, hidden, k_cache, v_cache, seq_stride, layer_stride);
}

int qwen_hip_model_embed(qwen_hip_model* m, const int* token_ids, int count, float* hidden) {
  if (!m || !token_ids || !hidden || count <= 0) return invalid("invalid embed arguments");
  if (!m->embed) return invalid("model has no embedding table (synthetic models, or qwen_hip_model_set_head)");
  std::lock_guard<std::mutex> lock(m->mu);
  return guarded_model([&]() -> int {
    launch_embed(m->embed, m->vocab, token_ids, count, hidden, m->stream);
    QWEN_HIP(hipGetLastError());
    return QWEN_OK;
  });
}

int qwen_hip_model_set_head(qwen_hip_model* m, int vocab, const uint16_t* embed_bf16, const uint16_t* norm_bf16) {
  if (!m || !embed_bf16 || !norm_bf16 || vocab <= 0 || vocab % 128 != 0 || vocab > (1 << 24))
    return invalid("invalid head arguments (vocab must be a positive multiple of 128)");
  std::lock_guard<std::mutex> lock(m->mu);
  return guarded_model([&]() -> int {
    QWEN_HIP(hipStreamSynchronize(m->stream));
    if (m->embed) QWEN_HIP(hipFree(m->embed));
    m->embed = nullptr;
    m->vocab = 0;
    const size_t table = (size_t)vocab * QWEN_HIDDEN * 2u;
    QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&m->embed), table));
    QWEN_HIP(hipMemcpy(m->embed, embed_bf16, table, hipMemcpyHostToDevice));
    if (!m->head_norm) QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&m->head_norm), QWEN_HIDDEN * 2u));
    QWEN_HIP(hipMemcpy(m->head_norm, norm_bf16, QWEN_HIDDEN * 2u, hipMemcpyHostToDevice));
    m->vocab = vocab;
    return QWEN_OK;
  });
}

int qwen_hip_model_vocab(const qwen_hip_model* m) { return m ? m->vocab : 0; }

namespace {
int run_head(qwen_hip_model* m, const float* hidden, int count, float* logits, int* token_ids) {
  if (!m || !hidden || count <= 0 || count > (1 << 20)) return invalid("invalid head arguments");
  if (!m->embed || !m->head_norm) return invalid("model has no head (synthetic models, or qwen_hip_model_set_head)");
  std::lock_guard<std::mutex> lock(m->mu);
  return guarded_model([&]() -> int {
    void* ws = m->head_ws.get(head_workspace_bytes(count, m->vocab));
    launch_head(hidden, count, m->head_norm, m->embed, m->vocab, ws, logits, token_ids, m->stream);
    QWEN_HIP(hipGetLastError());
    return QWEN_OK;
  });
}
}  // namespace

int qwen_hip_model_logits(qwen_hip_model* m, const float* hidden, int count, float* logits) {
  if (!logits) return invalid("invalid logits buffer");
  return run_head(m, hidden, count, logits, nullptr);
}

int qwen_hip_model_greedy(qwen_hip_model* m, const float* hidden, int count, int* token_ids) {
  if (!token_ids) return invalid("invalid token id buffer");
  return run_head(m, hidden, count, nullptr, token_ids);
}

int qwen_hip_model_time_kernel(qwen_hip_model* m, int kernel, int layer, int reps, float* avg_ms) {
  if (!m || !avg_ms || reps <= 0 || layer < 0 || layer >= m->layers) return invalid("invalid timing arguments");
  std::lock_guard<std::mutex> lock(m->mu);
  const LastCall c = m->last;
  if (c.kind == 0 || c.mode != QWEN_MODE_FAST) return invalid("time_kernel needs a preceding FAST decode/prefill");
  const bool decode = c.kind == 1;
  if ((kernel == QWEN_KERNEL_ATTN_DECODE && !decode) || (kernel == QWEN_KERNEL_ATTN_PREFILL && decode))
    return invalid("kernel does not belong to the last call");
  if (layer < c.first || layer >= c.first + c.count) return invalid("layer outside the last call's layer range");
  return guarded_model([&]() -> int {
    const int T = c.batch * c.seq_len;
    const AttnDecodePlan plan = plan_attn_decode(decode ? c.batch : 1, c.max_keys);
    const AttnPrefillPlan pplan = decode ? AttnPrefillPlan{1, 1} : plan_attn_prefill(c.seq_len, c.past, c.batch);
    const qwen_hip_model::Ws w =
        decode ? m->carve(T, c.batch, plan.nsplit) : m->carve_prefill(T, c.batch, c.max_keys, pplan);
    const FastLayer& f = m->fast[layer];
    float* kc = c.k_cache + (size_t)(layer - c.first) * c.layer_stride;
    float* vc = c.v_cache + (size_t)(layer - c.first) * c.layer_stride;
    int rep = 0;
    auto once = [&]() {
      // the decode attention reads the caches of the call's layers in turn, starting at `layer`: each launch
      // streams KV rows that no recent launch has read, as in a decode step (re-reading one layer's rows would
      // be served partly from the 256 MB last-level cache)
      const size_t la = (size_t)((layer - c.first + rep++) % c.count) * c.layer_stride;
      switch (kernel) {
        case QWEN_KERNEL_ATTN_DECODE:
          // the partials launch alone (without xq no merge follows): the kernel the roofline covers
          launch_attn_decode(w.qkv, (int)kQkvRows, c.k_cache + la, c.v_cache + la, c.seq_stride, c.positions,
                             c.batch, c.max_keys, plan, w.part, w.pml, w.budget, nullptr, nullptr, w.sx, w.sums,
                             m->stream);
          break;
        case QWEN_KERNEL_GEMM_GATE_UP:
          m->gemm(w, T, QWEN_HIDDEN, QWEN_INTERMEDIATE, f.gate, f.sw_gate, nullptr, w.tmp, QWEN_INTERMEDIATE,
                  kEpiSiluMul, f.up, f.sw_up, nullptr, 0, decode ? 0 : 1);
          break;
        case QWEN_KERNEL_GEMM_DOWN:
          m->gemm(w, T, QWEN_INTERMEDIATE, QWEN_HIDDEN, f.down, f.sw_down, nullptr, w.tmp, QWEN_HIDDEN, kEpiResidual,
                  nullptr, nullptr, w.att, 1, 0);
          break;
        case QWEN_KERNEL_GEMM_QKV:
          m->gemm(w, T, QWEN_HIDDEN, (int)kQkvRows, f.qkv, f.sw_qkv, f.b_qkv, w.tmp, kQkvRows, kEpiStore);
          break;
        case QWEN_KERNEL_GEMM_O:
          m->gemm(w, T, QWEN_HIDDEN, QWEN_HIDDEN, f.o, f.sw_o, nullptr, w.tmp, QWEN_HIDDEN, kEpiStore);
          break;
        case QWEN_KERNEL_ATTN_PREFILL:
          launch_attn_prefill(w.qkv, (int)kQkvRows, kc, vc, c.seq_stride, c.seq_len, c.past, c.batch, w.kvt, pplan,
                              w.part, w.pml, w.ctx, w.xq, w.sx, w.sums, m->stream);
          break;
        default:
          throw std::runtime_error("unknown kernel id");
      }
    };
    once();  // warm
    hipEvent_t e0, e1;
    QWEN_HIP(hipEventCreate(&e0));
    QWEN_HIP(hipEventCreate(&e1));
    QWEN_HIP(hipEventRecord(e0, m->stream));
    for (int i = 0; i < reps; ++i) once();
    QWEN_HIP(hipEventRecord(e1, m->stream));
    QWEN_HIP(hipEventSynchronize(e1));
    float ms = 0.0f;
    QWEN_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    QWEN_HIP(hipGetLastError());
    *avg_ms = ms / (float)reps;
    return QWEN_OK;
  });
}

int qwen_hip_quantize_int4(const float* w, int out_dim, int in_dim, uint8_t* packed, float* scales, void* stream) {
  if (!w || !packed || !scales || out_dim <= 0 || in_dim <= 0 || in_dim % 2 || in_dim > kMaxQuantRow)
    return invalid("invalid quantizer arguments (in_dim must be even and <= 8960)");
  return guarded_model([&]() -> int {
    launch_quantize_rows(w, out_dim, in_dim, 0, 0.0f, packed, scales, static_cast<hipStream_t>(stream));
    QWEN_HIP(hipGetLastError());
    return QWEN_OK;
  });
}

int qwen_hip_fill_kv_synthetic(float* cache, uint64_t rows, uint64_t seed, void* stream) {
  if (!cache) return invalid("null cache");
  if (rows == 0) return QWEN_OK;
  return guarded_model([&]() -> int {
    launch_kv_synthetic(cache, rows, synth_stream_host(seed, 1u << 21), static_cast<hipStream_t>(stream));
    QWEN_HIP(hipGetLastError());
    return QWEN_OK;
  });
}

int qwen_hip_eval_expf(uint32_t first_bits, uint32_t stride, uint64_t n, float* y, void* stream) {
  if (!y) return invalid("null output");
  if (n == 0) return QWEN_OK;
  if (n > (1ull << 32)) return invalid("n exceeds 2^32");
  return guarded_model([&]() -> int {
    launch_eval_expf(first_bits, stride, n, y, static_cast<hipStream_t>(stream));
    QWEN_HIP(hipGetLastError());
    return QWEN_OK;
  });
}

}  // extern "C"
