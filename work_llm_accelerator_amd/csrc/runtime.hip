// Host runtime: arena, RoPE tables, layer staging and the per-layer executors.
#include "runtime.hpp"

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <stdexcept>
#include <string>

#include "kernels.hpp"

namespace qwen {

namespace {
thread_local std::string g_last_error;
}
void set_last_error(const std::string& msg) { g_last_error = msg; }
const char* last_error_cstr() { return g_last_error.c_str(); }

void hip_check(hipError_t e, const char* what) {
  if (e != hipSuccess) throw HipError{e, what};
}

HostLayer resolve_host_layer(const uint8_t* wd, const float* sd, uint64_t wb, uint64_t sb) {
  HostLayer p;
  p.ln = sd + (sb + QWEN_OFF_INPUT_LN) / 4;
  p.post_ln = sd + (sb + QWEN_OFF_POST_LN) / 4;
  p.qw = wd + wb + QWEN_OFF_Q_W;
  p.kw = wd + wb + QWEN_OFF_K_W;
  p.vw = wd + wb + QWEN_OFF_V_W;
  p.ow = wd + wb + QWEN_OFF_O_W;
  p.qb = sd + (sb + QWEN_OFF_Q_B) / 4;
  p.kb = sd + (sb + QWEN_OFF_K_B) / 4;
  p.vb = sd + (sb + QWEN_OFF_V_B) / 4;
  p.qs = sd + (sb + QWEN_OFF_Q_S) / 4;
  p.ks = sd + (sb + QWEN_OFF_K_S) / 4;
  p.vs = sd + (sb + QWEN_OFF_V_S) / 4;
  p.os = sd + (sb + QWEN_OFF_O_S) / 4;
  p.gs = sd + (sb + QWEN_OFF_GATE_S) / 4;
  p.us = sd + (sb + QWEN_OFF_UP_S) / 4;
  p.ds = sd + (sb + QWEN_OFF_DOWN_S) / 4;
  p.gw = wd + wb + QWEN_OFF_GATE_W;
  p.uw = wd + wb + QWEN_OFF_UP_W;
  p.dw = wd + wb + QWEN_OFF_DOWN_W;
  return p;
}

// ---------------------------------------------------------------------------------------------
Arena::~Arena() {
  // Process teardown: the HIP runtime may already be gone; leave the block to the driver.
}

void Arena::reserve(size_t bytes) {
  if (bytes <= cap_) return;
  if (used_ != 0) throw std::runtime_error("arena grown while in use");
  if (base_) {
    QWEN_HIP(hipDeviceSynchronize());
    QWEN_HIP(hipFree(base_));
    base_ = nullptr;
    cap_ = 0;
  }
  const size_t want = bytes + (bytes >> 3) + (1u << 20);
  QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&base_), want));
  cap_ = want;
}

void* Arena::alloc(size_t bytes) {
  const size_t off = (used_ + 255u) & ~size_t(255u);
  if (off + bytes > cap_) throw std::runtime_error("arena capacity exceeded");
  used_ = off + bytes;
  return base_ + off;
}

// ---------------------------------------------------------------------------------------------
void Staging::begin(Arena& a) {
  if (!host_) QWEN_HIP(hipHostMalloc(reinterpret_cast<void**>(&host_), kBytes, hipHostMallocDefault));
  dev_ = static_cast<char*>(a.alloc(kBytes));
  used_ = 0;
  n_results_ = 0;
}

size_t Staging::take(size_t bytes) {
  const size_t at = (used_ + 255u) & ~size_t(255u);
  if (at + bytes > kBytes) throw std::runtime_error("staging capacity exceeded");
  used_ = at + bytes;
  return at;
}

void Staging::send(hipStream_t st) {
  pending_ = true;
  QWEN_HIP(hipMemcpyAsync(dev_, host_, used_, hipMemcpyHostToDevice, st));
}

void Staging::collect(void* host, const void* dev, size_t bytes, hipStream_t st) {
  if (n_results_ == 4) throw std::runtime_error("staging: too many results");
  const size_t at = take(bytes);
  pending_ = true;
  QWEN_HIP(hipMemcpyAsync(host_ + at, dev, bytes, hipMemcpyDeviceToHost, st));
  results_[n_results_++] = Result{host, at, bytes};
}

void Staging::deliver() {
  for (int i = 0; i < n_results_; ++i) std::memcpy(results_[i].host, host_ + results_[i].at, results_[i].bytes);
  n_results_ = 0;
}

// ---------------------------------------------------------------------------------------------
Runtime& Runtime::get() {
  static Runtime* rt = new Runtime();  // never destroyed: HIP objects outlive static teardown
  return *rt;
}

Runtime::Runtime() {
  // Default-priority stream (no priority other than the default is ever used).
  QWEN_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
}

void decode_rope_row_host(int position, float* out) {
  // qwen_decode_attention_kernel.cpp:29-42: angle in double with libm pow, cos, sin.
  for (int p = 0; p < QWEN_HEAD_DIM / 2; ++p) {
    const double angle = static_cast<double>(position) *
                         std::pow(static_cast<double>(QWEN_ROPE_THETA),
                                  -2.0 * static_cast<double>(p) / static_cast<double>(QWEN_HEAD_DIM));
    out[p] = static_cast<float>(std::cos(angle));
    out[64 + p] = static_cast<float>(std::sin(angle));
  }
}

const float* Runtime::prefill_rope(int positions) {
  if (positions <= prefill_rope_rows_) return prefill_rope_;
  int rows = 256;
  while (rows < positions) rows *= 2;
  if (rows > QWEN_MAX_SEQ) rows = QWEN_MAX_SEQ;
  float* fresh = nullptr;
  QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&fresh), sizeof(float) * 128u * (size_t)rows));
  launch_rope_table_prefill(fresh, 0, rows, stream);
  QWEN_HIP(hipGetLastError());
  QWEN_HIP(hipStreamSynchronize(stream));
  if (prefill_rope_) QWEN_HIP(hipFree(prefill_rope_));
  prefill_rope_ = fresh;
  prefill_rope_rows_ = rows;
  return prefill_rope_;
}

const float* Runtime::decode_rope(int positions) {
  if (positions <= decode_rope_rows_) return decode_rope_;
  int rows = 256;
  while (rows < positions) rows *= 2;
  if (rows > QWEN_MAX_SEQ) rows = QWEN_MAX_SEQ;
  std::vector<float> host((size_t)rows * 128u);
  for (int r = 0; r < rows; ++r) decode_rope_row_host(r, &host[(size_t)r * 128u]);
  float* fresh = nullptr;
  QWEN_HIP(hipMalloc(reinterpret_cast<void**>(&fresh), sizeof(float) * host.size()));
  QWEN_HIP(hipMemcpy(fresh, host.data(), sizeof(float) * host.size(), hipMemcpyHostToDevice));
  if (decode_rope_) QWEN_HIP(hipFree(decode_rope_));
  decode_rope_ = fresh;
  decode_rope_rows_ = rows;
  return decode_rope_;
}

// ---------------------------------------------------------------------------------------------
size_t staged_layer_bytes() { return QWEN_LAYER_BYTES + 64u * 256u + Staging::kBytes; }

DevLayer stage_layer(Arena& a, Staging& small, const HostLayer& h, hipStream_t st) {
  DevLayer d;
  d.qw = stage_in(a, h.qw, QWEN_Q_WEIGHT_BYTES, st);
  d.kw = stage_in(a, h.kw, QWEN_K_WEIGHT_BYTES, st);
  d.vw = stage_in(a, h.vw, QWEN_V_WEIGHT_BYTES, st);
  d.ow = stage_in(a, h.ow, QWEN_O_WEIGHT_BYTES, st);
  d.gw = stage_in(a, h.gw, QWEN_GATE_WEIGHT_BYTES, st);
  d.uw = stage_in(a, h.uw, QWEN_UP_WEIGHT_BYTES, st);
  d.dw = stage_in(a, h.dw, QWEN_DOWN_WEIGHT_BYTES, st);
  d.ln = small.add(h.ln, QWEN_HIDDEN);
  d.post_ln = small.add(h.post_ln, QWEN_HIDDEN);
  d.qb = small.add(h.qb, QWEN_HIDDEN);
  d.kb = small.add(h.kb, QWEN_KV_WIDTH);
  d.vb = small.add(h.vb, QWEN_KV_WIDTH);
  d.qs = small.add(h.qs, QWEN_HIDDEN);
  d.ks = small.add(h.ks, QWEN_KV_WIDTH);
  d.vs = small.add(h.vs, QWEN_KV_WIDTH);
  d.os = small.add(h.os, QWEN_HIDDEN);
  d.gs = small.add(h.gs, QWEN_INTERMEDIATE);
  d.us = small.add(h.us, QWEN_INTERMEDIATE);
  d.ds = small.add(h.ds, QWEN_HIDDEN);
  return d;
}

// ---------------------------------------------------------------------------------------------
// Executors.  Intermediates come from the arena; sizes in floats per token:
//   xn 1536, q 1536, k 256, v 256, ctx 1536 (attention);  pn 1536, s 8960 (MLP).
// The attention and MLP executors each take their own part, so one token's layer needs the sum.
namespace {
void carve_attention_part(DecodeWorkspace& w, float* p, size_t T) {
  auto take = [&](size_t n) {
    float* r = p;
    p += up64(n);
    return r;
  };
  w.xn = take(T * QWEN_HIDDEN);
  w.q = take(T * QWEN_HIDDEN);
  w.k = take(T * QWEN_KV_WIDTH);
  w.v = take(T * QWEN_KV_WIDTH);
  w.ctx = take(T * QWEN_HIDDEN);
}

void carve_mlp_part(DecodeWorkspace& w, float* p, size_t T) {
  auto take = [&](size_t n) {
    float* r = p;
    p += up64(n);
    return r;
  };
  w.pn = take(T * QWEN_HIDDEN);
  w.s = take(T * QWEN_INTERMEDIATE);
}
}  // namespace

// Three arena allocations (attention part, its scores, MLP part), each aligned to 256 bytes.
size_t decode_workspace_bytes(int tokens, int max_keys) {
  return (decode_workspace_floats(tokens) + attention_ordered_scores(tokens, max_keys)) * sizeof(float) + 3u * 256u;
}
// run_prefill_attention's xn, q, ctx, scores and run_prefill_mlp's pn, s: six allocations.
size_t prefill_workspace_bytes(int tokens, int past) {
  const size_t T = (size_t)tokens;
  return (4u * T * QWEN_HIDDEN + T * QWEN_INTERMEDIATE + attention_ordered_scores(tokens, past + tokens)) *
             sizeof(float) + 6u * 256u;
}

DecodeWorkspace carve_decode_workspace(float* base, int tokens) {
  const size_t T = (size_t)tokens;
  DecodeWorkspace w;
  carve_attention_part(w, base, T);
  carve_mlp_part(w, base + decode_attention_floats(T), T);
  return w;
}

namespace {

// Fused Q/K/V projection of T rows; normed: x is normalized already.
OrdProject qkv_project(const DevLayer& L, const float* x, int T, float* q, float* k, float* v) {
  OrdProject p;
  p.seg[0] = OrdSegment{L.qw, L.qs, L.qb, q, QWEN_HIDDEN, QWEN_HIDDEN};
  p.seg[1] = OrdSegment{L.kw, L.ks, L.kb, k, QWEN_KV_WIDTH, QWEN_KV_WIDTH};
  p.seg[2] = OrdSegment{L.vw, L.vs, L.vb, v, QWEN_KV_WIDTH, QWEN_KV_WIDTH};
  p.x = x;
  p.tokens = T;
  p.in_dim = QWEN_HIDDEN;
  return p;
}

OrdProject row_project(const float* x, int T, int in_dim, const uint8_t* w, const float* scale, float* y,
                       const float* residual) {
  OrdProject p;
  p.seg[0] = OrdSegment{w, scale, nullptr, y, QWEN_HIDDEN, QWEN_HIDDEN};
  p.x = x;
  p.tokens = T;
  p.in_dim = in_dim;
  p.residual = residual;
  return p;
}

// The MLP of T rows: s = SiLU(gate) * up of the normalized rows, then out = att + down(s).
void run_mlp(const DevLayer& L, const float* att, int T, float* out, float* pn, float* s, bool prefill,
             hipStream_t st) {
  OrdProject g;
  g.seg[0] = OrdSegment{L.gw, L.gs, nullptr, s, QWEN_INTERMEDIATE, QWEN_INTERMEDIATE};
  g.seg[1] = OrdSegment{L.uw, L.us, nullptr, nullptr, QWEN_INTERMEDIATE, QWEN_INTERMEDIATE};
  g.tokens = T;
  g.in_dim = QWEN_HIDDEN;
  g.prefill = prefill ? 1 : 0;
  if (T == 1 && !prefill) {
    g.x = att;
    g.norm_w = L.post_ln;
  } else {
    launch_rmsnorm_ordered(att, L.post_ln, pn, T, prefill, st);
    g.x = pn;
  }
  launch_gate_up_ordered(g, st);
  launch_project_ordered(row_project(s, T, QWEN_INTERMEDIATE, L.dw, L.ds, out, att), st);
  QWEN_HIP(hipGetLastError());
}

}  // namespace

void run_decode_attention_ws(const DevLayer& L, const float* x, const DecodeBatch& b, float* att,
                             const DecodeWorkspace& w, hipStream_t st) {
  const int T = b.tokens;
  const bool norm = ordered_chain_shape(QWEN_QKV_ROWS, T);  // the RMSNorm inside the projection's blocks
  if (!norm) launch_rmsnorm_ordered(x, L.ln, w.xn, T, false, st);
  OrdProject p = qkv_project(L, norm ? x : w.xn, T, w.q, w.k, w.v);
  p.norm_w = norm ? L.ln : nullptr;
  launch_project_ordered(p, st);
  // One sequence rotates and appends inside the scores launch.  With several, any of them may read rows that
  // another appends (caches that share rows), so the append is a launch before the scores.
  const bool fuse_rope = T == 1 && w.scores;
  if (!fuse_rope)
    launch_rope_append_decode(w.q, w.k, w.v, b.pos, b.rope, b.rope_per_token, b.k_cache, b.v_cache, b.cache_stride,
                              b.max_keys, T, st);
  if (w.scores) {
    OrdAttentionArgs a;
    a.q = w.q;
    a.k_cache = b.k_cache;
    a.v_cache = b.v_cache;
    a.cache_stride = b.cache_stride;
    a.pos = b.pos;
    a.max_keys = b.max_keys;
    a.ctx = w.ctx;
    if (fuse_rope) {
      a.k_new = w.k;
      a.v_new = w.v;
      a.rope = b.rope;
      a.rope_rows_are_tokens = b.rope_per_token;
    }
    launch_attention_ordered_split(a, T, w.scores, st);
  } else {
    launch_attention_ordered(w.q, b.k_cache, b.v_cache, b.cache_stride, b.pos, b.max_keys, T, w.ctx, st);
  }
  launch_project_ordered(row_project(w.ctx, T, QWEN_HIDDEN, L.ow, L.os, att, nullptr), st);
  QWEN_HIP(hipGetLastError());
}

void run_decode_mlp_ws(const DevLayer& L, const float* att, int T, float* out, const DecodeWorkspace& w,
                       hipStream_t st) {
  run_mlp(L, att, T, out, w.pn, w.s, false, st);
}

void run_decode_attention(const DevLayer& L, const float* x, const DecodeBatch& b, float* att, Arena& a,
                          hipStream_t st) {
  DecodeWorkspace w{};
  carve_attention_part(w, a.alloc_n<float>(decode_attention_floats((size_t)b.tokens)), (size_t)b.tokens);
  w.scores = a.alloc_n<float>(attention_ordered_scores(b.tokens, b.max_keys));
  run_decode_attention_ws(L, x, b, att, w, st);
}

void run_decode_mlp(const DevLayer& L, const float* att, int T, float* out, Arena& a, hipStream_t st) {
  DecodeWorkspace w{};
  carve_mlp_part(w, a.alloc_n<float>(decode_mlp_floats((size_t)T)), (size_t)T);
  run_decode_mlp_ws(L, att, T, out, w, st);
}

void run_prefill_attention(const DevLayer& L, const float* x, int T, int past, const float* rope, float* k_rows,
                           float* v_rows, float* att, Arena& a, hipStream_t st) {
  float* k_new = k_rows + (size_t)past * QWEN_KV_WIDTH;
  float* v_new = v_rows + (size_t)past * QWEN_KV_WIDTH;
  float* xn = a.alloc_n<float>((size_t)T * QWEN_HIDDEN);
  float* q = a.alloc_n<float>((size_t)T * QWEN_HIDDEN);
  float* ctx = a.alloc_n<float>((size_t)T * QWEN_HIDDEN);
  float* scores = a.alloc_n<float>(attention_ordered_scores(T, past + T));
  launch_rmsnorm_ordered(x, L.ln, xn, T, true, st);
  launch_project_ordered(qkv_project(L, xn, T, q, k_new, v_new), st);
  launch_rope_prefill(q, k_new, rope + (size_t)past * 128, T, st);
  OrdAttentionArgs args;
  args.q = q;
  args.k_cache = k_rows;
  args.v_cache = v_rows;
  args.max_keys = past + T;
  args.prefill = true;
  args.past = past;
  args.ctx = ctx;
  launch_attention_ordered_split(args, T, scores, st);
  launch_project_ordered(row_project(ctx, T, QWEN_HIDDEN, L.ow, L.os, att, nullptr), st);
  QWEN_HIP(hipGetLastError());
}

void run_prefill_mlp(const DevLayer& L, const float* att, int T, float* out, Arena& a, hipStream_t st) {
  float* pn = a.alloc_n<float>((size_t)T * QWEN_HIDDEN);
  float* s = a.alloc_n<float>((size_t)T * QWEN_INTERMEDIATE);
  run_mlp(L, att, T, out, pn, s, true, st);
}

}  // namespace qwen
