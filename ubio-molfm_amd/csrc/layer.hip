// Whole layers as one call: the attention layer (node projections, attention kernels, SO(2) output linears) and the
// feed-forward block, forward and input gradient, enqueued from the host in native code.  No kernels of their own:
// the calls, their order and their arguments are those of the single entry points, so the results are bitwise
// theirs.  What they save is the host's time per launch: an evaluation of 24 atoms is some 200 launches of 8 us of
// kernel on average, and forming each launch's arguments in Python took 4.6 ms per evaluation, three times the
// kernels' 1.5 ms; with these calls it takes 2.0 ms.
#include <algorithm>

#include "common.h"
#include "../../include/e2v2.h"

namespace e2v2 {
namespace {

constexpr int kOfM[9] = {0, 1, 1, 1, 2, 2, 2, 2, 2};    // degree of each m-row

#define E2V2_CALL(expr)                 \
  do {                                  \
    if (int rc_ = (expr)) return rc_;   \
  } while (0)

struct Mat {            // [batch][m][k] operand or result
  const void* p;
  int64_t ld, bs;
};

e2v2_gemm_args gemm_of(const Mat& a, bool a_bf16, const void* packed, int n_w, int pieces, const Mat& c, bool c_bf16,
                       int m, int n, int k, int batch) {
  e2v2_gemm_args G{};
  G.a = a.p; G.lda = a.ld; G.a_bs = a.bs; G.a_bf16 = a_bf16;
  G.b = packed; G.n_w = n_w; G.pieces = pieces;
  G.c = const_cast<void*>(c.p); G.ldc = c.ld; G.c_bs = c.bs; G.c_bf16 = c_bf16;
  G.m = m; G.n = n; G.k = k; G.batch = batch;
  return G;
}
void by_degree(e2v2_gemm_args& G, int first = 0) {
  for (int b = 0; b < G.batch; ++b) G.widx[b] = kOfM[first + b];
}
void with_bias(e2v2_gemm_args& G, const float* bias, int batches, int64_t bs = 0) {
  G.bias = bias;
  G.bias_batches = bias ? batches : 0;
  G.bias_bs = bs;
}

// The saved and scratch arrays of an attention layer, one after another (multiples of 16 bytes per node).
struct Layout {
  int64_t n, at = 0;
  char* base;
  char* take(int64_t bytes_per_node) {
    char* p = base ? base + at : nullptr;
    at += n * bytes_per_node;
    return p;
  }
};
struct Saved {
  char *y, *h1, *st, *qk, *v, *so2, *mrow, *srow, *cnt;
  int64_t per_node;
};
int so2_rows(const e2v2_attn_layer& W) { return W.zero_order ? 9 : 20; }
Saved saved_of(const e2v2_attn_layer& W, int64_t n, void* base) {
  const int es = W.pieces == 1 ? 2 : 4;
  Layout L{n, 0, static_cast<char*>(base)};
  Saved S;
  S.y = L.take((int64_t)9 * 4 * W.hid * es);
  S.h1 = L.take((int64_t)2 * W.hid * 4);
  S.qk = L.take((int64_t)2 * W.n_out * es);
  S.v = L.take((int64_t)9 * W.c * es);
  S.so2 = L.take((int64_t)so2_rows(W) * W.c * es);
  S.mrow = L.take(W.heads * 4);
  S.srow = L.take(W.heads * 4);
  S.cnt = L.take(W.heads * 4);
  S.st = L.take(16);                 // last: all before it stay on 128-byte lines, whose rows the gathers read
  S.per_node = n ? L.at / n : 0;
  return S;
}
struct FwdScratch {
  float *hq, *hk, *a;
  int64_t per_node;
};
FwdScratch fwd_scratch(const e2v2_attn_layer& W, int64_t n, void* base) {
  Layout L{n, 0, static_cast<char*>(base)};
  FwdScratch S;
  S.hq = reinterpret_cast<float*>(L.take((int64_t)3 * W.hid * 4));
  S.hk = reinterpret_cast<float*>(L.take((int64_t)3 * W.hid * 4));
  S.a = reinterpret_cast<float*>(L.take((int64_t)2 * W.hid * 4));
  S.per_node = n ? L.at / n : 0;
  return S;
}
struct BwdScratch {
  char* gso2;
  float *dq, *dk, *dv, *ga, *gh1, *gh;
  int64_t per_node;
};
BwdScratch bwd_scratch(const e2v2_attn_layer& W, int64_t n, void* base) {
  Layout L{n, 0, static_cast<char*>(base)};
  BwdScratch S;
  S.gso2 = L.take((int64_t)so2_rows(W) * W.c * (W.pieces == 1 ? 2 : 4));
  S.dq = reinterpret_cast<float*>(L.take((int64_t)W.n_out * 4));
  S.dk = reinterpret_cast<float*>(L.take((int64_t)W.n_out * 4));
  S.dv = reinterpret_cast<float*>(L.take((int64_t)9 * W.c * 4));
  S.ga = reinterpret_cast<float*>(L.take((int64_t)2 * W.hid * 4));
  S.gh1 = reinterpret_cast<float*>(L.take((int64_t)2 * W.hid * 4));
  S.gh = reinterpret_cast<float*>(L.take((int64_t)6 * W.hid * 4));
  S.per_node = n ? L.at / n : 0;
  return S;
}

int check_layer(const e2v2_attn_layer* W, const char* who) {
  E2V2_REQUIRE(W && (W->pieces == 1 || W->pieces == 3) && W->hid > 0 && W->hid % 128 == 0 && W->c == 256 &&
                   W->n_out == 1024 && W->heads == 128,
               "%s: built for 256 channels, 128 heads of 8 and a multiple of 128 hidden pairs", who);
  E2V2_REQUIRE(W->qk_fwd && W->qk_bwd && W->v_fwd && W->h1_fwd && W->h1_bwd && W->h2_fwd && W->h2_bwd &&
                   W->out_fwd[0] && W->out_fwd[1] && W->out_fwd[2] && W->out_bwd[0] && W->out_bwd[1] && W->out_bwd[2],
               "%s: null packed weight", who);
  return 0;
}

// The three per-degree output GEMMs in dispatch order (the longest k first forward, the largest result first
// backward; ties keep the degree order).
void out_order(const e2v2_attn_layer& W, bool backward, int (&o)[3]) {
  for (int i = 0; i < 3; ++i) o[i] = i;
  std::stable_sort(o, o + 3, [&](int a, int b) {
    const int64_t x = (int64_t)W.out_cnt[a] * (backward ? 2 * a + 1 : 1);
    const int64_t y = (int64_t)W.out_cnt[b] * (backward ? 2 * b + 1 : 1);
    return x > y;
  });
}
}  // namespace
}  // namespace e2v2

using namespace e2v2;

E2V2_API int e2v2_attn_layer_bytes(const e2v2_attn_layer* W, int64_t* saved, int64_t* fwd, int64_t* bwd) {
  if (int rc = check_layer(W, "attn_layer_bytes")) return rc;
  E2V2_REQUIRE(saved && fwd && bwd, "attn_layer_bytes: null pointer");
  *saved = saved_of(*W, 1, nullptr).per_node;
  *fwd = fwd_scratch(*W, 1, nullptr).per_node;
  *bwd = bwd_scratch(*W, 1, nullptr).per_node;
  return 0;
}

E2V2_API int e2v2_attn_layer_fwd(const e2v2_attn_layer* Wp, const e2v2_attn_args* args, const float* x, void* saved,
                                 void* scratch, float* out, hipStream_t s) {
  if (int rc = check_layer(Wp, "attn_layer_fwd")) return rc;
  const e2v2_attn_layer& W = *Wp;
  E2V2_REQUIRE(args && args->zero_order == W.zero_order && args->act_bf16 == (W.pieces == 1),
               "attn_layer_fwd: the attention arguments do not match the layer");
  const int n = args->n_rows;
  if (n == 0) return 0;
  E2V2_REQUIRE(x && saved && scratch && out, "attn_layer_fwd: null operand");
  const bool bf = W.pieces == 1;
  const int hid = W.hid, c = W.c;
  const Saved S = saved_of(W, n, saved);
  const FwdScratch T = fwd_scratch(W, n, scratch);
  E2V2_CALL(e2v2_qk_proj_fwd_s3(x, W.qk_fwd, W.qk_bias, S.y, T.hq, T.hk, n, hid, c, W.pieces, bf, s));
  const int64_t nc = (int64_t)n * c, nh = (int64_t)n * hid, no = (int64_t)n * W.n_out;
  e2v2_gemm_args g[3];
  g[0] = gemm_of({T.hq, 3 * hid, T.hk - T.hq}, false, W.h1_fwd, 2, W.pieces, {S.h1, hid, nh}, false, n, hid, 3 * hid, 2);
  g[0].widx[1] = 1;
  with_bias(g[0], W.h1_bias, 2, hid);
  g[1] = gemm_of({x, c, nc}, false, W.v_fwd, 3, W.pieces, {S.v, c, nc}, bf, n, c, c, 9);
  by_degree(g[1]);
  with_bias(g[1], W.v_bias, 1);
  E2V2_CALL(e2v2_gemm_s3_grouped(g, 2, s));
  const float* h1 = reinterpret_cast<const float*>(S.h1);
  for (int b = 0; b < 2; ++b)
    E2V2_CALL(e2v2_ln_silu_fwd(h1 + b * nh, W.ln_g[b], W.ln_b[b], T.a + b * nh,
                               reinterpret_cast<float*>(S.st) + (int64_t)2 * b * n, n, hid, W.ln_eps[b], s));
  e2v2_gemm_args h2 = gemm_of({T.a, hid, nh}, false, W.h2_fwd, 2, W.pieces, {S.qk, W.n_out, no}, bf, n, W.n_out, hid, 2);
  h2.widx[1] = 1;
  with_bias(h2, W.h2_bias, 2, W.n_out);
  E2V2_CALL(e2v2_gemm_s3(&h2, s));
  e2v2_attn_args A = *args;
  A.q = S.qk;
  A.k = S.qk + no * (bf ? 2 : 4);
  A.v = S.v;
  E2V2_CALL(e2v2_attn_fwd(&A, S.so2, reinterpret_cast<float*>(S.mrow), reinterpret_cast<float*>(S.srow),
                          reinterpret_cast<int32_t*>(S.cnt), s));
  int o[3];
  out_order(W, false, o);
  for (int i = 0; i < 3; ++i) {
    const int l = o[i], k = W.out_cnt[l] * c;
    g[i] = gemm_of({S.so2 + (int64_t)W.out_start[l] * n * (bf ? 2 : 4), k, (int64_t)n * k}, bf, W.out_fwd[l], 1, W.pieces,
                   {out + (int64_t)l * l * nc, c, nc}, false, n, c, k, 2 * l + 1);
    if (l == 0) with_bias(g[i], W.out_bias, 1);
  }
  return e2v2_gemm_s3_grouped(g, 3, s);
}

E2V2_API int e2v2_attn_layer_bwd(const e2v2_attn_layer* Wp, const e2v2_attn_args* args, const float* gout,
                                 const void* saved, void* scratch, void* workspace, size_t workspace_bytes, float* gx,
                                 float* ddvec, float* ddist, hipStream_t s) {
  if (int rc = check_layer(Wp, "attn_layer_bwd")) return rc;
  const e2v2_attn_layer& W = *Wp;
  E2V2_REQUIRE(args && args->zero_order == W.zero_order && args->act_bf16 == (W.pieces == 1),
               "attn_layer_bwd: the attention arguments do not match the layer");
  const int n = args->n_rows;
  if (n == 0) return 0;
  E2V2_REQUIRE(gout && saved && scratch && gx, "attn_layer_bwd: null operand");
  const bool bf = W.pieces == 1;
  const int hid = W.hid, c = W.c, es = bf ? 2 : 4;
  const Saved S = saved_of(W, n, const_cast<void*>(saved));
  const BwdScratch T = bwd_scratch(W, n, scratch);
  const int64_t nc = (int64_t)n * c, nh = (int64_t)n * hid, no = (int64_t)n * W.n_out;
  e2v2_gemm_args g[3];
  int o[3];
  out_order(W, true, o);
  for (int i = 0; i < 3; ++i) {
    const int l = o[i], k = W.out_cnt[l] * c;
    g[i] = gemm_of({gout + (int64_t)l * l * nc, c, nc}, false, W.out_bwd[l], 1, W.pieces,
                   {T.gso2 + (int64_t)W.out_start[l] * n * es, k, (int64_t)n * k}, bf, n, k, c, 2 * l + 1);
  }
  E2V2_CALL(e2v2_gemm_s3_grouped(g, 3, s));
  e2v2_attn_args A = *args;
  A.q = S.qk;
  A.k = S.qk + no * es;
  A.v = S.v;
  E2V2_CALL(e2v2_attn_bwd(&A, T.gso2, S.so2, reinterpret_cast<const float*>(S.mrow),
                          reinterpret_cast<const float*>(S.srow), reinterpret_cast<const int32_t*>(S.cnt), ddvec, ddist,
                          T.dq, T.dk, T.dv, workspace, workspace_bytes, s));
  e2v2_gemm_args h2 = gemm_of({T.dq, W.n_out, T.dk - T.dq}, false, W.h2_bwd, 2, W.pieces, {T.ga, hid, nh}, false, n, hid,
                              W.n_out, 2);
  h2.widx[1] = 1;
  E2V2_CALL(e2v2_gemm_s3(&h2, s));
  const float* h1 = reinterpret_cast<const float*>(S.h1);
  for (int b = 0; b < 2; ++b)
    E2V2_CALL(e2v2_ln_silu_bwd(h1 + b * nh, W.ln_g[b], W.ln_b[b],
                               reinterpret_cast<const float*>(S.st) + (int64_t)2 * b * n, T.ga + b * nh, T.gh1 + b * nh,
                               n, hid, s));
  e2v2_gemm_args hb = gemm_of({T.gh1, hid, nh}, false, W.h1_bwd, 2, W.pieces, {T.gh, 3 * hid, 3 * nh}, false, n, 3 * hid,
                              hid, 2);
  hb.widx[1] = 1;
  E2V2_CALL(e2v2_gemm_s3(&hb, s));
  return e2v2_qk_proj_bwd_s3(S.y, T.gh, T.gh + 3 * nh, W.qk_bwd, T.dv, gx, n, hid, c, c, W.pieces, bf, s);
}

static int check_ffn(const e2v2_ffn_layer* W, const char* who) {
  E2V2_REQUIRE(W && (W->pieces == 1 || W->pieces == 3) && W->c == 256 && W->hidden == 256,
               "%s: built for 256 channels and 256 hidden channels", who);
  E2V2_REQUIRE(W->w1_fwd && W->w1_bwd && W->gate_fwd && W->gate_bwd && W->w2_fwd && W->w2_bwd, "%s: null packed weight",
               who);
  return 0;
}

E2V2_API int e2v2_ffn_layer_fwd(const e2v2_ffn_layer* Wp, int n, const float* x, const float* res, float* h, float* sc,
                                float* y, hipStream_t s) {
  if (int rc = check_ffn(Wp, "ffn_layer_fwd")) return rc;
  const e2v2_ffn_layer& W = *Wp;
  if (n <= 0) return 0;
  E2V2_REQUIRE(x && h && sc && y, "ffn_layer_fwd: null operand");
  const int c = W.c, d = W.hidden;
  const int64_t nc = (int64_t)n * c, nd = (int64_t)n * d;
  e2v2_gemm_args g[2];
  g[0] = gemm_of({x, c, nc}, false, W.w1_fwd, 3, W.pieces, {h, d, nd}, false, n, d, c, 9);
  by_degree(g[0]);
  with_bias(g[0], W.b1, 1);
  g[1] = gemm_of({x, c, nc}, false, W.gate_fwd, 1, W.pieces, {sc, 3 * d, 3 * nd}, false, n, 3 * d, c, 1);
  with_bias(g[1], W.gate_b, 1);
  E2V2_CALL(e2v2_gemm_s3_grouped(g, 2, s));
  e2v2_gemm_args o = gemm_of({h, d, nd}, false, W.w2_fwd, 3, W.pieces, {y, c, nc}, false, n, c, d, 9);
  by_degree(o);
  with_bias(o, W.b2, 1);
  o.r = res;
  o.ldr = c;
  o.r_bs = nc;
  return e2v2_gemm_s3_gated(&o, sc, 3 * d, W.k1, W.k2, s);
}

E2V2_API int e2v2_ffn_layer_bwd(const e2v2_ffn_layer* Wp, int n, const float* gout, const float* h, const float* sc,
                                float* scratch, float* gx, hipStream_t s) {
  if (int rc = check_ffn(Wp, "ffn_layer_bwd")) return rc;
  const e2v2_ffn_layer& W = *Wp;
  if (n <= 0) return 0;
  E2V2_REQUIRE(gout && h && sc && scratch && gx, "ffn_layer_bwd: null operand");
  const int c = W.c, d = W.hidden;
  const int64_t nc = (int64_t)n * c, nd = (int64_t)n * d;
  float *gy = scratch, *gh = scratch + 9 * nd, *gsc = scratch + 18 * nd;      // 21 n hidden floats
  e2v2_gemm_args o = gemm_of({gout, c, nc}, false, W.w2_bwd, 3, W.pieces, {gy, d, nd}, false, n, d, c, 9);
  by_degree(o);
  E2V2_CALL(e2v2_gemm_s3(&o, s));
  E2V2_CALL(e2v2_gate_bwd(sc, h, gy, gsc, gh, n, W.k1, W.k2, s));
  e2v2_gemm_args g[2];
  g[0] = gemm_of({gsc, 3 * d, 3 * nd}, false, W.gate_bwd, 1, W.pieces, {gx, c, nc}, false, n, c, 3 * d, 1);
  g[1] = gemm_of({gh + nd, d, nd}, false, W.w1_bwd, 3, W.pieces, {gx + nc, c, nc}, false, n, c, d, 8);
  by_degree(g[1], 1);
  return e2v2_gemm_s3_grouped(g, 2, s);
}
