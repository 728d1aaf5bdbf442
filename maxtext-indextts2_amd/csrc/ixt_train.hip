// ixt_train.hip -- C ABI of the training step (include/ixt_train.h) over ixt_train_kernels.h.  Host code: buffer ownership, launch order.
// Reference: MaxText/train.py:255-472 (loss_fn, train_step), layers/* in MODEL_MODE_TRAIN, max_utils.py:563-654, maxtext_utils.py:825-846,
// optimizers.py:28-38.  Parameters, gradients and AdamW state live in FLAT f32 device buffers owned by the caller (so that the data-parallel
// exchange -- RCCL reduce-scatter + all-gather through torch.distributed -- works on them directly); this file owns activations and workspaces.
#include "../../include/ixt_train.h"
#include "ixt_kernels.h"
#include "ixt_train_kernels.h"
#include "ixt_train_attn.h"

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <initializer_list>
#include <string>
#include <vector>

static thread_local char t_err[512] = "";
static int t_set_err(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(t_err, sizeof(t_err), fmt, ap);
  va_end(ap);
  return code;
}
extern "C" const char* ixt_train_last_error(void) { return t_err; }
#define TCHK(expr)                                                                                                          \
  do {                                                                                                                      \
    hipError_t e_ = (expr);                                                                                                 \
    if (e_ != hipSuccess) return t_set_err(IXT_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
  } while (0)
#define TLAUNCH() TCHK(hipGetLastError())
#define TTRY(x) do { int rc_ = (x); if (rc_ != IXT_OK) return rc_; } while (0)

struct ParamInfo { std::string name; long offset, numel; };

struct LayerAct {   // saved for the backward pass
  bf16_t *h_in, *xn1, *q, *k, *v, *P, *ao, *h_mid, *xn2, *a, *b, *act;
  float *r1, *r2;
};

struct ixt_trainer {
  ixt_train_config cfg;
  int E, H, D, F, V, L, B, S, T, QN, Tc;
  int KVH, G, KN;           // grouped-query attention: kv heads, query heads per kv head, KVH * D
  std::vector<ParamInfo> params;
  long total = 0;
  // caller-owned flat buffers
  float *p = nullptr, *g = nullptr, *mu = nullptr, *nu = nullptr;
  bf16_t* pb = nullptr;   // bf16 copies of the parameters (owned here)
  // offsets
  long o_emb, o_fnorm, o_logits;
  // Rows of the vocabulary (bf16 copy of the logits kernel, the last parameter; logits and their gradients) lie Vp apart: an odd number of 128-byte lines, V or V + 64
  // columns.  With 127 or 129 times 2^12 bytes the 256 rows a tile fetches side by side lie in few memory channels: the product whose reduction runs along them
  // took 3.30 ms a chunk of 2048 rows of 264192 columns (0.67 PFLOP/s), one line further apart 1.72 (1.29; only one of the two operands: 2.9).  A whole step,
  // one layer of 2048, 4096 tokens: 264192 columns 25.6 -> 22.5 ms, 260096 24.8 -> 23.6; where V is an odd number of lines already, 64 more make it worse
  // (131008, then rows of 2^18 bytes: 12.91 -> 13.11 ms; 262080 24.09 -> 24.32); every other of 40 vocabularies, 16384 to 280576, is the same within 1.5 %
  long Vp;
  struct LOff { long ln1, wq, wk, wv, wo, ln2, wi0, wi1, wout; };
  std::vector<LOff> lo;
  std::vector<LayerAct> act;
  bf16_t *h_final = nullptr, *xn_f = nullptr, *rope_sin = nullptr, *rope_cos = nullptr;
  float* r_f = nullptr;
  bool walk = false;        // attention by ixt_train_attn.h (walk_pays): heads of 64 or 128, rows of at most TA_MOST tokens, operands of a batch row and weights of a head within the reach of a 32-bit offset
  long Sp;                  // columns between rows of P and dS: S, or whole tiles of 64, an odd number of them (walk)
  int2* reach = nullptr;
  // workspaces
  float *scores = nullptr, *dh = nullptr, *dxn = nullptr, *logits = nullptr, *row_loss = nullptr, *scal = nullptr, *part = nullptr, *norm_part = nullptr;   // norm_part: [norms][blocks][E], rows of at most 1024 (rmsnorm_bwd)
  bf16_t *dS = nullptr, *d_ao = nullptr, *dq = nullptr, *dk = nullptr, *dv = nullptr, *dact = nullptr, *da = nullptr, *db = nullptr, *dlog = nullptr,
         *dy_bf = nullptr;
  float *dkf = nullptr, *dvf = nullptr;   // grouped-query attention: dK / dV summed over a group's query heads in f32 before they round to bf16
  size_t scores_n = 0;
  std::vector<void*> allocs;
};

template <typename T_>
static int tmalloc(ixt_trainer* t, T_** p, size_t n) {
  void* q = nullptr;
  TCHK(hipMalloc(&q, n * sizeof(T_) + 256));
  t->allocs.push_back(q);
  *p = (T_*)q;
  return IXT_OK;
}

// the norms' backward (k_t_rmsnorm_bwd)
static int norm_rows(long T) { return T < 512 ? 1 : T < 8192 ? (int)(T / 512) : 16; }   // rows of a block
static long norm_blocks(long T) { return (T + norm_rows(T) - 1) / norm_rows(T); }
static void add_param(ixt_trainer* t, const std::string& name, long numel, long* off) {
  *off = t->total;
  t->params.push_back({name, t->total, numel});
  t->total += (numel + 63) / 64 * 64;   // 256-byte aligned segments
}

// Walks over the keys (ixt_train_attn.h) where they are the faster way.  A row of tokens is walked by one block of 64 rows after the other's start, 64 keys behind 64, three times: with few blocks the
// chip waits for the longest walk, while the products through memory have tiles of all keys at once; the more query heads a kv head has, the more launches these take.  us a layer (width 256, forward
// and backward, all tokens of one segment), walks / through memory, one row: 16 heads of 128, 512 tokens 205 / 195, 1024 297 / 288, 1536 406 / 414, 2048 499 / 579; 12 heads of 64, 512 tokens 159 / 160,
// 1024 224 / 216, 1536 296 / 302; 4 heads of 128, 128 tokens 122 / 124, 4096 719 / 608; 2 heads of 64, 256 tokens 120 / 122, 4096 528 / 409.  In groups of two, 4 heads of 64, 576 tokens 173 / 186, 2048
// 343 / 320; 8 heads of 128, 512 tokens 189 / 195, 2048 454 / 435; in groups of four, 8 heads of 128, 1024 tokens 321 / 331.  Of 398 such shapes (1 to 128 heads, 64 to 4096 tokens, groups of 1 to 32) the
// rule takes the slower way by more than 1 % for 11, by 13 % at most (4 heads of 128 in one group, 576 tokens); walks alone would for 106, by up to twice the time.
static bool walk_pays(long heads, int G, int D, int S) {
  const bool narrow = D == 64;
  if (S <= (narrow ? 256 : 128)) return true;
  const long blocks = heads * ((S + 63) / 64);
  if (G > 1) return S <= 512 || heads * G >= (narrow ? 16 : 32) || blocks >= 512;
  return blocks >= (S <= 512 ? (narrow ? 64 : 192) : (narrow ? 288 : 320));
}
extern "C" int ixt_train_create(const ixt_train_config* c, ixt_trainer** out) { return ixt_train_create_attention(c, IXT_TRAIN_ATTENTION_AUTO, out); }
extern "C" int ixt_train_create_attention(const ixt_train_config* c, int attention, ixt_trainer** out) {
  if (attention < IXT_TRAIN_ATTENTION_AUTO || attention > IXT_TRAIN_ATTENTION_MEMORY) return t_set_err(IXT_ERR_INVALID, "train step: attention %d", attention);
  if (!c || !out) return t_set_err(IXT_ERR_INVALID, "null argument");
  if (c->num_kv_heads <= 0 || c->num_query_heads % c->num_kv_heads) return t_set_err(IXT_ERR_INVALID, "train step: num_query_heads %% num_kv_heads != 0");
  if (c->head_dim % 8 || c->emb_dim % 8 || c->mlp_dim % 8 || c->vocab_size % 8 || c->seq_len % 8)
    return t_set_err(IXT_ERR_UNSUPPORTED, "train step: every dimension must be a multiple of 8");
  if (c->emb_dim > 256 * TN_FPT) return t_set_err(IXT_ERR_UNSUPPORTED, "train step: emb_dim %d above %d (k_t_rmsnorm_bwd keeps a row block's scale gradients in registers)", c->emb_dim, 256 * TN_FPT);
  if (c->batch <= 0 || c->seq_len <= 0 || c->num_decoder_layers <= 0) return t_set_err(IXT_ERR_INVALID, "bad sizes");
  ixt_trainer* t = new ixt_trainer();
  t->cfg = *c;
  t->E = c->emb_dim; t->H = c->num_query_heads; t->D = c->head_dim; t->F = c->mlp_dim; t->V = c->vocab_size; t->L = c->num_decoder_layers;
  t->B = c->batch; t->S = c->seq_len; t->T = t->B * t->S; t->QN = t->H * t->D;
  t->KVH = c->num_kv_heads; t->G = t->H / t->KVH; t->KN = t->KVH * t->D;
  t->Tc = c->logits_chunk > 0 ? c->logits_chunk : 2048;
  if (t->Tc > t->T) t->Tc = t->T;
  t->Vp = t->V >= 4096 && (t->V + 32) / 64 % 2 == 0 ? t->V + 64 : t->V;
  const long E = t->E, F = t->F, V = t->V, QN = t->QN, KN = t->KN;
  add_param(t, "params/token_embedder/embedding", V * E, &t->o_emb);
  t->lo.resize(t->L);
  for (int i = 0; i < t->L; ++i) {
    const std::string p = "params/decoder/layers_" + std::to_string(i) + "/";
    add_param(t, p + "pre_self_attention_layer_norm/scale", E, &t->lo[i].ln1);
    add_param(t, p + "self_attention/query/kernel", E * QN, &t->lo[i].wq);
    add_param(t, p + "self_attention/key/kernel", E * KN, &t->lo[i].wk);
    add_param(t, p + "self_attention/value/kernel", E * KN, &t->lo[i].wv);
    add_param(t, p + "self_attention/out/kernel", QN * E, &t->lo[i].wo);
    add_param(t, p + "mlp/mlp_layer_norm/scale", E, &t->lo[i].ln2);
    add_param(t, p + "mlp/wi_0/kernel", E * F, &t->lo[i].wi0);
    add_param(t, p + "mlp/wi_1/kernel", E * F, &t->lo[i].wi1);
    add_param(t, p + "mlp/wo/kernel", F * E, &t->lo[i].wout);
  }
  add_param(t, "params/decoder/decoder_norm/scale", E, &t->o_fnorm);
  add_param(t, "params/decoder/logits_dense/kernel", E * V, &t->o_logits);
  *out = nullptr;
  int rc = IXT_OK;
  auto fail = [&](int code) { ixt_train_destroy(t); return code; };
#define A(expr) do { rc = (expr); if (rc != IXT_OK) return fail(rc); } while (0)
  const size_t T = t->T, S = t->S, BH = (size_t)t->B * t->H;
  t->Sp = ((long)S + 63) / 64 * 64;
  t->Sp += t->Sp / 64 % 2 == 0 ? 64 : 0;
  t->walk = (t->D == 64 || t->D == 128) && S <= TA_MOST && S * (size_t)(QN > t->Sp ? QN : t->Sp) * 2 < (size_t)1 << 32;
  if (attention == IXT_TRAIN_ATTENTION_WALK && !t->walk) return fail(t_set_err(IXT_ERR_UNSUPPORTED, "train step: no walks over the keys with heads of %d, %d tokens a row", t->D, t->S));
  if (attention == IXT_TRAIN_ATTENTION_MEMORY || (attention == IXT_TRAIN_ATTENTION_AUTO && !walk_pays((long)t->B * t->H, t->G, t->D, t->S))) t->walk = false;
  if (!t->walk) t->Sp = S;
  A(tmalloc(t, &t->pb, (size_t)t->total + (size_t)E * (t->Vp - V)));
  t->act.resize(t->L);
  for (int i = 0; i < t->L; ++i) {
    LayerAct& a = t->act[i];
    A(tmalloc(t, &a.h_in, T * E)); A(tmalloc(t, &a.xn1, T * E)); A(tmalloc(t, &a.q, T * QN)); A(tmalloc(t, &a.k, T * KN)); A(tmalloc(t, &a.v, T * KN));
    A(tmalloc(t, &a.P, BH * S * t->Sp)); A(tmalloc(t, &a.ao, T * QN)); A(tmalloc(t, &a.h_mid, T * E)); A(tmalloc(t, &a.xn2, T * E));
    A(tmalloc(t, &a.a, T * F)); A(tmalloc(t, &a.b, T * F)); A(tmalloc(t, &a.act, T * F)); A(tmalloc(t, &a.r1, T)); A(tmalloc(t, &a.r2, T));
  }
  A(tmalloc(t, &t->h_final, T * E)); A(tmalloc(t, &t->xn_f, T * E)); A(tmalloc(t, &t->r_f, T));
  // (behind the logits the scores hold the parts of a cut product, too: whichever way attention goes, the cut stays a matter of the shape alone)
  t->scores_n = std::max(t->walk ? (size_t)0 : BH * S * S, V >= 65536 ? (size_t)4 * t->Tc * E : (size_t)0);
  if (t->scores_n > 0) A(tmalloc(t, &t->scores, t->scores_n));
  A(tmalloc(t, &t->dh, T * E)); A(tmalloc(t, &t->dxn, T * E));
  // (a chunk's logits are bf16, at the front of a buffer of f32 words that holds the parts of cut weight gradients later on)
  A(tmalloc(t, &t->logits, (size_t)t->Tc * V)); A(tmalloc(t, &t->dlog, (size_t)t->Tc * t->Vp)); A(tmalloc(t, &t->row_loss, T)); A(tmalloc(t, &t->scal, (size_t)16));
  A(tmalloc(t, &t->part, (size_t)4096));
  // The norms' scale gradients without atomics, for rows of at most 1024: at 2048 x 768 the atomics are 10 of a launch's 23 us, and the parts 39 MB for 25 norms.
  // 33 norms of 16384 x 2048 would take 277 MB for 13 of 145 us, 0.2 % of a step: wider rows keep the atomics, and with them last bits that vary from run to run.
  if (E <= 1024) A(tmalloc(t, &t->norm_part, (size_t)(2 * t->L + 1) * norm_blocks(t->T) * E));
  A(tmalloc(t, &t->dS, BH * S * t->Sp));
  if (t->walk) A(tmalloc(t, &t->reach, (size_t)t->B * 64));
  A(tmalloc(t, &t->d_ao, T * QN)); A(tmalloc(t, &t->dq, T * QN)); A(tmalloc(t, &t->dk, T * KN));
  A(tmalloc(t, &t->dv, T * KN));
  if (t->G > 1 && !t->walk) { A(tmalloc(t, &t->dkf, T * KN)); A(tmalloc(t, &t->dvf, T * KN)); } A(tmalloc(t, &t->dact, T * F)); A(tmalloc(t, &t->da, T * F)); A(tmalloc(t, &t->db, T * F)); A(tmalloc(t, &t->dy_bf, T * E));
#undef A
  // RoPE tables: the same host recipe as the decode path (embeddings.py:270-307)
  {
    const int half = t->D / 2;
    std::vector<uint16_t> sn((size_t)S * half), cs((size_t)S * half);
    auto f2bf_h = [](float f) { uint32_t u; memcpy(&u, &f, 4); u += 0x7fffu + ((u >> 16) & 1u); return (uint16_t)(u >> 16); };
    for (int i = 0; i < half; ++i) {
      const float frac = (float)(2 * i) / (float)t->D;
      const float ts = (float)((double)c->rope_min_timescale * pow((double)c->rope_max_timescale / (double)c->rope_min_timescale, (double)frac));
      for (size_t p = 0; p < S; ++p) {
        const float ang = (float)p / ts;
        sn[p * half + i] = f2bf_h((float)sin((double)ang));
        cs[p * half + i] = f2bf_h((float)cos((double)ang));
      }
    }
    if (tmalloc(t, &t->rope_sin, sn.size()) != IXT_OK || tmalloc(t, &t->rope_cos, cs.size()) != IXT_OK ||
        hipMemcpy(t->rope_sin, sn.data(), sn.size() * 2, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(t->rope_cos, cs.data(), cs.size() * 2, hipMemcpyHostToDevice) != hipSuccess)
      return fail(t_set_err(IXT_ERR_HIP, "rope table upload failed"));
  }
  *out = t;
  return IXT_OK;
}

extern "C" int ixt_train_destroy(ixt_trainer* t) {
  if (!t) return IXT_OK;
  (void)hipDeviceSynchronize();
  for (void* p : t->allocs) (void)hipFree(p);
  delete t;
  return IXT_OK;
}

extern "C" int64_t ixt_train_total_numel(ixt_trainer* t) { return t ? t->total : 0; }
extern "C" int ixt_train_param_count(ixt_trainer* t) { return t ? (int)t->params.size() : 0; }
extern "C" int ixt_train_param_info(ixt_trainer* t, int index, char* name_out, int name_cap, int64_t* offset, int64_t* numel) {
  if (!t || index < 0 || index >= (int)t->params.size() || !name_out || !offset || !numel) return t_set_err(IXT_ERR_INVALID, "bad argument");
  snprintf(name_out, name_cap, "%s", t->params[index].name.c_str());
  *offset = t->params[index].offset;
  *numel = t->params[index].numel;
  return IXT_OK;
}
extern "C" int ixt_train_bind(ixt_trainer* t, float* params, float* grads, float* adam_mu, float* adam_nu) {
  if (!t || !params || !grads || !adam_mu || !adam_nu) return t_set_err(IXT_ERR_INVALID, "null argument");
  t->p = params; t->g = grads; t->mu = adam_mu; t->nu = adam_nu;
  return IXT_OK;
}
extern "C" int ixt_train_refresh_bf16(ixt_trainer* t, void* stream) {
  if (!t || !t->p) return t_set_err(IXT_ERR_INVALID, "bind the parameter buffers first");
  hipLaunchKernelGGL(k_t_cast_bf16, dim3((unsigned)((t->o_logits / 4 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, t->p, t->pb, t->o_logits, 0L);
  hipLaunchKernelGGL(k_t_cast_bf16, dim3((unsigned)((t->V / 4 + 255) / 256), t->E), dim3(256), 0, (hipStream_t)stream, t->p + t->o_logits, t->pb + t->o_logits, (long)t->V, t->Vp);
  TLAUNCH();
  return IXT_OK;
}

// ---------------------------------------------------------------------------------------------------------------- launches
// The three products of a linear layer y = x W, W [K][N]: x W (W's columns contiguous), dy W^T (its k contiguous), x^T dy (both by columns).
enum { TL_XW, TL_DX, TL_DW };
template <bool TA, bool TB, int BM, int BN = BM, bool FOLD = false>
static int gemm_launch(hipStream_t st, TGemm& g) {
  // waves and their tiles: 256 x 256: 2 x 4 of 128 x 64; 256 x 128: 4 x 2 and 128 x 128: 2 x 2 of 64 x 64; 128 x 64: 4 of 32 x 64; 64 x 64: 2 x 2 of 32 x 32
  constexpr int WM = BN == BM ? 2 : 4, WN = BN == 256 ? 4 : BN == 64 && BM == 128 ? 1 : 2, MI = BM / 16 / WM, NI = BN / 16 / WN, NS = 4, lds = (TA && TB ? NS : NS + 1) * (BM + BN) * 64;
  const auto kernel = k_tgemm<TA, TB, MI, NI, WM, WN, NS, FOLD>;
  TCHK((lds_room<&k_tgemm<TA, TB, MI, NI, WM, WN, NS, FOLD>>(lds)));
  if (g.nb1 == 0) g.nb1 = g.nb2 = 1;
  g.mt = (g.M + BM - 1) / BM;
  for (int i = 0; i < 3; ++i) g.nt[i] = i < g.nprob ? (g.N[i] + BN - 1) / BN : 0;
  const int total = g.mt * (g.nt[0] + g.nt[1] + g.nt[2]) * g.parts * g.nb1 * g.nb2;
  hipLaunchKernelGGL(kernel, dim3(8 * ((total + 7) / 8)), dim3(64 * WM * WN), lds, st, g);
  TLAUNCH();
  return IXT_OK;
}
// One product per (batch row, kv head), element strides between them for each operand.  The score-sized ones (a head's S x S) take square tiles, those
// with head_dim columns tall ones; the smaller tile of each pair where the larger would leave CUs without a block (causal tiles count half).
static int attn_gemm(hipStream_t st, bool ta, bool tb, const bf16_t* A, long lda, const bf16_t* B, long ldb, void* C, long ldc, int M, int N, int K, int out, int causal, int nb1, int nb2,
                     long sa1, long sa2, long sb1, long sb2, long sc1, long sc2) {
  TGemm g{};
  g.A[0] = A; g.lda[0] = lda; g.B[0] = B; g.ldb[0] = ldb; g.C[0] = C; g.ldc[0] = ldc;
  g.M = M; g.N[0] = N; g.K[0] = K; g.nprob = g.parts = 1; g.out = out; g.causal = causal;
  g.nb1 = nb1; g.nb2 = nb2; g.sa1 = sa1; g.sa2 = sa2; g.sb1 = sb1; g.sb2 = sb2; g.sc1 = sc1; g.sc2 = sc2;
  auto blocks = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * nb1 * nb2 / (causal == TC_LOWER ? 2 : 1); };
  if (!tb) {
    if (blocks(256, 256) >= 512) return gemm_launch<false, false, 256>(st, g);
    if (blocks(128, 128) >= 200) return gemm_launch<false, false, 128>(st, g);
    return gemm_launch<false, false, 64>(st, g);
  }
  if (N > 64 && blocks(256, 128) >= 512) return ta ? gemm_launch<true, true, 256, 128>(st, g) : gemm_launch<false, true, 256, 128>(st, g);
  if (blocks(128, 64) >= 200) return ta ? gemm_launch<true, true, 128, 64>(st, g) : gemm_launch<false, true, 128, 64>(st, g);
  return ta ? gemm_launch<true, true, 64>(st, g) : gemm_launch<false, true, 64>(st, g);
}
// attention by walks (ixt_train_attn.h): forward, the queries' gradients, behind them the keys' and values'
enum { TA_FWD, TA_DQ, TA_DKV };
template <int D, int N>
static int attn_back_t(hipStream_t st, const TAttn& a, int what) {
  const int heads = a.B * (what == TA_DKV ? a.KVH : a.H);
  const dim3 grid((unsigned)((heads + 7) / 8 * 8 * ((a.S + 64 * N - 1) / (64 * N))));
  TCHK((lds_room<&k_t_attn_dq<D, N>>(TA_LDS_IMAGES(D, 4))));
  TCHK((lds_room<&k_t_attn_dkv<D, N>>(TA_LDS_DKV(D, N))));
  if (what == TA_DQ) hipLaunchKernelGGL((k_t_attn_dq<D, N>), grid, dim3(256), TA_LDS_IMAGES(D, 4), st, a);
  else hipLaunchKernelGGL((k_t_attn_dkv<D, N>), grid, dim3(256), TA_LDS_DKV(D, N), st, a);
  TLAUNCH();
  return IXT_OK;
}
// Rows of at most 512 tokens: a wave holds its scores (48 heads of 64 x 512: 18.8 us, by three walks 32, before either looked for weights to divide; 21 us in a whole step now).
template <int D>
static int attn_forward_t(hipStream_t st, const TAttn& a) {
  const dim3 grid((unsigned)((a.B * a.H + 7) / 8 * 8 * ((a.S + 63) / 64)));
  TCHK((lds_room<&k_t_attn_fwd<D, true>>(TA_LDS(D, 4))));
  if (a.S <= 64 * TA_HELD) hipLaunchKernelGGL((k_t_attn_fwd<D, true>), grid, dim3(256), TA_LDS(D, 4), st, a);
  else hipLaunchKernelGGL((k_t_attn_fwd<D, false>), grid, dim3(256), TA_LDS(D, 3), st, a);
  TLAUNCH();
  return IXT_OK;
}
// Back: 32 rows a wave where that leaves two blocks a CU, 16 below (us queries' and keys' gradients, 32 / 16 rows: 192 blocks of 128 rows, heads of 64 24.2 14.2 / 19.2 11.9; 2048 blocks, heads of 128
// 392 251 / 482 298; heads of 64, 1536 blocks 251 159 / 272 157)
static int attn_walk(hipStream_t st, const TAttn& a, int D, int what) {
  if (what == TA_FWD) return D == 64 ? attn_forward_t<64>(st, a) : attn_forward_t<128>(st, a);
  const bool wide = (long)a.B * (what == TA_DKV ? a.KVH : a.H) * ((a.S + 127) / 128) >= 512;
  if (D == 64) return wide ? attn_back_t<64, 2>(st, a, what) : attn_back_t<64, 1>(st, a, what);
  return wide ? attn_back_t<128, 2>(st, a, what) : attn_back_t<128, 1>(st, a, what);
}
static void softmax_fwd(hipStream_t st, const float* scores, const int32_t* seg, bf16_t* P, int S, int B, int H) {
  const dim3 grid(S, B * H), waves((S + 3) / 4, B * H);
  if (S <= 512) hipLaunchKernelGGL(k_t_softmax_fwd_wave<2>, waves, dim3(256), 0, st, scores, seg, P, S, H);
  else if (S <= 2048) hipLaunchKernelGGL(k_t_softmax_fwd_wave<8>, waves, dim3(256), 0, st, scores, seg, P, S, H);
  else if (S <= 4096) hipLaunchKernelGGL(k_t_softmax_fwd_reg<16>, grid, dim3(256), 0, st, scores, seg, P, S, H);
  else hipLaunchKernelGGL(k_t_softmax_fwd, grid, dim3(256), 0, st, scores, seg, P, S, H);
}
static void softmax_bwd(hipStream_t st, const float* dP, const bf16_t* P, bf16_t* dS, int S, int BH) {
  const dim3 grid(S, BH), waves((S + 3) / 4, BH);
  if (S <= 512) hipLaunchKernelGGL(k_t_softmax_bwd_wave<2>, waves, dim3(256), 0, st, dP, P, dS, S);
  else if (S <= 2048) hipLaunchKernelGGL(k_t_softmax_bwd_reg<8>, grid, dim3(256), 0, st, dP, P, dS, S);
  else if (S <= 4096) hipLaunchKernelGGL(k_t_softmax_bwd_reg<16>, grid, dim3(256), 0, st, dP, P, dS, S);
  else hipLaunchKernelGGL(k_t_softmax_bwd, grid, dim3(256), 0, st, dP, P, dS, S);
}
// Rows of 16384 columns and more by sixteen waves (32000 columns 82 -> 76 us for 2048 rows); where two such blocks a CU would have more in work than the memory-side cache holds beside what
// is written, the LDS keeps it to one (264192 columns: 804 us by two, 737 by one, 971 by blocks of four waves).
static int xent(hipStream_t st, const bf16_t* logits, const int32_t* targets, const int32_t* seg, bf16_t* dlog, float* row_loss, int n, int V, long ld) {
  if (V < 16384) {
    hipLaunchKernelGGL(k_t_xent, dim3(n), dim3(256), 0, st, logits, targets, seg, dlog, row_loss, V, ld);
  } else {
    constexpr int two = 2 * 8192 * sizeof(float), one = 96 * 1024;
    TCHK(lds_room<&k_t_xent_wide>(one));
    hipLaunchKernelGGL(k_t_xent_wide, dim3(n), dim3(1024), (size_t)V * sizeof(bf16_t) * 512 > (size_t)192 << 20 ? one : two, st, logits, targets, seg, dlog, row_loss, V, ld);
  }
  TLAUNCH();
  return IXT_OK;
}
// TL_DX: n is the reduction (the layer's outputs), c of the first entry the result; ldw: where the rows of w (TL_XW: and of c) lie further apart than n
struct TOperand { const bf16_t* x; const bf16_t* w; void* c; int n; long ldw = 0; };
// TL_DX of several entries: the sum of their products.
// M: rows (tokens; TL_DW: the layer's inputs); K: reduction (TL_DX: the entries' n); scratch: for reductions cut in parts, or nullptr
static int gemm(hipStream_t st, int what, int M, int K, std::initializer_list<TOperand> ops, int out, long ld_x, int N_dx = 0, const bf16_t* res = nullptr, float* scratch = nullptr,
                size_t scratch_floats = 0) {
  TGemm g{};
  g.M = M; g.R = res; g.out = out; g.parts = 1;
  const int sums = what == TL_DX ? (int)ops.size() : 1;
  int i = 0;
  for (const TOperand& o : ops) {
    g.A[i] = o.x; g.B[i] = o.w; g.C[i] = o.c;
    const long ldw = o.ldw ? o.ldw : o.n;
    if (what == TL_XW) { g.lda[i] = ld_x; g.ldb[i] = g.ldc[i] = ldw; g.N[i] = o.n; g.K[i] = K; }
    else if (what == TL_DX) { g.lda[i] = ld_x; g.ldb[i] = ldw; g.ldc[i] = N_dx; g.N[i] = N_dx; g.K[i] = o.n; }
    else { g.lda[i] = ld_x; g.ldb[i] = ldw; g.ldc[i] = o.n; g.N[i] = o.n; g.K[i] = K; }
    ++i;
  }
  g.nprob = sums > 1 ? 1 : i;
  auto tiles = [&](int b) {
    long t = 0;
    for (int k = 0; k < g.nprob; ++k) t += (g.N[k] + b - 1) / b;
    return t * ((M + b - 1) / b);
  };
  // A weight gradient of few output tiles over a long reduction (2048 x 2048 over 16384 tokens: 64 tiles of 256 x 256) is cut in four parts, whose
  // products are added up in order (k_t_sum_parts); a reduction that is no multiple of 256 is not cut.  The cut is a matter of the shape alone, so that no
  // choice of tiles changes a sum.
  if (out == TG_F32 && scratch != nullptr && g.K[0] >= 2048 && g.K[0] % 256 == 0) {
    bool all = true;
    long need = 0;
    for (int k = 0; k < g.nprob; ++k) {
      all = all && (long)((g.N[k] + 127) / 128) * ((M + 127) / 128) <= 256;
      need += 4L * M * g.N[k];
    }
    if (all && (size_t)need <= scratch_floats) {
      g.parts = 4;
      g.kpart = g.K[0] / 4;
      float* at = scratch;
      for (int k = 0; k < g.nprob; ++k) { g.C[k] = at; g.cpart[k] = (long)M * g.N[k]; at += 4 * g.cpart[k]; }
    }
  }
  // Sums, and cuts, inside the block (FOLD) where whole reductions give the chip enough tiles and the largest tile is not the one to take: 2048 x 768 outputs,
  // three products with K 768 33 -> 29 us, two with K 2048 49 -> 47; the weight gradients of 768 x 2304 over 2048 tokens 33 -> 22.  Fewer tiles than CUs
  // keep the parts (768 x 768: 14 us against 19).
  bool fold = what != TL_XW && tiles(256) * g.parts < 192 && (sums > 1 || g.parts > 1) && (g.parts == 1 || tiles(64) >= 256);
  for (const TOperand& o : ops) fold = fold && (sums == 1 || (o.n == g.K[0] && o.ldw == 0));
  if (fold) {
    g.nsum = sums;
    if (g.parts > 1) {
      g.fold = g.kpart / 32;
      g.parts = 1;
      int k = 0;
      for (const TOperand& o : ops) g.C[k++] = o.c;
    }
    if (what == TL_DX) return tiles(128) >= 200 ? gemm_launch<false, false, 128, 128, true>(st, g) : gemm_launch<false, false, 64, 64, true>(st, g);
    return gemm_launch<true, true, 64, 64, true>(st, g);   // (cut in four: fewer than 48 tiles of 256 x 256, 192 of 128 x 128 at most)
  }
  if (sums > 1) {
    int k = 0;
    for (const TOperand& o : ops) {
      const TOperand one{o.x, o.w, ops.begin()->c, o.n, o.ldw};
      TTRY(gemm(st, what, M, o.n, {one}, k++ == 0 ? out : TG_F32_ADD, o.n, N_dx, res, scratch, scratch_floats));
    }
    return IXT_OK;
  }
  // 256 x 256 tiles wherever they occupy three quarters of the CUs; 128 x 128 down to 200 of those, 64 x 64 below.  Measured in us, 128 / 64:
  // 96 tiles of 128 x 128 with K 768 15.1 / 9.9, K 2048 29.2 / 18.9; 192 tiles, K 2048 32.2 / 24.6; 256 tiles, K 768 14.8 / 17.7; 512 tiles 22.6 / 28.9.
  const int bm = tiles(256) * g.parts >= 192 ? 256 : tiles(128) * g.parts >= 200 ? 128 : 64;
#define GO(TA_, TB_) TTRY(bm == 256 ? (gemm_launch<TA_, TB_, 256>(st, g)) : bm == 128 ? (gemm_launch<TA_, TB_, 128>(st, g)) : (gemm_launch<TA_, TB_, 64>(st, g)))
  if (what == TL_XW) GO(false, true);
  else if (what == TL_DX) GO(false, false);
  else GO(true, true);
#undef GO
  if (g.parts > 1) {
    int k = 0;
    for (const TOperand& o : ops) {
      hipLaunchKernelGGL(k_t_sum_parts, dim3((unsigned)((g.cpart[k] / 4 + 255) / 256)), dim3(256), 0, st, reinterpret_cast<const float*>(g.C[k]), g.parts, g.cpart[k], reinterpret_cast<float*>(o.c));
      TLAUNCH();
      ++k;
    }
  }
  return IXT_OK;
}
// 16 rows per block (16384 x 2048: 182 -> 141 us with the next row in flight and the bf16 copy included), fewer below 8192 rows: a block's rows
// are a chain, but every block adds its sums to the same E words
static void rmsnorm_bwd(hipStream_t st, const float* dy, const bf16_t* x, const bf16_t* scale, const float* rstd, float* dh, bf16_t* dh_bf, float* dscale, float* part, int E, long T) {
  const int rpb = norm_rows(T);
  const dim3 grid((unsigned)norm_blocks(T));
  if (E <= 1024) hipLaunchKernelGGL(k_t_rmsnorm_bwd<4>, grid, dim3(256), 0, st, dy, x, scale, rstd, dh, dh_bf, dscale, part, E, T, rpb);
  else if (E <= 2048) hipLaunchKernelGGL(k_t_rmsnorm_bwd<8>, grid, dim3(256), 0, st, dy, x, scale, rstd, dh, dh_bf, dscale, part, E, T, rpb);
  else hipLaunchKernelGGL(k_t_rmsnorm_bwd<TN_FPT>, grid, dim3(256), 0, st, dy, x, scale, rstd, dh, dh_bf, dscale, part, E, T, rpb);
}
#define EW(n) dim3((unsigned)(((long)(n) + 255) / 256)), dim3(256), 0, st

extern "C" int ixt_train_forward_backward(ixt_trainer* t, const int32_t* inputs, const int32_t* positions, const int32_t* segmentation,
                                          const int32_t* targets, const int32_t* targets_segmentation, float* loss_and_weights_dev, void* stream) {
  if (!t || !inputs || !positions || !segmentation || !targets || !targets_segmentation || !loss_and_weights_dev)
    return t_set_err(IXT_ERR_INVALID, "null argument");
  if (!t->p) return t_set_err(IXT_ERR_INVALID, "bind the parameter buffers first");
  hipStream_t st = (hipStream_t)stream;
  const int E = t->E, H = t->H, D = t->D, F = t->F, V = t->V, S = t->S, T = t->T, QN = t->QN, B = t->B, KVH = t->KVH, G = t->G, KN = t->KN;
  const long HD = (long)H * D;
  const bf16_t* pb = t->pb;
  const float eps = t->cfg.normalization_layer_epsilon;
  // The gradients that several blocks add to start from zero: the embedding's and the norms' (the last one behind the loop's); every other one is stored
  // whole.  The gaps between parameters, where there are any, are part of the norm: cleared with everything else.
  bool gaps = false;
  for (const ParamInfo& p : t->params) gaps = gaps || p.numel % 64 != 0;
  const long stride = t->L > 1 ? t->lo[1].ln1 - t->lo[0].ln1 : 0;
  const long n0 = gaps ? t->total : (long)V * E;
  float* const g0 = gaps ? t->g : t->g + t->o_emb;
  hipLaunchKernelGGL(k_t_zero, dim3((unsigned)((n0 + 1023) / 1024 + ((long)2 * t->L * E + 1023) / 1024)), dim3(256), 0, st, g0, n0, t->g + t->lo[0].ln1, t->g + t->lo[0].ln2, stride, t->L, E);
  hipLaunchKernelGGL(k_t_zero, dim3((unsigned)((E + 1023) / 1024)), dim3(256), 0, st, t->g + t->o_fnorm, (long)E, t->g, t->g, 0L, 0, 4);
  TLAUNCH();
  // ------------------------------------------------------------------ forward (layers/* in train mode)
  bf16_t* h = t->act[0].h_in;
  hipLaunchKernelGGL(k_embed, dim3((E / 8 + 255) / 256, T), dim3(256), 0, st, pb + t->o_emb, inputs, h, E, V);
  TLAUNCH();
  for (int l = 0; l < t->L; ++l) {
    LayerAct& a = t->act[l];
    const ixt_trainer::LOff& o = t->lo[l];
    hipLaunchKernelGGL(k_t_rmsnorm_fwd, dim3(T), dim3(256), 0, st, a.h_in, pb + o.ln1, a.xn1, a.r1, E, eps);
    TTRY(gemm(st, TL_XW, T, E, {{a.xn1, pb + o.wq, a.q, QN}, {a.xn1, pb + o.wk, a.k, KN}, {a.xn1, pb + o.wv, a.v, KN}}, TG_BF16, E));
    const auto rope = t->walk ? k_t_rope<false, true> : k_t_rope<false, false>;
    hipLaunchKernelGGL(rope, EW((long)T * (H + KVH) * (D / 8)), a.q, a.k, positions, t->rope_sin, t->rope_cos, H, KVH, D, (long)T);
    // scores[b,h] = Q_h K_(h / G)^T (sm_scale 1: the query kernel carries 1/sqrt(d), attentions.py:1900-1904).  Grouped-query attention
    // (attentions.py:1206-1271: query heads reshaped to [kv heads, G]): query head kvh G + g of every kv head in launch g, batches (b, kvh).
    const TAttn ta{a.q, a.k, a.v, segmentation, a.P, a.ao, t->reach, t->d_ao, t->dS, t->dq, t->dk, t->dv, B, S, H, KVH, t->Sp};
    if (t->walk) {
      TTRY(attn_walk(st, ta, D, TA_FWD));
    } else {
      const long SS = (long)S * S;
      for (int g = 0; g < G; ++g)
        TTRY(attn_gemm(st, false, false, a.q + (long)g * D, HD, a.k, KN, t->scores + g * SS, S, S, S, D, TG_F32, TC_LOWER, B, KVH, (long)S * HD, (long)G * D, (long)S * KN, D, H * SS, G * SS));
      softmax_fwd(st, t->scores, segmentation, a.P, S, B, H);
      for (int g = 0; g < G; ++g)
        TTRY(attn_gemm(st, false, true, a.P + g * SS, S, a.v, KN, a.ao + (long)g * D, HD, S, D, S, TG_BF16, TC_K_TO_ROW, B, KVH, H * SS, G * SS, (long)S * KN, D, (long)S * HD, (long)G * D));
    }
    TTRY(gemm(st, TL_XW, T, QN, {{a.ao, pb + o.wo, a.h_mid, E}}, TG_BF16_RES, QN, 0, a.h_in));
    hipLaunchKernelGGL(k_t_rmsnorm_fwd, dim3(T), dim3(256), 0, st, a.h_mid, pb + o.ln2, a.xn2, a.r2, E, eps);
    TTRY(gemm(st, TL_XW, T, E, {{a.xn2, pb + o.wi0, a.a, F}, {a.xn2, pb + o.wi1, a.b, F}}, TG_BF16, E));
    hipLaunchKernelGGL(k_t_swiglu_fwd, EW((long)T * F / 8), a.a, a.b, a.act, (long)T * F);
    bf16_t* h_next = l + 1 < t->L ? t->act[l + 1].h_in : t->h_final;
    TTRY(gemm(st, TL_XW, T, F, {{a.act, pb + o.wout, h_next, E}}, TG_BF16_RES, F, 0, a.h_mid));
    TLAUNCH();
  }
  hipLaunchKernelGGL(k_t_rmsnorm_fwd, dim3(T), dim3(256), 0, st, t->h_final, pb + t->o_fnorm, t->xn_f, t->r_f, E, eps);
  // ------------------------------------------------------------------ logits, loss and their gradients, a chunk of rows at a time
  for (int t0 = 0; t0 < T; t0 += t->Tc) {
    const int n = T - t0 < t->Tc ? T - t0 : t->Tc;
    const bf16_t* xn = t->xn_f + (long)t0 * E;
    TTRY(gemm(st, TL_XW, n, E, {{xn, pb + t->o_logits, t->logits, V, t->Vp}}, TG_BF16, E));
    TTRY(xent(st, reinterpret_cast<const bf16_t*>(t->logits), targets + t0, targets_segmentation + t0, t->dlog, t->row_loss + t0, n, V, t->Vp));
    // d xn_f = dlogits . W^T ; dW += xn_f^T . dlogits
    TTRY(gemm(st, TL_DX, n, V, {{t->dlog, pb + t->o_logits, t->dxn + (long)t0 * E, V, t->Vp}}, TG_F32, t->Vp, E, nullptr, t->scores, V >= 65536 ? t->scores_n : 0));   // (the score buffer is idle)
    TTRY(gemm(st, TL_DW, E, n, {{xn, t->dlog, t->g + t->o_logits, V, t->Vp}}, t0 == 0 ? TG_F32 : TG_F32_ADD, E));
  }
  hipLaunchKernelGGL(k_t_reduce, dim3(1), dim3(256), 0, st, t->row_loss, (long)T, 0, loss_and_weights_dev, 0);
  // total_weights = number of target positions with a non-zero segment id (train.py:309)
  hipLaunchKernelGGL(k_t_nonzero, EW(T), targets_segmentation, t->row_loss, (long)T);          // row_loss is free again after the reduction above
  hipLaunchKernelGGL(k_t_reduce, dim3(1), dim3(256), 0, st, t->row_loss, (long)T, 0, loss_and_weights_dev + 1, 0);
  TLAUNCH();
  // ------------------------------------------------------------------ backward
  float* const spare = t->logits;                          // idle from here on: scratch of the cut weight-gradient products
  const size_t spare_n = (size_t)t->Tc * V;
  hipLaunchKernelGGL(k_t_zero, dim3((unsigned)(((long)T * E + 1023) / 1024)), dim3(256), 0, st, t->dh, (long)T * E, t->g, t->g, 0L, 0, 4);
  const auto norm_part = [&](int q) { return t->norm_part != nullptr ? t->norm_part + (size_t)q * norm_blocks(T) * E : nullptr; };
  rmsnorm_bwd(st, t->dxn, t->h_final, pb + t->o_fnorm, t->r_f, t->dh, t->dy_bf, t->g + t->o_fnorm, norm_part(2 * t->L), E, T);
  for (int l = t->L - 1; l >= 0; --l) {
    LayerAct& a = t->act[l];
    const ixt_trainer::LOff& o = t->lo[l];
    // MLP: h_out = h_mid + wo(act)
    TTRY(gemm(st, TL_DX, T, E, {{t->dy_bf, pb + o.wout, t->dact, E}}, TG_BF16, E, F));                   // d act = dy . Wout^T
    TTRY(gemm(st, TL_DW, F, T, {{a.act, t->dy_bf, t->g + o.wout, E}}, TG_F32, F, 0, nullptr, spare, spare_n));   // d Wout = act^T . dy
    hipLaunchKernelGGL(k_t_swiglu_bwd, EW((long)T * F / 8), t->dact, a.a, a.b, t->da, t->db, (long)T * F);
    TTRY(gemm(st, TL_DX, T, F, {{t->da, pb + o.wi0, t->dxn, F}, {t->db, pb + o.wi1, t->dxn, F}}, TG_F32, F, E, nullptr, spare, spare_n));   // d xn2 = da . Wi0^T + db . Wi1^T
    TTRY(gemm(st, TL_DW, E, T, {{a.xn2, t->da, t->g + o.wi0, F}, {a.xn2, t->db, t->g + o.wi1, F}}, TG_F32, E, 0, nullptr, spare, spare_n));
    rmsnorm_bwd(st, t->dxn, a.h_mid, pb + o.ln2, a.r2, t->dh, t->dy_bf, t->g + o.ln2, norm_part(t->L + l), E, T);
    // attention: h_mid = h_in + out(ao)
    TTRY(gemm(st, TL_DX, T, E, {{t->dy_bf, pb + o.wo, t->d_ao, E}}, TG_BF16, E, QN));                    // d ao = dy . Wo^T
    TTRY(gemm(st, TL_DW, QN, T, {{a.ao, t->dy_bf, t->g + o.wo, E}}, TG_F32, QN, 0, nullptr, spare, spare_n));   // d Wo = ao^T . dy
    if (t->walk) {
      const TAttn ta{a.q, a.k, a.v, segmentation, a.P, a.ao, t->reach, t->d_ao, t->dS, t->dq, t->dk, t->dv, B, S, H, KVH, t->Sp};
      TTRY(attn_walk(st, ta, D, TA_DQ));
      TTRY(attn_walk(st, ta, D, TA_DKV));
    } else {
      // dP = d_ao V^T (f32) ; dV = P^T d_ao ; dS = P o (dP - rowsum(dP o P)) ; dQ = dS K ; dK = dS^T Q.  With G query heads per kv head, dV and dK
      // are the sums over the group: accumulated in f32 over the G launches, rounded to bf16 once.
      const long SS = (long)S * S;
      for (int g = 0; g < G; ++g)
        TTRY(attn_gemm(st, false, false, t->d_ao + (long)g * D, HD, a.v, KN, t->scores + g * SS, S, S, S, D, TG_F32, TC_LOWER, B, KVH, (long)S * HD, (long)G * D, (long)S * KN, D, H * SS, G * SS));
      if (G == 1) {
        TTRY(attn_gemm(st, true, true, a.P, S, t->d_ao, HD, t->dv, HD, S, D, S, TG_BF16, TC_K_FROM_ROW, B, H, H * SS, SS, (long)S * HD, D, (long)S * HD, D));
      } else {
        for (int g = 0; g < G; ++g)
          TTRY(attn_gemm(st, true, true, a.P + g * SS, S, t->d_ao + (long)g * D, HD, t->dvf, KN, S, D, S, g > 0 ? TG_F32_ADD : TG_F32, TC_K_FROM_ROW, B, KVH, H * SS, G * SS, (long)S * HD,
                         (long)G * D, (long)S * KN, D));
        hipLaunchKernelGGL(k_t_f32_to_bf16, EW((long)T * KN / 8), t->dvf, t->dv, (long)T * KN);
      }
      softmax_bwd(st, t->scores, a.P, t->dS, S, B * H);
      for (int g = 0; g < G; ++g)
        TTRY(attn_gemm(st, false, true, t->dS + g * SS, S, a.k, KN, t->dq + (long)g * D, HD, S, D, S, TG_BF16, TC_K_TO_ROW, B, KVH, H * SS, G * SS, (long)S * KN, D, (long)S * HD, (long)G * D));
      if (G == 1) {
        TTRY(attn_gemm(st, true, true, t->dS, S, a.q, HD, t->dk, HD, S, D, S, TG_BF16, TC_K_FROM_ROW, B, H, H * SS, SS, (long)S * HD, D, (long)S * HD, D));
      } else {
        for (int g = 0; g < G; ++g)
          TTRY(attn_gemm(st, true, true, t->dS + g * SS, S, a.q + (long)g * D, HD, t->dkf, KN, S, D, S, g > 0 ? TG_F32_ADD : TG_F32, TC_K_FROM_ROW, B, KVH, H * SS, G * SS, (long)S * HD,
                         (long)G * D, (long)S * KN, D));
        hipLaunchKernelGGL(k_t_f32_to_bf16, EW((long)T * KN / 8), t->dkf, t->dk, (long)T * KN);
      }
    }
    const auto rope = t->walk ? k_t_rope<true, true> : k_t_rope<true, false>;
    hipLaunchKernelGGL(rope, EW((long)T * (H + KVH) * (D / 8)), t->dq, t->dk, positions, t->rope_sin, t->rope_cos, H, KVH, D, (long)T);
    // d xn1 = dq Wq^T + dk Wk^T + dv Wv^T
    TTRY(gemm(st, TL_DX, T, QN, {{t->dq, pb + o.wq, t->dxn, QN}, {t->dk, pb + o.wk, t->dxn, KN}, {t->dv, pb + o.wv, t->dxn, KN}}, TG_F32, QN, E, nullptr, spare, spare_n));
    TTRY(gemm(st, TL_DW, E, T, {{a.xn1, t->dq, t->g + o.wq, QN}, {a.xn1, t->dk, t->g + o.wk, KN}, {a.xn1, t->dv, t->g + o.wv, KN}}, TG_F32, E, 0, nullptr, spare, spare_n));
    rmsnorm_bwd(st, t->dxn, a.h_in, pb + o.ln1, a.r1, t->dh, l > 0 ? t->dy_bf : nullptr, t->g + o.ln1, norm_part(l), E, T);
    TLAUNCH();
  }
  if (t->norm_part != nullptr)
    hipLaunchKernelGGL(k_t_scale_grads, dim3((E + 63) / 64, 2 * t->L + 1), dim3(1024), 0, st, t->norm_part, (int)norm_blocks(T), E, t->g, t->L, t->lo[0].ln1, t->lo[0].ln2,
                       t->L > 1 ? t->lo[1].ln1 - t->lo[0].ln1 : 0L, t->o_fnorm);
  hipLaunchKernelGGL(k_t_embed_bwd, dim3((E + 255) / 256, T), dim3(256), 0, st, t->dh, inputs, t->g + t->o_emb, E, V);
  TLAUNCH();
  return IXT_OK;
}

extern "C" int ixt_train_apply(ixt_trainer* t, float total_weights, float clip_threshold, float lr, float b1, float b2, float eps, float eps_root,
                               float weight_decay, int count, float* norms_out_dev, void* stream) {
  if (!t || !t->p || !norms_out_dev || count < 1) return t_set_err(IXT_ERR_INVALID, "bad argument");
  hipStream_t st = (hipStream_t)stream;
  const int nblk = 2048;
  hipLaunchKernelGGL(k_t_sumsq_partial, dim3(nblk), dim3(256), 0, st, t->g, t->total, t->part);
  hipLaunchKernelGGL(k_t_reduce, dim3(1), dim3(256), 0, st, t->part, (long)nblk, 0, t->scal, 0);
  hipLaunchKernelGGL(k_t_clip_scale, dim3(1), dim3(1), 0, st, t->scal, total_weights + 1e-8f, clip_threshold, t->scal + 1, norms_out_dev);   // EPS = 1e-8 (globals.py:20)
  AdamArgs a;
  a.lr = lr; a.b1 = b1; a.b2 = b2; a.eps = eps; a.eps_root = eps_root; a.wd = weight_decay;
  a.bc1 = 1.0f - powf(b1, (float)count);
  a.bc2 = 1.0f - powf(b2, (float)count);
  const long ol = t->o_logits;
  hipLaunchKernelGGL(k_t_adamw, EW(ol), t->p, t->g, t->mu, t->nu, t->pb, t->scal + 1, ol, 0L, a);
  hipLaunchKernelGGL(k_t_adamw, dim3((unsigned)((t->V + 255) / 256), t->E), dim3(256), 0, st, t->p + ol, t->g + ol, t->mu + ol, t->nu + ol, t->pb + ol, t->scal + 1, (long)t->V, t->Vp, a);
  TLAUNCH();
  return IXT_OK;
}
