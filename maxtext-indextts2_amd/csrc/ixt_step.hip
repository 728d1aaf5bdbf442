// ixt_step.hip -- the one-launch pass of few rows: which shapes take it, its buffers, its launch.
#include "ixt_internal.h"
#include "ixt_step.h"

#include <atomic>

// Which shapes: those whose rows, normed, and whose attention's pages fit the LDS of a CU and whose (tile, chain) pairs fit a block; other models of few rows take the
// launches of ixt_small.h.
#define STEP_LDS (150 * 1024)
struct StepPlan { bool ok; int rpl, nblk[STEP_PHASES], tpb[STEP_PHASES], attw, att_floats, early; size_t lds; };
static StepPlan step_plan(const ixt_ctx* c, int R) {
  StepPlan p{};
  const AttnGeom& g = c->geom;
  auto chains = [](int K) { return (K + IXT_CHAIN - 1) / IXT_CHAIN; };
  const int ce = chains(c->E), co = chains(c->QN), cd = chains(c->F);
  if (R < 1 || R > 16 || ce > 4 || co > 16 || cd > 16 || c->P != 32 || !(c->D == 64 || c->D == 128) || !(c->GQ == 1 || c->GQ == 2)) return p;
  while ((1 << p.rpl) < R) ++p.rpl;
  p.tpb[STEP_QKV] = STEP_NW / ce;
  p.tpb[STEP_O] = STEP_NW / co;
  p.tpb[STEP_UP] = STEP_NW / ce & ~1;
  p.tpb[STEP_DOWN] = STEP_NW / cd;
  auto blocks = [](int tiles, int tpb) { return (tiles + tpb - 1) / tpb; };
  p.nblk[STEP_QKV] = blocks(c->NQKV / 16, p.tpb[STEP_QKV]);
  p.nblk[STEP_O] = blocks(c->E / 16, p.tpb[STEP_O]);
  p.nblk[STEP_UP] = blocks(2 * c->F / 16, p.tpb[STEP_UP]);
  p.nblk[STEP_DOWN] = blocks(c->E / 16, p.tpb[STEP_DOWN]);
  const size_t norm = ((size_t)(c->E / 8) << p.rpl) * 16 + STEP_NW * 1024 + 64 * sizeof(float);
  const int mpgp = (g.mpg + 3) & ~3;
  p.att_floats = c->GQ * (c->D + ((g.Tmax + 63) & ~63) + mpgp + STEP_NW + mpgp * c->D) + mpgp;
  // Two (row, kv head) pairs a block beyond 128: the attention's blocks hold no weights, and the later their CUs are free the later those behind them start (16 heads of
  // 500 keys, us a step: 12 slots 1018 with one pair a block, 963 with two, 16 slots 1069 / 1005).  Up to there a CU's rate for two pairs' pages counts more (8 slots 817 / 918).
  p.attw = R * c->KV > 128 && sizeof(float) * 2 * p.att_floats <= STEP_LDS ? STEP_NW / 2 : STEP_NW;
  p.nblk[STEP_ATT] = blocks(R * c->KV, STEP_NW / p.attw);
  p.early = std::max(0, std::min(p.nblk[STEP_UP], 256 - p.nblk[STEP_ATT] - p.nblk[STEP_O])) & ~7;
  const size_t att = sizeof(float) * (size_t)p.att_floats * (STEP_NW / p.attw);
  auto plain = [&](int K) { const size_t np = (size_t)(K / 8) << p.rpl; return (np <= 8 * STEP_NW * 64 ? np * 16 : 0) + STEP_NW * 1024; };   // (step_dot)
  p.lds = std::max(std::max(norm, att), std::max(plain(c->QN), plain(c->F)));
  p.ok = p.lds <= STEP_LDS;
  return p;
}
template <int HD, int GQ>
static int launch_step_t(const StepArgs& a, int L, size_t lds, hipStream_t st) {
  static bool attr_done = false;
  if (!attr_done) {
    HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_step<HD, GQ>), hipFuncAttributeMaxDynamicSharedMemorySize, STEP_LDS));
    attr_done = true;
  }
  hipLaunchKernelGGL((k_step<HD, GQ>), dim3((unsigned)(L * a.per_layer)), dim3(STEP_NW * 64), lds, st, a);
  LAUNCHCHK();
  return IXT_OK;
}
// the buffers of k_step, once, at ixt_create (the launch may be captured)
int step_init(ixt_ctx* c) {
  if (c->moe || c->gemma || c->fp8 || c->L < 1 || !step_plan(c, 1).ok) return IXT_OK;
  TRY(dmalloc(c, &c->step_layers, (size_t)c->L));
  TRY(dmalloc(c, &c->step_ws, (size_t)c->L * 16 * (2 * c->QN + 2 * c->E + c->F)));
  TRY(dmalloc(c, &c->step_cnt, ((size_t)c->L * STEP_PHASES * STEP_NS + 1) * 32));
  std::vector<StepLayer> t((size_t)c->L);
  auto at = [&](const void* p) { return (int64_t)(reinterpret_cast<intptr_t>(p) - reinterpret_cast<intptr_t>(c->step_ws)); };
  for (int l = 0; l < c->L; ++l) {
    const LayerW& w = c->layers[l];
    t[l] = StepLayer{at(w.wqkv), at(w.wo), at(w.wi), at(w.wout), at(w.ln1), at(w.ln2), at(c->kpages_l[l]), at(c->vpages_l[l])};
  }
  static std::atomic<int32_t> contexts{0};
  c->step_token = contexts.fetch_add(1) % 0x7fffffff + 1;
  HIPCHK(hipMemcpy(c->step_layers, t.data(), sizeof(StepLayer) * t.size(), hipMemcpyHostToDevice));
  return IXT_OK;
}
bool step_fits(const ixt_ctx* c, int R) { return c->step_layers != nullptr && step_plan(c, R).ok; }
// every layer of R rows; *hidden = the rows behind the last one.  fresh: step_attn
int launch_step(ixt_ctx* c, int R, const int32_t* tokens, int fresh, const bf16_t** hidden, hipStream_t st) {
  const StepPlan p = step_plan(c, R);
  StepArgs a;
  a.layers = c->step_layers; a.ws = c->step_ws; a.lstride = (size_t)16 * (2 * c->QN + 2 * c->E + c->F);
  a.h0 = c->h_a; a.cnt = c->step_cnt; a.err = c->split_cnt + (size_t)16 * c->KV * 4;
  a.R = R; a.E = c->E; a.F = c->F; a.QN = c->QN; a.NQKV = c->NQKV; a.rpl = p.rpl; a.fresh = fresh;
  a.token = c->step_token; a.nl = c->L; a.per_layer = 0; a.attw = p.attw; a.att_floats = p.att_floats; a.early = p.early;
  for (int i = 0; i < STEP_PHASES; ++i) { a.nblk[i] = p.nblk[i]; a.tpb[i] = p.tpb[i]; a.per_layer += p.nblk[i]; }
  a.eps = c->cfg.normalization_layer_epsilon;
  a.row_slot = c->row_slot; a.row_pos = c->row_pos; a.row_active = c->row_active; a.page_map = c->ps.page_map;
  a.rope_sin = c->rope_sin; a.rope_cos = c->rope_cos; a.g = c->geom;
  hipLaunchKernelGGL(k_step_begin, dim3(R), dim3(256), 0, st, tokens, c->embedding, c->E, c->h_a, c->step_cnt, c->L * STEP_PHASES * STEP_NS + 1, a.token, a.err);
  LAUNCHCHK();
  *hidden = c->step_ws + (size_t)c->L * a.lstride - (size_t)16 * c->E;
#define ST(HD_, GQ_) if (c->D == HD_ && c->GQ == GQ_) return launch_step_t<HD_, GQ_>(a, c->L, p.lds, st);
  ST(128, 1) ST(128, 2) ST(64, 1) ST(64, 2)
#undef ST
  return set_err(IXT_ERR_UNSUPPORTED, "step geometry hd=%d gq=%d", c->D, c->GQ);
}
