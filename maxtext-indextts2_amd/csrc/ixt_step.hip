// ixt_step.hip -- the one-launch pass of few rows, and the launches between the attentions of some: which shapes take them, their buffers, their launches.
#include "ixt_internal.h"
#include "ixt_mid.h"
#include "ixt_step.h"

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
  HIPCHK((lds_room<&k_step<HD, GQ>>(STEP_LDS)));
  hipLaunchKernelGGL((k_step<HD, GQ>), dim3((unsigned)(L * a.per_layer)), dim3(STEP_NW * 64), lds, st, a);
  LAUNCHCHK();
  return IXT_OK;
}
// k_mid: up to 64 rows whose norm is four pieces of 512 features a lane's share at most; a projection's units (16 a block) as in ixt_mid.h
struct MidPlan { bool ok; int early, nblk[MID_PHASES], tpb[MID_PHASES]; size_t lds; };
static MidPlan mid_plan(const ixt_ctx* c, int R) {
  MidPlan p{};
  const int G = (R + 15) / 16;
  if (G < 1 || G > 4 || c->E > 2048 || c->QN > 16 * IXT_CHAIN || c->F > 16 * IXT_CHAIN) return p;
  int steps = 0;
  auto dot = [&](int phase, int K, int ntile, int even, int least = 96) {
    const int nc = (K + IXT_CHAIN - 1) / IXT_CHAIN;
    int tpb = nc > 8 ? 1 : std::min(8, 16 / nc & ~1);
    while (tpb > 2 && (ntile + tpb - 1) / tpb < least) tpb -= 2;      // (a small projection over more CUs)
    if (even && tpb < 2) return false;
    p.tpb[phase] = tpb;
    p.nblk[phase] = (ntile + tpb - 1) / tpb;
    if (tpb > 1 && K / 32 <= MID_BUF_STEPS) steps = std::max(steps, K / 32);
    return true;
  };
  p.ok = dot(MID_O, c->QN, c->E / 16, 0) && dot(MID_UP, c->E, 2 * c->F / 16, 1) && dot(MID_DOWN, c->F, c->E / 16, 0) && dot(MID_QKV, c->E, c->NQKV / 16, 0, 160);
  p.nblk[MID_DOWN] = (p.nblk[MID_DOWN] + 7 & ~7) * MID_SPLIT;
  p.early = std::max(0, std::min(p.nblk[MID_UP], 256 - p.nblk[MID_O] - (R + MID_NW - 1) / MID_NW)) & ~7;
  p.nblk[MID_N1] = p.nblk[MID_N2] = (R + MID_NW - 1) / MID_NW;
  p.lds = (size_t)std::max({2 * steps, 16 * G, c->E / 64 + 1}) * 1024;
  return p;
}
static bool step_model(const ixt_ctx* c) { return !c->moe && !c->gemma && !c->fp8 && c->L >= 1; }
// Four row groups only where the weights of a layer are worth the phases' ends.  ms a step, a launch a phase / k_mid, eight layers of so many MB each (heads of 64 or 128, 60 to 270 keys):
//            14             29             45             63             116
//   48 rows  0.400 / 0.382  0.436 / 0.409  0.480 / 0.451  0.516 / 0.472  0.600 / 0.532
//   49       0.406 / 0.411  0.437 / 0.442  0.485 / 0.486  0.520 / 0.500  0.614 / 0.571
//   64       0.412 / 0.416  0.441 / 0.445  0.492 / 0.496  0.534 / 0.515  0.641 / 0.593
bool mid_fits(const ixt_ctx* c, int R) {
  const size_t layer = ((size_t)c->E * (c->NQKV + 2 * c->F) + (size_t)(c->QN + c->F) * c->E) * sizeof(bf16_t);
  return c->mid_ws != nullptr && R >= 17 && R <= std::min(layer >= (size_t)48 << 20 ? 64 : 48, c->mid_rows) && mid_plan(c, R).ok;
}
static size_t mid_words(const ixt_ctx* c) { return (size_t)(c->L + 1) * MID_PHASES * STEP_NS; }      // lines of its counters
// the buffers of k_step and k_mid, once, at ixt_create (the launch may be captured)
int step_init(ixt_ctx* c) {
  const bool step = step_model(c) && step_plan(c, 1).ok, mid = step_model(c) && c->Rmax >= 17 && mid_plan(c, 17).ok;
  if (!step && !mid) return IXT_OK;
  const size_t step_elems = step ? (size_t)c->L * 16 * (2 * c->QN + 2 * c->E + c->F) : 0;
  TRY(dmalloc(c, &c->step_layers, (size_t)c->L));
  TRY(dmalloc(c, &c->step_ws, step_elems + (mid ? (size_t)64 * (5 * c->E + c->F) : 0)));
  if (mid) {
    c->mid_ws = c->step_ws + step_elems;
    TRY(dmalloc(c, &c->mid_cnt, mid_words(c) * 32));
  }
  c->step_ok = step;
  TRY(dmalloc(c, &c->step_cnt, (size_t)c->L * STEP_PHASES * STEP_NS * 32));
  std::vector<StepLayer> t((size_t)c->L);
  auto at = [&](const void* p) { return (int64_t)(reinterpret_cast<intptr_t>(p) - reinterpret_cast<intptr_t>(c->step_ws)); };
  for (int l = 0; l < c->L; ++l) {
    const LayerW& w = c->layers[l];
    t[l] = StepLayer{at(w.wqkv), at(w.wo), at(w.wi), at(w.wout), at(w.ln1), at(w.ln2), at(c->kpages_l[l]), at(c->vpages_l[l])};
  }
  HIPCHK(hipMemcpy(c->step_layers, t.data(), sizeof(StepLayer) * t.size(), hipMemcpyHostToDevice));
  return IXT_OK;
}
bool step_fits(const ixt_ctx* c, int R) { return c->step_ok && step_plan(c, R).ok; }
FrontRows step_front(const ixt_ctx* c) { return FrontRows{c->embedding, c->h_a, c->E, c->step_cnt, c->L * STEP_PHASES * STEP_NS}; }
FrontRows mid_front(const ixt_ctx* c) { return FrontRows{c->embedding, c->mid_ws, c->E, c->mid_cnt, (int)mid_words(c)}; }
// every layer of R rows (tokens nullptr: what step_front names is done); *hidden = the rows behind the last one.  fresh: step_attn
int launch_step(ixt_ctx* c, int R, const int32_t* tokens, int fresh, const bf16_t** hidden, hipStream_t st) {
  const StepPlan p = step_plan(c, R);
  c->forms |= IXT_FORM_STEP;
  StepArgs a;
  a.layers = c->step_layers; a.ws = c->step_ws; a.lstride = (size_t)16 * (2 * c->QN + 2 * c->E + c->F);
  a.h0 = c->h_a; a.cnt = c->step_cnt; a.wait = c->wait();
  a.R = R; a.E = c->E; a.F = c->F; a.QN = c->QN; a.NQKV = c->NQKV; a.rpl = p.rpl; a.fresh = fresh;
  a.per_layer = 0; a.attw = p.attw; a.att_floats = p.att_floats; a.early = p.early;
  for (int i = 0; i < STEP_PHASES; ++i) { a.nblk[i] = p.nblk[i]; a.tpb[i] = p.tpb[i]; a.per_layer += p.nblk[i]; }
  a.eps = c->cfg.normalization_layer_epsilon;
  a.row_slot = c->row_slot; a.row_pos = c->row_pos; a.row_active = c->row_active; a.page_map = c->ps.page_map;
  a.rope_sin = c->rope_sin; a.rope_cos = c->rope_cos; a.g = c->geom;
  if (tokens != nullptr) {
    hipLaunchKernelGGL(k_step_begin, dim3(R), dim3(256), 0, st, tokens, step_front(c), c->gave);
    LAUNCHCHK();
  }
  *hidden = c->step_ws + (size_t)c->L * a.lstride - (size_t)16 * c->E;
#define ST(HD_, GQ_) if (c->D == HD_ && c->GQ == GQ_) return launch_step_t<HD_, GQ_>(a, c->L, p.lds, st);
  ST(128, 1) ST(128, 2) ST(64, 1) ST(64, 2)
#undef ST
  return set_err(IXT_ERR_UNSUPPORTED, "step geometry hd=%d gq=%d", c->D, c->GQ);
}

template <int G>
static int launch_mid_t(const MidArgs& a, int blocks, size_t lds, hipStream_t st) {
  HIPCHK((lds_room<&k_mid<G>>(2 * MID_BUF_STEPS * 1024)));
  hipLaunchKernelGGL(k_mid<G>, dim3((unsigned)blocks), dim3(MID_NW * 64), lds, st, a);
  LAUNCHCHK();
  return IXT_OK;
}
// What stands between the attentions of layers l and l + 1 (-1: the embedding and what is in front of the first attention).  Behind the last layer: the rows, *hidden, and with
// `final` their norm for the head, *normed.
int launch_mid(ixt_ctx* c, int R, int l, const int32_t* tokens, bool final, const bf16_t** hidden, const bf16_t** normed, hipStream_t st) {
  const MidPlan p = mid_plan(c, R);
  c->forms |= IXT_FORM_MID;
  const int G = (R + 15) / 16, lines = MID_PHASES * STEP_NS;
  bf16_t *h[2], *ws = c->mid_ws;
  auto take = [&](size_t n) { bf16_t* q = ws; ws += n; return q; };
  MidArgs a;
  h[0] = take((size_t)64 * c->E); h[1] = take((size_t)64 * c->E);
  a.hmid = take((size_t)64 * c->E); a.xn1 = take((size_t)64 * c->E); a.xn2 = take((size_t)64 * c->E); a.act = take((size_t)64 * c->F);
  const bool end = l == c->L - 1;
  a.layers = c->step_layers; a.base = c->step_ws; a.layer = l; a.next = end ? -1 : l + 1;
  a.ao = c->ao; a.qbuf = c->qbuf; a.hin = h[(l + 2) & 1]; a.hout = h[(l + 1) & 1];
  a.scale = end ? c->final_norm : c->layers[l + 1].ln1;
  a.cnt = c->mid_cnt + (size_t)(l + 1) * lines * 32; a.wait = c->wait();
  a.R = R; a.E = c->E; a.F = c->F; a.QN = c->QN; a.NQKV = c->NQKV;
  a.early = p.early;
  a.eps = c->cfg.normalization_layer_epsilon;
  a.row_slot = c->row_slot; a.row_pos = c->row_pos; a.row_active = c->row_active; a.page_map = c->ps.page_map;
  a.rope_sin = c->rope_sin; a.rope_cos = c->rope_cos; a.g = c->geom;
  int blocks = 0, before = -1;
  for (int i = 0; i < MID_PHASES; ++i) {
    const bool here = i <= MID_DOWN ? l >= 0 : i == MID_N1 ? !end || final : !end;
    a.tpb[i] = p.tpb[i];
    a.nblk[i] = here ? p.nblk[i] : 0;
    a.prev[i] = before;
    if (here) before = i;
    blocks += a.nblk[i];
  }
  if (l < 0 && tokens != nullptr) {
    hipLaunchKernelGGL(k_step_begin, dim3(R), dim3(256), 0, st, tokens, mid_front(c), c->gave);
    LAUNCHCHK();
  }
  if (hidden) *hidden = a.hout;
  if (normed) *normed = a.xn1;
  return G == 2 ? launch_mid_t<2>(a, blocks, p.lds, st) : G == 3 ? launch_mid_t<3>(a, blocks, p.lds, st) : launch_mid_t<4>(a, blocks, p.lds, st);
}
