"""The many-row matrix product's tiles: 256 x 128, 64 x 64, 64 x 16 and 128 x 128 with two blocks on a CU, forced in turn, and the rule that chooses
among all of them, against the oracle's bits.  Sizes: ragged last row groups and blocks, partial column groups, fewer chunks than ring slots, a short last
chain, several rounds of blocks."""
import numpy as np
import pytest

import helpers as H
from test_gpu_ops import _dot_case, _st, _vp, ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg_id", [4, 5, 6, 7])
@pytest.mark.parametrize("R,K,N", [(128, 1024, 256), (250, 1152, 256), (200, 2048, 144), (129, 640, 16), (256, 512, 80), (130, 128, 496)])
def test_forced_tile(ctx, cfg_id, R, K, N):
  eng = ctx["eng"]
  H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"ring_cfg", cfg_id))
  try:
    rng = np.random.default_rng(R + K + N + cfg_id)
    _dot_case(ctx, H.rand_bf16(rng, (R, K)), H.rand_bf16(rng, (K, N), 0.05))
  finally:
    H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"ring_cfg", 0))


@pytest.mark.parametrize("R,K,N", [(128, 512, 400), (129, 640, 496), (250, 384, 256), (145, 256, 432)])
def test_chosen_tile(ctx, R, K, N):
  rng = np.random.default_rng(R + K + N)
  _dot_case(ctx, H.rand_bf16(rng, (R, K)), H.rand_bf16(rng, (K, N), 0.05))


@pytest.mark.parametrize("R,V", [(32, 4112), (33, 4112), (64, 4112), (65, 4112), (127, 4112), (40, 16), (130, 16), (130, 48), (40, 80), (130, 144)])
def test_unembedding_of_some_rows(ctx, R, V):
  """33 rows and more: the sampling epilogue on 64-row tiles (rounded logits and the first index of the maximum), a vocabulary that is no multiple of a
  tile, down to one that ends inside the first column group (its pairs of maximum and index are those of a whole one)."""
  torch, O = ctx["torch"], ctx["O"]
  cfg = H.make_config(per_device_batch_size=float(R), pagedattn_num_pages=256, vocab_size=V)
  w = H.synth.synth_weights(cfg, 3)
  eng, _ = H.make_engine(cfg, w)
  E = cfg.emb_dim
  y = H.rand_bf16(np.random.default_rng(R), (R, E))
  lg = np.zeros((R, V), np.float32)
  wl = w["params/decoder/logits_dense/kernel"].reshape(E, V)
  O.lib().orc_dot_rows(O._p(y, O._u16p), E, R, O._p(wl, O._u16p), E, V, O._p(lg, O._f32p), V)
  lg = O.bf16_to_f32(O.f32_to_bf16(lg)).reshape(R, V)
  logits = torch.empty((R, V), dtype=torch.float32, device="cuda")
  amax = torch.empty((R,), dtype=torch.int32, device="cuda")
  H.lib.check(eng.lib.ixt_op_unembed_argmax(eng._ctx, _vp(H.dev_bf16(y)), R, _vp(logits), _vp(amax), _st(torch)))
  assert np.array_equal(logits.cpu().numpy().view(np.uint32), lg.view(np.uint32))
  assert np.array_equal(amax.cpu().numpy(), np.argmax(lg, axis=-1).astype(np.int32))


@pytest.mark.parametrize("rows", [16, 17, 64, 65, 127])
def test_gelu_gate_and_query_scale_epilogues(rows):
  """A Gemma-2 prompt of that many rows, one prefill call: up to 16 rows split-K dots with kernels of their own, from 17 on RoPE, the query scale, the page
  write and the gelu gate as epilogues; then a few steps, token by token against the oracle."""
  from test_gpu_engine import run_pair
  cfg = H.make_config("gemma2-tiny", max_prefill_predict_length=128, max_target_length=160, per_device_batch_size=2.0, pagedattn_num_pages=64, head_dim=128,
                      base_num_query_heads=4, base_num_kv_heads=2, sliding_window_size=24)
  w = H.synth.synth_weights(cfg, 9)
  run_pair(cfg, w, [(H.synth.synth_prompt(cfg.vocab_size, 128, 70)[0], rows)], steps=4)
