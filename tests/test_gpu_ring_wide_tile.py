"""The many-row matrix product's tile of 128 x 192 (three column tiles a wave), forced, in each epilogue that it has, against the oracle's bits: edges of a row group and of its row blocks,
partial column groups, fewer chunks than ring slots, a short last chain.  Hybrid decoders, whose oracle is one of 64 bits: the bits of the tile of 128 x 128."""
import numpy as np
import pytest

import helpers as H
import lulenex_helpers as LH
import suzulix_helpers as SH
import vazilorn_helpers as ZH
import vilepel_helpers as VH
from test_gpu_engine import run_pair
from test_gpu_ops import _dot_case, ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,K,N", [(128, 128, 192), (191, 640, 208), (192, 256, 16), (193, 1152, 320), (250, 2048, 208), (250, 512, 256)])
def test_sums(ctx, R, K, N):
  eng = ctx["eng"]
  H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"ring_cfg", 8))
  try:
    rng = np.random.default_rng(R + K + N)
    _dot_case(ctx, H.rand_bf16(rng, (R, K)), H.rand_bf16(rng, (K, N), 0.05))
  finally:
    H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"ring_cfg", 0))


@pytest.mark.parametrize("model,rows", [("ixt-tiny", 150), ("ixt-tiny", 192), ("ixt-tiny", 209), ("gemma2-tiny", 209)])
def test_a_prompt(model, rows):
  """RoPE and the page write, and residuals, of a whole pass; the units' product, whose gate pairs are an even number of column tiles, takes another."""
  cfg = H.make_config(model, max_prefill_predict_length=224, max_target_length=240, per_device_batch_size=1.0)
  run_pair(cfg, H.synth.synth_weights(cfg, 7), [(H.synth.synth_prompt(cfg.vocab_size, 224, 71)[0], rows)], steps=2, options={"ring_cfg": 8})


@pytest.mark.parametrize("rows", [150, 209])
def test_a_prompt_of_llama31_positions(rows):
  cfg = H.make_config(rope_type="llama3.1", max_prefill_predict_length=224, max_target_length=240)
  run_pair(cfg, H.synth.synth_weights(cfg, 8), [(H.synth.synth_prompt(cfg.vocab_size, 224, 72)[0], rows)], steps=2, options={"ring_cfg": 8})


# (tanh norms behind the last products; a unit without a gate; routed units without a gate and routed down products)
HYBRIDS = {
    "tanh norms": (ZH, ZH.with_mlp(ZH.attn(), ZH.dense(200))),
    "unit": (LH, LH.with_mlp(LH.parallel(), LH.dense(330))),
    "routed units": (SH, SH.with_mlp(SH.retention(), SH.moe(ff=330, experts=3, top=2, shared=210))),
}


@pytest.mark.parametrize("rows", [191, 300])
@pytest.mark.parametrize("name", list(HYBRIDS))
def test_hybrid_decoders(tmp_path, name, rows):
  helpers, layer = HYBRIDS[name]
  cfg = helpers.model([layer], width=230)
  eng, _ = VH.engine(VH.write_model(tmp_path, cfg, helpers.random_weights(cfg, 3)), dtype="bfloat16", target=320, rows=320, pages=40)
  t, got = VH.tokens(cfg, rows, 5), []
  for tile in (1, 8):
    H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"ring_cfg", tile))
    got.append(VH.run_portions(VH.scheduler(eng), f"r{tile}", t, (rows,)))
  assert np.isfinite(got[0]).all() and float(np.abs(got[0]).max()) > 0
  assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
  eng.close()
