"""The many-row matrix product's tile of 128 x 192 (three column tiles a wave), forced, in each epilogue that it has, against the oracle's bits: edges of a row group and of its row blocks,
partial column groups, fewer chunks than ring slots, a short last chain."""
import numpy as np
import pytest

import helpers as H
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
