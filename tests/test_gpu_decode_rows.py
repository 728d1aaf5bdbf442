"""Decode steps of 33 rows and more with few kv heads, both sides of the line between the eight-wave and the four-wave attention: tokens and logits of every
step against the oracle, then the same steps with four waves only, bit for bit."""
import numpy as np
import pytest

import helpers as H
from test_gpu_engine import run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,kv,heads,dim", [(64, 1, 2, 64), (65, 4, 4, 64), (64, 4, 8, 64), (33, 2, 4, 128), (128, 2, 2, 128), (129, 2, 2, 64)])
def test_steps_of_few_kv_heads(rows, kv, heads, dim):
  cfg = H.make_config(per_device_batch_size=float(rows), base_num_query_heads=heads, base_num_kv_heads=kv, head_dim=dim, max_prefill_predict_length=48, max_target_length=64,
                      pagedattn_num_pages=2 * rows + 2, pagedattn_tokens_per_page=32, base_num_decoder_layers=1)
  w = H.synth.synth_weights(cfg, rows + kv)
  rng = np.random.default_rng(rows)
  prompts = [(H.synth.synth_prompt(cfg.vocab_size, 48, i)[0], int(n)) for i, n in enumerate(np.r_[48, 1, rng.integers(1, 49, rows - 2)])]
  eight = run_pair(cfg, w, prompts, steps=4)
  four = run_pair(cfg, w, prompts, steps=4, options={"small_attn_max_blocks": 0})
  assert np.array_equal(eight, four)


@pytest.mark.parametrize("rows,dim", [(63, 64), (65, 256)])
def test_steps_of_capped_rows(rows, dim):
  """Gemma-2 decode rows on both sides of the tiled attention's first row: every row has pages of its own, so the per-row kernels serve them."""
  cfg = H.make_config("gemma2-tiny", per_device_batch_size=float(rows), head_dim=dim, max_prefill_predict_length=48, max_target_length=64, pagedattn_num_pages=2 * rows + 2,
                      pagedattn_tokens_per_page=32, sliding_window_size=24, base_num_decoder_layers=1)
  w = H.synth.synth_weights(cfg, rows)
  prompts = [(H.synth.synth_prompt(cfg.vocab_size, 48, i)[0], 1 + (29 * i) % 48) for i in range(rows)]
  run_pair(cfg, w, prompts, steps=4)
