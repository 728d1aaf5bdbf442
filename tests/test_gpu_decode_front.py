"""A decode step's first and last launch (page advance, rows, embedding; tokens, state, results) on both sides of the forms that share the first one: few rows,
some rows, many; the last slot idle, pages taken on the way.  Tokens, logits, page state and slots against the oracle."""
import numpy as np
import pytest

import helpers as H
from test_gpu_engine import run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [2, 16, 17, 64, 65, 257])
def test_steps_with_an_idle_slot(slots):
  cfg = H.make_config(per_device_batch_size=float(slots), max_prefill_predict_length=32, max_target_length=64, pagedattn_num_pages=2 * slots + 2, pagedattn_tokens_per_page=32,
                      base_num_decoder_layers=1)
  prompts = [(H.synth.synth_prompt(cfg.vocab_size, 32, i)[0], 32 - (5 * i) % 7) for i in range(slots - 1)]
  run_pair(cfg, H.synth.synth_weights(cfg, slots), prompts, steps=6)


@pytest.mark.parametrize("slots, heads", [(33, 16), (130, 4), (128, 4), (256, 2), (257, 8)])
def test_rows_of_mixed_lengths(slots, heads):
  """512 to 2048 blocks of attention: rows go to them longest first; short, long, equal and idle ones among each other.  More: as they lie."""
  cfg = H.make_config(per_device_batch_size=float(slots), max_prefill_predict_length=64, max_target_length=96, pagedattn_num_pages=5 * slots + 3, pagedattn_tokens_per_page=32,
                      base_num_decoder_layers=1, base_num_query_heads=heads, base_num_kv_heads=heads)
  prompts = [(H.synth.synth_prompt(cfg.vocab_size, 64, i)[0], 1 + (37 * i) % 64 if i % 3 else 40) for i in range(slots - 1)]
  run_pair(cfg, H.synth.synth_weights(cfg, slots), prompts, steps=3)


def test_results_belong_to_their_step():
  """A result holds its own step's tokens, whatever the engine does afterwards."""
  cfg = H.make_config(per_device_batch_size=3.0)
  engine, params = H.make_engine(cfg, H.synth.synth_weights(cfg, 3))
  toks, n = H.synth.synth_prompt(cfg.vocab_size, cfg.max_prefill_predict_length, 5)
  state = engine.init_decode_state()
  for slot in range(3):
    prefix, _ = engine.prefill(params=params, padded_tokens=toks, true_length=n, slot=slot)
    state = engine.insert(prefix, state, slot)
  results, seen = [], []
  for _ in range(4):
    state, result = engine.generate(params, state)
    results.append(result)
    seen.append(result.data.cpu().numpy().copy())
  for i, result in enumerate(results):
    assert np.array_equal(result.data.cpu().numpy(), seen[i]) and np.array_equal(seen[i][:, 2], np.full(3, seen[0][0, 2] + i)) and np.all(seen[i][:, 1] == 1)
