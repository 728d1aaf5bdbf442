"""Passes of 17 to 64 rows with one launch between two attentions (k_mid): tokens, logits, keys and values of every step against the oracle, bit for bit, at the edges
of its tiles -- short last chains, one to sixteen chains, rows of two to four groups, projections whose rows go through LDS and those whose do not, idle slots,
portions of prompts -- and the same with a launch a phase."""
import numpy as np
import pytest

import helpers as H
from test_gpu_engine import run_pair
from test_gpu_step import _config

pytestmark = pytest.mark.gpu

CASES = [
    # rows, emb, query heads, kv heads, dim, mlp, longest prompt, layers
    (17, 384, 2, 2, 64, 512, 9, 3),
    (24, 640, 2, 1, 128, 1152, 7, 2),
    (32, 1152, 4, 4, 64, 4608, 5, 2),
    (33, 768, 12, 12, 64, 2048, 40, 2),
    (48, 2048, 16, 16, 128, 7168, 3, 1),
    (49, 1536, 20, 10, 128, 8192, 3, 1),
    (64, 1536, 2, 2, 128, 8192, 3, 2),
    (57, 2048, 4, 4, 128, 4736, 4, 2),
    (48, 128, 4, 4, 64, 256, 33, 2),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_decode_rows(case):
  rows, longest = case[0], case[6]
  cfg = _config(*case)
  w = H.synth.synth_weights(cfg, rows)
  rng = np.random.default_rng(rows)
  lengths = [longest, 1, max(1, longest - 1)] + [int(n) for n in rng.integers(1, longest + 1, rows - 4)]      # one slot stays idle
  prompts = [(H.synth.synth_prompt(cfg.vocab_size, longest, i)[0], n) for i, n in enumerate(lengths)]
  one = run_pair(cfg, w, prompts, steps=4, forms=2)
  assert np.array_equal(one, run_pair(cfg, w, prompts, steps=4, options={"mid_rows": 0}, forms=0))


@pytest.mark.parametrize("rope", ["default", "llama3.1"])
@pytest.mark.parametrize("dim,heads,kv", [(64, 4, 2), (128, 2, 2)])
def test_portions_of_a_prompt(rope, dim, heads, kv):
  """Portions of 17 to 64 rows behind portions of any size, idle rows of the last group in between; tiles of the matrix units' attention and rows of their own."""
  cfg = _config(2, 512, heads, kv, dim, 1024, 150, 2, use_chunked_prefill=True, rope_type=rope, rope_max_timescale=500000 if rope == "llama3.1" else 10000)
  w = H.synth.synth_weights(cfg, 5)
  prompts = [(H.synth.synth_prompt(cfg.vocab_size, 150, i)[0], n) for i, n in enumerate((150, 97))]
  chunks = [[17, 48, 5, 80], [32, 65]]
  one = run_pair(cfg, w, prompts, steps=3, chunks=chunks)
  for options in ({"mid_rows": 0}, {"attn_tile_min_rows": 1}, {"attn_tile": 0}):
    assert np.array_equal(one, run_pair(cfg, w, prompts, steps=3, chunks=chunks, options=options))


def test_replays_of_a_captured_step():
  """The launches of a step taken down once and replayed, with other work in between: every token is the eager step's."""
  import torch
  case = (20, 512, 4, 4, 64, 1024, 12, 3)

  def run(graph):
    cfg = _config(*case, ixt_use_hip_graph=graph)
    eng, params = H.make_engine(cfg, H.synth.synth_weights(cfg, 8))
    state = eng.init_decode_state()
    for slot in range(20):
      prefix, _ = eng.prefill(params=params, padded_tokens=H.synth.synth_prompt(cfg.vocab_size, 12, slot)[0], true_length=1 + slot % 12, slot=slot)
      state = eng.insert(prefix, state, slot)
    out = []
    for _ in range(6):
      state, result = eng.generate(params, state)
      out.append(result.data.cpu().numpy().copy())
      torch.randn(1 << 20, device="cuda").sum().item()
    assert eng.exchange_status() == 0
    return np.stack(out)

  assert np.array_equal(run(True), run(False))
