"""Passes of few rows as one launch (k_step): tokens, logits, keys and values of every step against the oracle, bit for bit, at the edges of its tiles -- short last
chains, one to sixteen chains, blocks of sums of squares that are not whole, rows around the powers of two, contexts around pages and around the keys of a
round of waves, idle slots, prompts in portions of at most 16 rows -- and the same with five launches a layer."""
import numpy as np
import pytest

import helpers as H
from test_gpu_engine import run_pair

pytestmark = pytest.mark.gpu

CASES = [
    # rows, emb, query heads, kv heads, dim, mlp, longest prompt, layers
    (1, 384, 2, 2, 64, 512, 33, 3),
    (2, 640, 2, 1, 128, 1152, 64, 2),
    (3, 1152, 4, 4, 64, 4608, 31, 2),
    (5, 768, 12, 12, 64, 2048, 40, 2),
    (8, 2048, 16, 16, 128, 7168, 32, 1),
    (9, 2048, 2, 2, 128, 8192, 20, 2),
    (16, 512, 10, 10, 64, 1024, 70, 2),
    (1, 512, 2, 2, 64, 512, 1100, 2),
    (14, 512, 10, 10, 64, 512, 560, 1),
]


def _config(rows, emb, heads, kv, dim, mlp, longest, layers, **keys):
  pages = -(-(longest + 8) // 32)
  return H.make_config(per_device_batch_size=float(rows), base_emb_dim=emb, base_num_query_heads=heads, base_num_kv_heads=kv, head_dim=dim, base_mlp_dim=mlp,
                       base_num_decoder_layers=layers, max_prefill_predict_length=longest, max_target_length=longest + 8, pagedattn_num_pages=rows * pages + 2,
                       pagedattn_tokens_per_page=32, **keys)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_steps_as_one_launch(case):
  rows, longest = case[0], case[6]
  cfg = _config(*case)
  w = H.synth.synth_weights(cfg, rows)
  rng = np.random.default_rng(rows)
  lengths = [longest, 1, max(1, longest - 1)][:rows] + [int(n) for n in rng.integers(1, longest + 1, max(0, rows - 4))]      # from four rows on one slot stays idle
  prompts = [(H.synth.synth_prompt(cfg.vocab_size, longest, i)[0], n) for i, n in enumerate(lengths)]
  one = run_pair(cfg, w, prompts, steps=5, forms=1)
  assert np.array_equal(one, run_pair(cfg, w, prompts, steps=5, options={"small_step": 0}, forms=0))


@pytest.mark.parametrize("rope", ["default", "llama3.1"])
def test_portions_of_a_prompt(rope):
  """Rows of a pass that see each other's keys, and those of earlier portions, in pages that the pass writes to."""
  cfg = _config(2, 512, 4, 2, 64, 1024, 48, 2, use_chunked_prefill=True, rope_type=rope, rope_max_timescale=500000 if rope == "llama3.1" else 10000)
  w = H.synth.synth_weights(cfg, 5)
  prompts = [(H.synth.synth_prompt(cfg.vocab_size, 48, i)[0], n) for i, n in enumerate((48, 37))]
  chunks = [[16, 9, 7, 16], [1, 13, 8, 15]]
  one = run_pair(cfg, w, prompts, steps=4, chunks=chunks)
  assert np.array_equal(one, run_pair(cfg, w, prompts, steps=4, chunks=chunks, options={"small_step": 0}))


def test_packed_rows():
  """Three prompts in one pass of 16 rows: rows of other groups in between."""
  import torch
  cfg = _config(3, 512, 2, 2, 128, 1024, 32, 2, ixt_staging_groups=3, ixt_max_packed_rows=16, use_chunked_prefill=True)
  w = H.synth.synth_weights(cfg, 9)
  lens = np.array([7, 1, 8], np.int32)
  toks = np.concatenate([H.synth.synth_prompt(cfg.vocab_size, 32, i)[0][:n] for i, n in enumerate(lens)]).astype(np.int32)
  out = []
  for step in (1, 0):
    eng, params = H.make_engine(cfg, w)
    H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"small_step", step))
    cache, prefix, _ = eng.prefill_concat(params=params, padded_tokens=toks, decoder_positions=np.concatenate([np.arange(n) for n in lens]).astype(np.int32),
                                          decoder_segment_ids=np.repeat(np.arange(3) + 1, lens).astype(np.int32), start_pos=np.array([0, 7, 8], np.int32), true_lengths=lens, num_prompts=3)
    out.append((prefix["logits"].cpu().numpy().view(np.uint32), prefix["tokens"].cpu().numpy()))
    assert eng.exchange_status() == 0
    del eng
    torch.cuda.synchronize()
  assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


def test_passes_of_two_engines_on_two_streams():
  """Steps of two models in flight on two streams: never two whole steps as one launch beside each other (each would hold compute units that the other's blocks have to
  start on), and every token is what a model alone gives."""
  import torch
  lens, steps = (33, 20), 200
  cfgs = [_config(1, 2048, 16, 16, 128, 7168, 33 + steps, 2), _config(1, 768, 12, 12, 64, 2048, 33 + steps, 6)]
  engines = [H.make_engine(cfg, H.synth.synth_weights(cfg, i)) for i, cfg in enumerate(cfgs)]
  streams = [torch.cuda.Stream() for _ in cfgs]

  def begin(i):
    toks = H.synth.synth_prompt(cfgs[i].vocab_size, 33, i)[0]
    eng, params = engines[i]
    prefix, _ = eng.prefill(params=params, padded_tokens=toks, true_length=lens[i], slot=0)
    return eng.insert(prefix, eng.init_decode_state(), 0)

  def run(together):
    out, states = [[], []], [None, None]
    order = [0, 1] * steps if together else [0] * steps + [1] * steps
    for i in (0, 1):
      with torch.cuda.stream(streams[i]):
        states[i] = begin(i)
    torch.cuda.synchronize()
    for i in order:
      with torch.cuda.stream(streams[i]):
        states[i], result = engines[i][0].generate(engines[i][1], states[i])
        out[i].append(result.data.clone())
      if not together:
        streams[i].synchronize()
    torch.cuda.synchronize()
    for i in (0, 1):
      assert engines[i][0].exchange_status() == 0
      engines[i][0].release_pages(0)
    return [torch.stack(o).cpu().numpy() for o in out]

  alone, both = run(False), run(True)
  assert all(np.array_equal(x, y) for x, y in zip(alone, both))
