"""The prefill attention on the f32 matrix units (k_attn_mtile: 32-token pages) against the kernels that walk one row at a time: token ids, f32 logits
and K/V bit for bit at the edges of its forms (256, 512, 1024, 2048, 4096 keys), with windows and soft caps, and with scores so far apart that the
quotients of the softmax leave the range of the corrected reciprocal (e below 2^-96)."""
import numpy as np
import pytest

import helpers as H
from test_gpu_tile_attn import _prefill_long

pytestmark = pytest.mark.gpu


def _same(a, b):
  assert np.array_equal(a[0], b[0])
  assert np.array_equal(a[1], b[1])
  for (ka, va), (kb, vb) in zip(a[2], b[2]):
    assert np.array_equal(ka, kb) and np.array_equal(va, vb)
  assert a[3] == [0, 0, 0, 0] and b[3] == [0, 0, 0, 0]


@pytest.mark.parametrize("hd,nq,nkv", [(128, 2, 2), (64, 4, 1), (128, 4, 2)])
@pytest.mark.parametrize("length,chunk", [(257, 256), (530, 127), (1041, 240), (2061, 250)])
@pytest.mark.parametrize("spread", [1.0, 64.0])
def test_matrix_tile_equals_row_kernel(hd, nq, nkv, length, chunk, spread):
  cfg = H.make_config(base_emb_dim=256, base_num_query_heads=nq, base_num_kv_heads=nkv, head_dim=hd, base_mlp_dim=384, base_num_decoder_layers=2,
                      vocab_size=1024, model_name="default", per_device_batch_size=1.0, use_chunked_prefill=True, prefill_chunk_size=256,
                      max_prefill_predict_length=256, max_target_length=2112, pagedattn_tokens_per_page=32, pagedattn_num_pages=70)
  w = H.synth.synth_weights(cfg, 23)
  for name in w:
    if name.endswith("query/kernel"):                    # scores `spread` times as far apart (exact: a power of two)
      w[name] = H.synth.f32_to_bf16_bits(H.synth.bf16_bits_to_f32(w[name]) * np.float32(spread)).reshape(w[name].shape)
  toks = np.random.default_rng(length).integers(1, cfg.vocab_size, size=length).astype(np.int32)
  a = _prefill_long(cfg, w, toks, chunk, {"attn_tile": 1, "attn_tile_min_rows": 1})
  b = _prefill_long(cfg, w, toks, chunk, {"attn_tile": 0})
  _same(a, b)


@pytest.mark.parametrize("hd,nq,nkv", [(128, 8, 2), (64, 2, 2)])
def test_matrix_tile_of_the_longest_prefixes(hd, nq, nkv):
  """4200 keys: all four rounds of the last form (3073 .. 4096 keys), then the vector units, which take over past 4096; four query heads a kv head."""
  cfg = H.make_config(base_emb_dim=256, base_num_query_heads=nq, base_num_kv_heads=nkv, head_dim=hd, base_mlp_dim=384, base_num_decoder_layers=1,
                      vocab_size=1024, model_name="default", per_device_batch_size=1.0, use_chunked_prefill=True, prefill_chunk_size=256,
                      max_prefill_predict_length=256, max_target_length=4352, pagedattn_tokens_per_page=32, pagedattn_num_pages=140)
  w = H.synth.synth_weights(cfg, 37)
  toks = np.random.default_rng(hd).integers(1, cfg.vocab_size, size=4200).astype(np.int32)
  matrix, vector, rows = (_prefill_long(cfg, w, toks, 240, {"attn_tile": tile, "attn_tile_min_rows": 1}) for tile in (1, 2, 0))
  _same(matrix, rows)
  _same(vector, rows)


@pytest.mark.parametrize("hd,nq,nkv", [(256, 4, 2), (256, 8, 2), (64, 4, 2), (256, 2, 2)])
@pytest.mark.parametrize("window", [70, 4096])
def test_matrix_tile_with_cap_and_window(hd, nq, nkv, window):
  """Local and global sub-layers, capped scores; 256-column values (two output passes, in one block and in two)."""
  cfg = H.make_config(model_name="gemma2-tiny", override_model_config=True, head_dim=hd, base_num_query_heads=nq, base_num_kv_heads=nkv, sliding_window_size=window,
                      per_device_batch_size=1.0, use_chunked_prefill=True, prefill_chunk_size=256, max_prefill_predict_length=256, max_target_length=640,
                      pagedattn_tokens_per_page=32, pagedattn_num_pages=24)
  w = H.synth.synth_weights(cfg, 29)
  toks = np.random.default_rng(window).integers(1, cfg.vocab_size, size=600).astype(np.int32)
  a = _prefill_long(cfg, w, toks, 250, {"gemma_tile": 1, "attn_tile_min_rows": 1})
  b = _prefill_long(cfg, w, toks, 250, {"gemma_tile": 0})
  _same(a, b)


@pytest.mark.parametrize("model,hd,nq,nkv", [("ixt-tiny", 64, 4, 2), ("ixt-tiny", 128, 8, 8), ("gemma2-tiny", 256, 4, 2)])
@pytest.mark.parametrize("portion", [2, 40])
def test_rows_of_many_page_groups(model, hd, nq, nkv, portion):
  """One mixed step: 62 rows that continue sequences of their own (up to as many page groups in a tile as it has rows, dealt among blocks where CUs are idle)
  and a portion of a prompt; logits, tokens and new K/V against the per-row kernels."""
  import torch
  slots, longest = 63, 300
  cfg = H.make_config(model, per_device_batch_size=float(slots), head_dim=hd, base_num_query_heads=nq, base_num_kv_heads=nkv, base_num_decoder_layers=1,
                      max_prefill_predict_length=longest, max_target_length=longest + 64, pagedattn_tokens_per_page=32, pagedattn_num_pages=slots * 12 + 1)
  w = H.synth.synth_weights(cfg, 31)
  rng = np.random.default_rng(portion)
  lens = [int(n) for n in rng.integers(1, longest, slots)]
  toks = [rng.integers(1, cfg.vocab_size, n + 64).astype(np.int32) for n in lens]

  def step(options):
    eng, params = H.make_engine(cfg, w)
    for name, value in options.items():
      H.lib.check(eng.lib.ixt_set_option(eng._ctx, name.encode(), value))
    for slot, n in enumerate(lens):
      eng.prefill(params=params, padded_tokens=toks[slot][:n], true_length=n, slot=slot)
    entries = [(slot, n, toks[slot][n:n + 1], [0]) for slot, n in enumerate(lens[:-1])]
    entries.append((slots - 1, lens[-1], toks[-1][lens[-1]:lens[-1] + portion], [portion - 1]))
    logits, first = eng.step(entries)
    kv = [H.bits(t).copy() for slot in (0, 7, slots - 1) for t in eng.gather_kv(0, slot, lens[slot] + 1)]
    out = logits.cpu().numpy().view(np.uint32), first.cpu().numpy(), kv
    torch.cuda.synchronize()
    return out

  a, b = step({"attn_tile_min_rows": 1}), step({"attn_tile": 0})
  assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
  assert all(np.array_equal(x, y) for x, y in zip(a[2], b[2]))
