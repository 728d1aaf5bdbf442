"""The prefill attention on the f32 matrix units where more blocks than CUs take four waves each (513 .. 1024 keys), against the kernels that walk one row at a
time: chunks whose tiles see all keys of a super-block, some, or none, at the edges of the form, with and without windows and caps; and heads of 256 with both through
the forms of three and four rounds (2049 .. 3072 .. 4096 keys)."""
import numpy as np
import pytest

import helpers as H
from test_gpu_tile_attn import _prefill_long
from test_gpu_tile_attn_matrix import _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,hd,nq,nkv,window,option", [("default", 64, 12, 12, 0, "attn_tile"), ("default", 128, 16, 8, 0, "attn_tile"), ("gemma2-tiny", 256, 8, 4, 140, "gemma_tile"),
                                                         ("gemma2-tiny", 128, 16, 4, 4096, "gemma_tile")])
@pytest.mark.parametrize("length,chunk", [(1024, 530), (513, 513)])
def test_two_blocks_a_cu(model, hd, nq, nkv, window, option, length, chunk):
  keys = dict(model_name=model, override_model_config=True, sliding_window_size=window) if window else dict(model_name=model, base_emb_dim=256, base_mlp_dim=384, vocab_size=1024)
  cfg = H.make_config(head_dim=hd, base_num_query_heads=nq, base_num_kv_heads=nkv, base_num_decoder_layers=1, per_device_batch_size=1.0, use_chunked_prefill=True,
                      prefill_chunk_size=530, max_prefill_predict_length=530, max_target_length=1056, pagedattn_tokens_per_page=32, pagedattn_num_pages=36, **keys)
  w = H.synth.synth_weights(cfg, 41)
  toks = np.random.default_rng(length).integers(1, cfg.vocab_size, size=length).astype(np.int32)
  _same(_prefill_long(cfg, w, toks, chunk, {option: 1, "attn_tile_min_rows": 1}), _prefill_long(cfg, w, toks, chunk, {option: 0}))


@pytest.mark.parametrize("nq,nkv,window,length,chunk", [(8, 4, 4096, 3330, 256), (8, 4, 700, 3330, 250), (4, 4, 2100, 3072, 256), (8, 2, 4096, 3073, 130),
                                                        (8, 4, 4096, 1025, 40), (4, 4, 30, 545, 17)])
def test_heads_of_256_at_many_keys(nq, nkv, window, length, chunk):
  cfg = H.make_config(model_name="gemma2-tiny", override_model_config=True, head_dim=256, base_num_query_heads=nq, base_num_kv_heads=nkv, sliding_window_size=window,
                      base_num_decoder_layers=1, per_device_batch_size=1.0, use_chunked_prefill=True, prefill_chunk_size=256, max_prefill_predict_length=256,
                      max_target_length=3360, pagedattn_tokens_per_page=32, pagedattn_num_pages=108)
  w = H.synth.synth_weights(cfg, 43)
  toks = np.random.default_rng(length).integers(1, cfg.vocab_size, size=length).astype(np.int32)
  _same(_prefill_long(cfg, w, toks, chunk, {"gemma_tile": 1, "attn_tile_min_rows": 1}), _prefill_long(cfg, w, toks, chunk, {"gemma_tile": 0}))
