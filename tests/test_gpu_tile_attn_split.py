"""Prefill attention with heads of 128 behind the last whole round of blocks (k_attn_mscores and k_attn_mtile by halves of a value, beside the whole tiles' launch) against the kernels that
walk one row at a time: token ids, f32 logits and K/V bit for bit; a chunk that is split in part, chunks that are split as a whole, one, two and four query heads a kv head."""
import numpy as np
import pytest

import helpers as H
from test_gpu_tile_attn import _prefill_long
from test_gpu_tile_attn_matrix import _same

pytestmark = pytest.mark.gpu


# (16 kv heads: 16 tiles a round; tiles of 16, 8 and 4 rows.  Chunks of 300, 170 and 260 rows behind 2560 keys and more: split in part, in units of 1, 2 and 4 tiles, 20 heads in rounds that they do not fill)
@pytest.mark.parametrize("nq,nkv,length,chunk", [(16, 16, 1400, 340), (16, 16, 2500, 350), (16, 16, 3500, 500), (32, 16, 1500, 170), (32, 16, 1300, 301), (16, 4, 2300, 300),
                                                  (16, 16, 3400, 300), (16, 4, 3400, 300), (32, 16, 3250, 170), (20, 20, 3200, 260)])
def test_split_tiles_equal_the_row_kernel(nq, nkv, length, chunk):
  cfg = H.make_config(base_emb_dim=256, base_num_query_heads=nq, base_num_kv_heads=nkv, head_dim=128, base_mlp_dim=384, base_num_decoder_layers=1,
                      vocab_size=1024, model_name="default", per_device_batch_size=1.0, use_chunked_prefill=True, prefill_chunk_size=512,
                      max_prefill_predict_length=512, max_target_length=3584, pagedattn_tokens_per_page=32, pagedattn_num_pages=116)
  w = H.synth.synth_weights(cfg, 41)
  toks = np.random.default_rng(length).integers(1, cfg.vocab_size, size=length).astype(np.int32)
  _same(*(_prefill_long(cfg, w, toks, chunk, {"attn_tile": tile, "attn_tile_min_rows": 1}) for tile in (1, 0)))
