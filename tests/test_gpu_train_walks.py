"""The training step's attention by walks over the keys (heads of 64 and 128) where its tiles, its held rows and its ranges end, with segments that it may pass over and segments that it
must not: against the f32 oracle, within what rounding the backward signals to bf16 gives (tests/test_gpu_train.py: 2 % of every gradient, 1e-4 of the loss)."""
import importlib

import numpy as np
import pytest

from test_gpu_train import f32_params, packed_batch, train_config
from test_gpu_train_shapes import step_and_oracle

AT = importlib.import_module("maxtext-indextts2_amd.audio_training")
pytestmark = pytest.mark.gpu

SEGMENTS = {
    "one": lambda S, r: np.ones(S),
    # a few tokens, then padding over several tiles
    "padded": lambda S, r: (np.arange(S) < max(5, S // 3)).astype(int),
    # packed rows: segments that end inside tiles and on their edges
    "packed": lambda S, r: 1 + np.searchsorted(np.sort(np.r_[64, 128, r.integers(1, S, 5)]), np.arange(S), side="right"),
    # a segment that comes back behind another one, across tiles
    "returning": lambda S, r: 1 + np.arange(S) // 40 % 2,
}


@pytest.mark.parametrize("segments", list(SEGMENTS))
@pytest.mark.parametrize("dim,heads,kv,length,rows", [(64, 2, 2, 64, 2), (64, 3, 1, 136, 1), (64, 2, 2, 512, 1), (64, 4, 2, 584, 2), (128, 2, 2, 128, 1), (128, 2, 1, 520, 1), (128, 1, 1, 1096, 1)])
def test_walks(dim, heads, kv, length, rows, segments):
  cfg = train_config(base_emb_dim=64, base_num_query_heads=heads, base_num_kv_heads=kv, head_dim=dim, base_mlp_dim=72, vocab_size=264, max_target_length=length,
                     per_device_batch_size=float(rows), base_num_decoder_layers=1)
  rng = np.random.default_rng(length + dim)
  b = AT.synthetic_batch(cfg, 7)
  for r in range(rows):
    seg = SEGMENTS[segments](length, rng).astype(np.int32)
    b["inputs_segmentation"][r] = seg
    b["targets_segmentation"][r] = seg
    b["inputs_position"][r] = np.arange(length)
  m, grads, o = step_and_oracle(cfg, f32_params(cfg, 11), b)
  assert abs(m["learning/loss"] - o["learning/loss"]) <= 1e-4 * abs(o["learning/loss"])
  for k, g in grads.items():
    ref = o["grads"][k]
    assert float((g - ref).norm()) <= 2e-2 * float(ref.norm()) + 1e-12, k


@pytest.mark.parametrize("dim,length", [(32, 520), (96, 1032), (32, 2056), (64, 4104)])
def test_attention_through_memory(dim, length):
  """Heads of other sizes and longer rows: scores, softmax (rows of up to 2048, 4096 and more columns) and products one behind the other."""
  cfg = train_config(base_emb_dim=64, base_num_query_heads=2, base_num_kv_heads=1, head_dim=dim, base_mlp_dim=72, vocab_size=264, max_target_length=length, per_device_batch_size=1.0,
                     base_num_decoder_layers=1)
  m, grads, o = step_and_oracle(cfg, f32_params(cfg, 13), packed_batch(cfg, 43))
  assert abs(m["learning/loss"] - o["learning/loss"]) <= 1e-4 * abs(o["learning/loss"])
  for k, g in grads.items():
    ref = o["grads"][k]
    assert float((g - ref).norm()) <= 2e-2 * float(ref.norm()) + 1e-12, k


def test_wide_walks():
  """Enough heads for 32 rows a wave on the way back (512 blocks of 128 rows), rows that end inside a tile."""
  cfg = train_config(base_emb_dim=64, base_num_query_heads=16, base_num_kv_heads=16, head_dim=64, base_mlp_dim=72, vocab_size=264, max_target_length=152, per_device_batch_size=16.0,
                     base_num_decoder_layers=1)
  b = AT.synthetic_batch(cfg, 9)
  b["inputs_segmentation"][:] = (np.arange(152)[None] < 152 - 9 * np.arange(16)[:, None]).astype(np.int32)
  b["targets_segmentation"][:] = b["inputs_segmentation"]
  m, grads, o = step_and_oracle(cfg, f32_params(cfg, 12), b)
  assert abs(m["learning/loss"] - o["learning/loss"]) <= 1e-4 * abs(o["learning/loss"])
  for k, g in grads.items():
    ref = o["grads"][k]
    assert float((g - ref).norm()) <= 2e-2 * float(ref.norm()) + 1e-12, k
