"""The decode step of a gated-delta layer that takes the low-rank columns' second product in (bfloat16, at most 16 rows, heads of whole 16-column tiles, at most 256 low-rank columns) and,
beyond these, the launch in front of it: logits of decoded tokens against the float64 restatement."""
import numpy as np
import pytest
import torch

import vilepel_helpers as VH
import vilepel_ref as V

pytestmark = pytest.mark.gpu


def decoded(tmp_path, layers, slots, n):
  cfg = VH.model(layers)
  w = VH.random_weights(cfg, 2)
  eng, params = VH.engine(VH.write_model(tmp_path, cfg, w), dtype="bfloat16", slots=slots, pages=8 * slots, rows=64)
  state, toks = eng.init_decode_state(), []
  for i in range(slots):
    t = VH.tokens(cfg, 1 + (5 * i) % 11, 60 + i)
    padded = np.zeros(eng.max_prefill_length, np.int32)
    padded[:len(t)] = t
    prefix, first = eng.prefill(params=params, padded_tokens=padded, true_length=len(t), slot=i)
    state = eng.insert(prefix, state, i)
    toks.append(t.tolist() + [int(first.data[0, 0])])
  prompts, got = [len(t) - 1 for t in toks], [[] for _ in toks]
  state["logits"] = torch.empty((slots, 1, cfg["vocab"]), dtype=torch.float32, device="cuda")
  for _ in range(n):
    state, r = eng.generate(params, state)
    for i in range(slots):
      got[i].append(state["logits"][i, 0].cpu().numpy())
      toks[i].append(int(r.data[i, 0]))
  for i in range(slots):
    VH.check(np.stack(got[i]), V.forward(cfg, w, np.array(toks[i][:-1], np.int32))[prompts[i]:], "bfloat16", i)
  eng.close()


# (low-rank columns: dim + vdim; 272 and dim 24 go the other way)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(1, 1, 16, 16), (3, 3, 48, 80), (4, 2, 128, 128), (2, 1, 16, 240), (2, 2, 16, 256), (1, 1, 144, 16), (2, 2, 24, 16)])
def test_sizes(tmp_path, heads, kv_heads, dim, vdim):
  decoded(tmp_path, [VH.with_mlp(VH.delta(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, conv=4), None)], 2, 12)


@pytest.mark.parametrize("slots", [1, 15, 16, 17])
def test_rows(tmp_path, slots):
  """Two layers of different low-rank columns: each row's own sums, nothing of the other layer's operand."""
  decoded(tmp_path, [VH.with_mlp(VH.delta(heads=3, kv_heads=3, dim=32, vdim=48, conv=3), None), VH.with_mlp(VH.delta(heads=2, kv_heads=1, dim=64, vdim=160, conv=4), None)], slots, 12)


# (33 rows; key sizes 16, 64, 128 and 512.  528 blocks or 264: four waves a block; 792 and, with key size 256, any: eight)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(16, 16, 16, 48), (16, 8, 48, 80), (16, 16, 128, 32), (24, 24, 120, 24), (16, 4, 144, 16), (8, 8, 264, 48)])
def test_waves_of_a_block(tmp_path, heads, kv_heads, dim, vdim):
  """More blocks than two a CU: by four waves where three blocks of them, but two of eight, are on a CU, or where a head has too few value columns for eight."""
  decoded(tmp_path, [VH.with_mlp(VH.delta(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, conv=4), None)], 33, 4)
