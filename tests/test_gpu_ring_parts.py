"""f32 sums of few tiles over a long K, three blocks a tile: against the oracle's bits and against one block a tile, several launches behind one another (the words
through which blocks hand their sums on are zero between launches); ragged rows and columns, a short last chain, seventeen and eighteen chains."""
import numpy as np
import pytest

import helpers as H
from test_gpu_ops import _dot_case, _st, _vp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def wide():
  import torch
  from oracle import oracle as O
  cfg = H.make_config(max_prefill_predict_length=256, max_target_length=288, base_mlp_dim=9216, pagedattn_num_pages=64)
  eng, _ = H.make_engine(cfg, H.synth.synth_weights(cfg, 0))
  return {"eng": eng, "O": O, "torch": torch}


@pytest.mark.parametrize("R,K,N", [(130, 9216, 48), (200, 8448, 80), (250, 9088, 16), (256, 8704, 32)])
def test_parts_against_the_oracle(wide, R, K, N):
  rng = np.random.default_rng(R + K + N)
  _dot_case(wide, H.rand_bf16(rng, (R, K)), H.rand_bf16(rng, (K, N), 0.05))


@pytest.mark.parametrize("R,K,N", [(256, 9216, 2304), (129, 9216, 2064), (190, 8320, 2000)])
def test_parts_equal_whole_sums(wide, R, K, N):
  torch, eng = wide["torch"], wide["eng"]
  g = torch.Generator(device="cuda").manual_seed(R + N)
  out = []
  for launch in range(4):
    x, w = (torch.randn(shape, generator=g, device="cuda").mul_(f).bfloat16() for shape, f in (((R, K), 1.0), ((K, N), 0.05)))
    got = []
    for parts in (1, 0):
      H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"ring_parts", parts))
      out = torch.full((R, N), float("nan"), device="cuda")
      H.lib.check(eng.lib.ixt_op_dot(eng._ctx, _vp(x), _vp(w), _vp(out), R, K, N, _st(torch)))
      got.append(out)
    H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"ring_parts", 1))
    assert torch.equal(got[0].view(torch.int32), got[1].view(torch.int32)), launch
  assert eng.exchange_status() == 0


def test_a_hand_over_that_gave_up_leaves_nothing_behind(wide):
  """Takers that do not wait at all, then launches with patience, which must not find a word of the late hand-over."""
  torch, eng = wide["torch"], wide["eng"]
  g = torch.Generator(device="cuda").manual_seed(3)
  x, w = (torch.randn(shape, generator=g, device="cuda").mul_(f).bfloat16() for shape, f in (((256, 9216), 1.0), ((9216, 2304), 0.05)))

  def run(polls, parts=1):
    for name, value in ((b"wait_polls", polls), (b"ring_parts", parts)):
      H.lib.check(eng.lib.ixt_set_option(eng._ctx, name, value))
    out = torch.full((256, 2304), float("nan"), device="cuda")
    H.lib.check(eng.lib.ixt_op_dot(eng._ctx, _vp(x), _vp(w), _vp(out), 256, 9216, 2304, _st(torch)))
    return out.view(torch.int32)

  try:
    whole = run(1 << 20, 0)
    for _ in range(4):
      run(0)
      assert torch.equal(run(1 << 20), whole)
    assert eng.exchange_status() == 1                     # (with no look at all some taker was early)
  finally:
    for name, value in ((b"wait_polls", 1 << 20), (b"ring_parts", 1)):
      H.lib.check(eng.lib.ixt_set_option(eng._ctx, name, value))
