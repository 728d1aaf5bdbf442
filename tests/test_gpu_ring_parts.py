"""f32 sums of few tiles over a long K, three blocks a tile: against the oracle's bits and against one block a tile, several launches behind one another (the words
through which blocks hand their sums on are zero between launches); ragged rows and columns, short last chains, six to eighteen chains."""
import ctypes

import numpy as np
import pytest

import helpers as H
from test_gpu_ops import _st, _vp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def wide():
  import torch
  from oracle import oracle as O
  cfg = H.make_config(max_prefill_predict_length=256, max_target_length=288, base_mlp_dim=9216, pagedattn_num_pages=64)
  eng, _ = H.make_engine(cfg, H.synth.synth_weights(cfg, 0))
  return {"eng": eng, "O": O, "torch": torch}


PARTS = 8


def _forms(eng):
  out = ctypes.c_int32(-1)
  H.lib.check(eng.lib.ixt_pass_forms(eng._ctx, ctypes.byref(out)))
  return out.value


# rows, K, columns: 6, 7, 8 chains (a part of one chain or two) and 11 beside tiles of 64 x 64, 12 and 16 beside 64 x 32, 17 and 18 beside both; short last chains, ragged rows and columns
CASES = [(256, 3072, 2304), (200, 3456, 2064), (193, 4096, 2560), (250, 5504, 2320), (190, 6144, 2000), (300, 6144, 1520), (161, 8192, 1600), (256, 8448, 2304), (129, 8576, 2064),
         (250, 9088, 2304), (256, 9216, 2048)]


@pytest.mark.parametrize("R,K,N", CASES)
def test_parts_against_the_oracle(wide, R, K, N):
  """Rows at the edges of the tiles, every column."""
  torch, eng, O = wide["torch"], wide["eng"], wide["O"]
  rng = np.random.default_rng(R + K + N)
  x, w = H.rand_bf16(rng, (R, K)), H.rand_bf16(rng, (K, N), 0.05)
  rows = sorted({0, 15, 16, 63, 64, 127, 128, R - 2, R - 1})
  ref, some = np.zeros((len(rows), N), np.float32), np.ascontiguousarray(x[rows])
  O.lib().orc_dot_rows(O._p(some, O._u16p), K, len(rows), O._p(w, O._u16p), K, N, O._p(ref, O._f32p), N)
  xd, wd, out = H.dev_bf16(x), H.dev_bf16(w), torch.empty((R, N), dtype=torch.float32, device="cuda")
  H.lib.check(eng.lib.ixt_op_dot(eng._ctx, _vp(xd), _vp(wd), _vp(out), R, K, N, _st(torch)))
  assert _forms(eng) == PARTS
  assert np.array_equal(out.cpu().numpy()[rows].view(np.uint32), ref.view(np.uint32))


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
      assert _forms(eng) == (PARTS if parts else 0)
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
