"""The many-row matrix product's tiles: 256 x 128, 64 x 64, 64 x 16 and 128 x 128 with two blocks on a CU, forced in turn, and the rule that chooses
among all of them, against the oracle's bits.  Sizes: ragged last row groups and blocks, partial column groups, fewer chunks than ring slots, a short last
chain, several rounds of blocks."""
import numpy as np
import pytest

import helpers as H
from test_gpu_ops import _dot_case, ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg_id", [4, 5, 6, 7])
@pytest.mark.parametrize("R,K,N", [(128, 1024, 256), (250, 1152, 256), (200, 2048, 144), (129, 640, 16), (256, 512, 80), (130, 128, 496)])
def test_forced_tile(ctx, cfg_id, R, K, N):
  eng = ctx["eng"]
  H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"ring_cfg", cfg_id))
  try:
    rng = np.random.default_rng(R + K + N + cfg_id)
    _dot_case(ctx, H.rand_bf16(rng, (R, K)), H.rand_bf16(rng, (K, N), 0.05))
  finally:
    H.lib.check(eng.lib.ixt_set_option(eng._ctx, b"ring_cfg", 0))


@pytest.mark.parametrize("R,K,N", [(128, 512, 400), (129, 640, 496), (250, 384, 256), (145, 256, 432)])
def test_chosen_tile(ctx, R, K, N):
  rng = np.random.default_rng(R + K + N)
  _dot_case(ctx, H.rand_bf16(rng, (R, K)), H.rand_bf16(rng, (K, N), 0.05))
