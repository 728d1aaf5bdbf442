"""The f32 product on the matrix units (k_dot32): a prompt of so many rows in one step of a float32 hybrid decoder against the restatement, and the same prompt
in portions that take other forms of it.  The first test has its row blocks (16, 32, 64; 65 and more: several) over one chain of 512 k, the second its
chains: added in the wave or left as slices, a short last one, one column tile a wave or two."""
import numpy as np
import pytest

import vilepel_helpers as VH
import vilepel_ref as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 32, 33, 64, 65, 100])
def test_row_blocks(tmp_path, rows):
  cfg = VH.mixed_model()
  w = VH.random_weights(cfg, 21)
  eng, _ = VH.engine(VH.write_model(tmp_path, cfg, w), rows=128, target=128)
  s = VH.scheduler(eng)
  t = VH.tokens(cfg, rows, 60 + rows)
  want = V.forward(cfg, w, t)
  for rid, cuts in enumerate(((rows,), (7, 16, 33))):
    VH.check(VH.run_portions(s, rid, t, cuts), want, "float32", (rows, cuts))
    s.release(rid)
  eng.close()


def test_chains(tmp_path):
  """Widths 1160 (K 1280: two and a half chains) and 5504 (ten and three quarters).  The gate's 11008 columns: 129 rows take two column tiles a wave, 65 one,
  both with the chains added in the wave (the workspace holds one slice of 129 rows); 33, 20 and 5 rows leave a slice a chain.  The sums are the same whatever
  the form, and nothing else in the layer looks at the number of rows: every cut has the same bits."""
  cfg = VH.model([VH.with_mlp(VH.latent(), VH.dense(ff=5504))], width=1160)
  w = VH.random_weights(cfg, 5)
  eng, _ = VH.engine(VH.write_model(tmp_path, cfg, w), rows=129, target=136, pages=80)
  s = VH.scheduler(eng)
  t = VH.tokens(cfg, 129, 8)
  want, whole = V.forward(cfg, w, t), None
  for rid, cuts in enumerate(((129,), (65, 64), (33,), (20, 5))):
    got = VH.run_portions(s, rid, t, cuts)
    VH.check(got, want, "float32", cuts)
    whole = got if whole is None else whole
    assert np.array_equal(got.view(np.uint32), whole.view(np.uint32)), cuts
    s.release(rid)
  eng.close()


@pytest.mark.parametrize("rows", [3, 64, 65])
def test_chains_of_experts(tmp_path, rows):
  """Routed units of 1300 features (K 1408: three slices of the experts' down product), few rows and more than 64 (the slices are summed in front of the norm
  up to there, and by it beyond)."""
  cfg = VH.model([VH.with_mlp(VH.latent(), VH.moe(ff=1300, experts=5, top=2))], width=520)
  w = VH.random_weights(cfg, 6)
  eng, _ = VH.engine(VH.write_model(tmp_path, cfg, w), rows=96, target=96)
  s = VH.scheduler(eng)
  t = VH.tokens(cfg, rows, 9)
  VH.check(VH.run_portions(s, 0, t, (rows,)), V.forward(cfg, w, t), "float32", rows)
  eng.close()
