"""The f32 product on the matrix units at the edges of its row blocks (16, 32, 64; 65 and more: several) and of its chains of 512 k: a prompt of that many rows in
one step of a float32 hybrid decoder against the restatement, and the same prompt in portions that take other row blocks."""
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
