"""The gates of the ring products, whose weights come from tables in LDS (csrc/ixt_device.h, ixt_gate_at; csrc/ixt_kernels.h, k_gate_tables), over the tables' whole range and past both of its
ends, inside a model, against the oracle's bits."""
import numpy as np
import pytest

import helpers as H
from test_gpu_engine import run_pair

pytestmark = pytest.mark.gpu


def scaled(bits, exponents, axis):
  shape = [1, 1]
  shape[axis] = -1
  f = H.synth.bf16_bits_to_f32(bits).astype(np.float32) * np.exp2(exponents).astype(np.float32).reshape(shape)
  return H.synth.f32_to_bf16_bits(f)


@pytest.mark.parametrize("model,tile", [("ixt-tiny", 0), ("ixt-tiny", 1), ("ixt-tiny", 2), ("ixt-tiny", 4), ("ixt-tiny", 5), ("ixt-tiny", 7), ("gemma2-tiny", 0), ("gemma2-tiny", 2), ("gemma2-tiny", 4)])
def test_gates_from_the_tables_in_a_model(model, tile):
  """Column f of the gate's kernel is scaled by 2^-16 .. 2^9, row f of the down kernel by its inverse: arguments of both signs from below 2^-10 to beyond 2^7, each of whose gates counts as much as the
  others.  silu (llama2 blocks) and Gemma's gelu, every tile that the units' product has, 150 rows in one pass.  Tokens, logits, keys and values bit for bit."""
  cfg = H.make_config(model, max_prefill_predict_length=160, max_target_length=192, per_device_batch_size=1.0, base_mlp_dim=640)
  w = H.synth.synth_weights(cfg, 5)
  e = np.arange(640) % 26 - 16
  names = [n for n in w if "/mlp" in n and n.endswith("wi_0/kernel")]
  assert names
  for n in names:
    w[n] = scaled(w[n], e, 1)
    down = n.replace("wi_0/kernel", "wo/kernel")
    w[down] = scaled(w[down], -e, 0)
  toks, _ = H.synth.synth_prompt(cfg.vocab_size, 160, 70)
  run_pair(cfg, w, [(toks, 150)], steps=2, options={"ring_cfg": tile})
