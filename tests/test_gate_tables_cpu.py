"""The gates of the units' ring products come from tables of 2 x 2177 weights (csrc/ixt_device.h, ixt_gate_at): bf16(a w(a)) with w(a) taken where |a| is clamped to
2^-10 .. 2^7.  Every bf16 value of a, infinities included, against the oracle's gate: the clamp takes nothing away.  Bits are compared, there is no tolerance."""
import os
import re

import numpy as np
import pytest

import helpers as H
from oracle import oracle as O


def constant(name):
  with open(os.path.join(H.importlib.import_module("maxtext-indextts2_amd.build").CSRC, "ixt_device.h"), encoding="utf-8") as f:
    return eval(re.search(rf"#define {name} (.*?)(//|\n)", f.read()).group(1), {"__builtins__": {}})


LO, N = constant("IXT_GATE_LO"), constant("IXT_GATE_N")
f32 = np.float32


def rbf(x):
  return O.bf16_to_f32(O.f32_to_bf16(x))


def of(fn, x):
  x = np.ascontiguousarray(x, f32)
  out = np.empty_like(x)
  getattr(O.lib(), fn)(O._p(x, O._f32p), O._p(out, O._f32p), x.size)
  return out


def sigmoid(a):
  return rbf(f32(1) / (f32(1) + of("orc_exp_vec", -a)))


def cdf(a):
  u = rbf(a + rbf(f32(0.044677734375) * rbf(rbf(a * a) * a)))
  return rbf(f32(0.5) * rbf(f32(1) + rbf(of("orc_tanh_vec", rbf(f32(0.796875) * u)))))


@pytest.mark.parametrize("weight,gate", [(sigmoid, "orc_swiglu"), (cdf, "orc_geglu")])
def test_table_gives_the_oracles_gate(weight, gate):
  bits = np.arange(65536, dtype=np.uint16)
  bits = bits[(bits & 0x7fff) <= 0x7f80]               # no NaN
  a = O.bf16_to_f32(bits)
  entry = np.arange(2 * N)
  with np.errstate(all="ignore"):
    table = weight(O.bf16_to_f32((entry % N + LO | entry // N << 15).astype(np.uint16)))
    at = np.clip((bits & 0x7fff).astype(np.int64), LO, LO + N - 1) - LO + (bits >> 15).astype(np.int64) * N
    for b in (0x3f80, 0xbfdb):
      b = np.full(bits.size, b, np.uint16)
      ref = np.empty(bits.size, np.uint16)
      getattr(O.lib(), gate)(O._p(bits, O._u16p), O._p(b, O._u16p), O._p(ref, O._u16p), bits.size)
      got = rbf(a * table[at]) * O.bf16_to_f32(b)
      same = np.where(np.isnan(got), np.isnan(O.bf16_to_f32(ref)), O.f32_to_bf16(got) == ref)
      assert same.all(), (gate, a[~same][:8])
