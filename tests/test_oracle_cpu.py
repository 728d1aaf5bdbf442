"""CPU suite: the oracle against its committed golden vectors and against the invariants the reference's own tests
state for this path; host logic; and the C-ABI export check (no GPU compute)."""
import ctypes
import hashlib
import os
import re
import subprocess

import numpy as np
import pytest

import helpers as H
from oracle import oracle as O


@pytest.fixture(scope="module")
def tiny():
  cfg = H.make_config(per_device_batch_size=2.0)
  w = H.synth.synth_weights(cfg, 0)
  return cfg, w


def _decode(orc, prompts, steps):
  pres, firsts = [], []
  for s, (t, tl) in enumerate(prompts):
    p, r = orc.prefill(t, tl, slot=s)
    pres.append(p)
    firsts.append(int(r[0, 0]))
  ds = orc.init_decode_state()
  for s in range(len(prompts)):
    ds = orc.insert(pres[s], ds, s)
  out = [firsts + [0] * (orc.cfg.max_slots - len(firsts))]
  for _ in range(steps):
    ds, r = orc.generate(ds)
    out.append(r[:, 0].tolist())
  return np.array(out, np.int32)


def test_golden_tiny(tiny):
  cfg, w = tiny
  g = np.load(os.path.join(H.GOLDEN, "tiny_decode.npz"))
  prompts = [(g["prompt_tokens"][i], int(g["true_lengths"][i])) for i in range(2)]
  got = _decode(H.make_oracle(cfg, w), prompts, int(g["steps"]))
  assert np.array_equal(got, g["tokens"])


def test_golden_c1():
  g = np.load(os.path.join(H.GOLDEN, "c1_decode.npz"))
  cfg = H.make_config(model_name="c1-134m", per_device_batch_size=1.0, max_prefill_predict_length=64, max_target_length=128,
                      pagedattn_tokens_per_page=32, pagedattn_num_pages=8)
  w = H.synth.synth_weights(cfg, int(g["weight_seed"]))
  got = _decode(H.make_oracle(cfg, w), [(g["prompt_tokens"][0], int(g["true_lengths"][0]))], 16)
  assert np.array_equal(got, g["tokens"][:17])


def test_chunked_equals_unchunked_exact(tiny):
  """tests/maxengine_test.py:166-300: cache and first token equal between unchunked / 1 chunk / 2 chunks (exact)."""
  cfg, w = tiny
  toks, tl = H.synth.synth_prompt(cfg.vocab_size, 32, 7)
  a = H.make_oracle(cfg, w)
  pa, ra = a.prefill(toks, tl, slot=0, want_logits=True)
  b = H.make_oracle(cfg, w)
  n1 = 11
  b.prefill(toks[:n1], n1, slot=0)
  rest = np.zeros(32, np.int32)
  rest[:tl - n1] = toks[n1:tl]
  pb, rb = b.prefill(rest, tl - n1, slot=0, existing_prefix_tokens=toks[:n1], want_logits=True)
  assert np.array_equal(ra, rb)
  assert np.array_equal(pa["logits"].view(np.uint32), pb["logits"].view(np.uint32))
  for layer in range(cfg.num_decoder_layers):
    ka, va = a.model.gather_kv(layer, a.page_state.page_map[0], tl)
    kb, vb = b.model.gather_kv(layer, b.page_state.page_map[0], tl)
    assert np.array_equal(ka, kb) and np.array_equal(va, vb)
  for f in a.page_state.__dataclass_fields__:
    assert np.array_equal(getattr(a.page_state, f), getattr(b.page_state, f))


def test_prefill_plus_autoregress_equals_longer_prefill(tiny):
  """tests/model_test.py:115-191 / tests/attention_test.py:361-406 (there with tolerances): here the teacher-forced
  autoregressive logits equal the longer prefill's last-row logits bit for bit."""
  cfg, w = tiny
  toks, tl = H.synth.synth_prompt(cfg.vocab_size, 32, 9)
  tl = 20
  a = H.make_oracle(cfg, w)
  pa, ra = a.prefill(toks, tl, slot=0)
  ds = a.insert(pa, a.init_decode_state(), 0)
  seq = list(toks[:tl])
  for step in range(5):
    seq.append(int(ds["tokens"][0, 0]))
    ds, r = a.generate(ds, want_logits=True)
    b = H.make_oracle(cfg, w)
    buf = np.zeros(32, np.int32)
    buf[:len(seq)] = seq
    pb, rb = b.prefill(buf, len(seq), slot=0, want_logits=True)
    assert np.array_equal(ds["logits"][0].view(np.uint32), pb["logits"][0].view(np.uint32)), step
    assert int(r[0, 0]) == int(rb[0, 0])


def test_batch_rows_are_independent(tiny):
  """A slot's tokens do not depend on what the other slots hold (decode_batch rows are independent units)."""
  cfg, w = tiny
  p0 = H.synth.synth_prompt(cfg.vocab_size, 32, 21)
  p1 = H.synth.synth_prompt(cfg.vocab_size, 32, 22)
  both = _decode(H.make_oracle(cfg, w), [p0, p1], 12)
  solo = _decode(H.make_oracle(cfg, w), [p0], 12)
  assert np.array_equal(both[:, 0], solo[:, 0])


def test_mfma_model_matches_hardware_vectors():
  """The oracle's integer model of one v_mfma_f32_16x16x32_bf16 (orc_mfma_step8 x 4) against 16 000 input/output vectors
  recorded from the instruction itself on an MI355X (tools/mfma_dump.hip -> tests/golden/make_mfma_golden.py): gaussians,
  wide exponent spreads, cancellation, accumulators far above / below the products, zeros of both signs, bf16 subnormals."""
  from oracle import oracle as O
  g = np.load(os.path.join(H.GOLDEN, "mfma_step_hw.npz"))
  a, b = np.ascontiguousarray(g["a"]), np.ascontiguousarray(g["b"])
  c = np.ascontiguousarray(g["c"]).view(np.float32)
  out = np.zeros(c.shape, np.float32)
  O.lib().orc_mfma_cases(O._p(a, O._u16p), O._p(b, O._u16p), O._p(c, O._f32p), O._p(out, O._f32p), len(c))
  bad = np.flatnonzero(out.view(np.uint32) != g["d"])
  assert len(c) == 16000 and bad.size == 0, bad[:8]


@pytest.mark.parametrize("R,K,N,spread,zf", [(3, 128, 40, 0, 0.0), (5, 640, 136, 3, 0.0), (4, 1024, 264, 12, 0.3), (2, 2048, 520, 40, 0.1), (17, 512, 128, 1, 0.0)])
def test_vector_dot_equals_definition(R, K, N, spread, zf):
  """orc_dot_rows (AVX2: int32 lanes + exact double arithmetic) against the definition (orc_mfma_step8 chained, scalar)."""
  from oracle import oracle as O
  rng = np.random.default_rng(K + N)
  x = rng.standard_normal((R, K)) * np.exp2(rng.integers(-spread, spread + 1, (R, K)))
  w = rng.standard_normal((K, N)) * np.exp2(rng.integers(-spread, spread + 1, (K, N)))
  x[rng.random((R, K)) < zf] = 0
  w[rng.random((K, N)) < zf] = 0
  xb, wb = O.f32_to_bf16(x.astype(np.float32)), O.f32_to_bf16(w.astype(np.float32))
  o1, o2 = np.zeros((R, N), np.float32), np.zeros((R, N), np.float32)
  O.lib().orc_dot_rows(O._p(xb, O._u16p), K, R, O._p(wb, O._u16p), K, N, O._p(o1, O._f32p), N)
  O.lib().orc_dot_rows_scalar(O._p(xb, O._u16p), K, R, O._p(wb, O._u16p), K, N, O._p(o2, O._f32p), N)
  assert np.array_equal(o1.view(np.uint32), o2.view(np.uint32))
  ref = O.bf16_to_f32(xb).astype(np.float64) @ O.bf16_to_f32(wb).astype(np.float64)
  scale = (np.abs(O.bf16_to_f32(xb).astype(np.float64)) @ np.abs(O.bf16_to_f32(wb).astype(np.float64)))
  assert (np.abs(o1 - ref) <= 1e-6 * scale + 1e-30).all()     # the truncating adder stays within ~2^-20 of the exact dot


def test_rope_against_complex_reference():
  """tests/llama_test.py:79-103: RotaryEmbedding vs complex multiply under the half-split layout (rtol 1e-1, atol 1e-4)."""
  hd, T = 128, 64
  sn, cs = O.rope_tables(hd, T)
  rng = np.random.default_rng(0)
  x = rng.standard_normal((4, hd)).astype(np.float32)
  xb = O.f32_to_bf16(x)
  for pos in (0, 1, 17, 63):
    v = xb.copy()
    O.lib().orc_rope(O._p(v, O._u16p), 4, hd, O._p(sn[pos], O._u16p), O._p(cs[pos], O._u16p))
    got = O.bf16_to_f32(v).reshape(4, hd)
    xf = O.bf16_to_f32(xb).reshape(4, hd).astype(np.float64)
    half = hd // 2
    freq = 1.0 / (10000.0 ** (2 * np.arange(half) / hd))
    z = (xf[:, :half] + 1j * xf[:, half:]) * np.exp(1j * pos * freq)
    ref = np.concatenate([z.real, z.imag], axis=-1)
    np.testing.assert_allclose(got, ref, rtol=1e-1, atol=5e-2)


def test_bf16_rounding_matches_torch():
  import torch
  rng = np.random.default_rng(1)
  x = np.concatenate([rng.standard_normal(100000).astype(np.float32) * 10.0 ** rng.integers(-20, 20, 100000),
                      np.array([0.0, -0.0, 1.0, 1.00390625, 1.01171875, np.inf, -np.inf, 3.3895314e38], np.float32)]).astype(np.float32)
  ours = O.f32_to_bf16(x)
  ref = torch.from_numpy(x).to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)
  assert np.array_equal(ours, ref)
  assert np.array_equal(H.synth.f32_to_bf16_bits(x), ref)
  out = np.zeros_like(ours)
  O.lib().orc_f32_to_bf16(O._p(x, O._f32p), O._p(out, O._u16p), x.size)
  assert np.array_equal(out, ref)


def test_exp_accuracy():
  x = np.linspace(-85.0, 85.0, 200001).astype(np.float32)
  y = np.zeros_like(x)
  O.lib().orc_exp_vec(O._p(x, O._f32p), O._p(y, O._f32p), x.size)
  ref = np.exp(np.clip(x.astype(np.float64), -80.0, 80.0))
  rel = np.abs(y.astype(np.float64) - ref) / ref
  assert rel.max() < 2.5e-7  # ~2 ulp; the clamp to [-80, 80] is part of the canonical definition
  assert np.all(np.isfinite(y)) and np.all(y > 0)


def test_audio_mapping_table():
  """extend_tokenizer.py:29-46 as realised in audio_token_mapping_adjusted.json (fixture made by make_golden.py)."""
  g = np.load(os.path.join(H.GOLDEN, "audio_token_mapping_adjusted.npz"))
  assert str(g["sha256"]).startswith("06712843")
  a2e = g["audio_to_embedding"]
  assert a2e.shape == (8192,) and np.all(a2e >= 0)
  ours = np.array([O.audio_id_to_embedding_row(a) for a in range(8192)], np.int32)
  assert np.array_equal(ours, a2e)
  assert np.array_equal(H.synth.audio_id_to_row(np.arange(8192)), a2e)
  rows, aud = g["embedding_rows"], g["embedding_audio_id"]
  assert rows.shape == (8290,) and rows.max() == 264191 and int(np.sum(aud == -1)) == 98
  assert np.array_equal(rows[aud >= 0][np.argsort(aud[aud >= 0])], a2e)
  assert np.array_equal(rows[aud == -1], np.arange(264094, 264192))  # pad rows


def test_abi_exports_every_declared_symbol():
  """libixt.so must export exactly the entry points include/ixt.h declares (no compute calls here)."""
  hdr = open(os.path.join(H.ROOT, "include", "ixt.h")).read()
  declared = set(re.findall(r"\b(ixt_[a-z0-9_]+)\s*\(", hdr))
  assert declared == set(H.lib.SIGNATURES), declared ^ set(H.lib.SIGNATURES)
  H.importlib.import_module("maxtext-indextts2_amd.build").build()
  lib = H.lib.load()
  for name in declared:
    assert hasattr(lib, name), name
  assert lib.ixt_last_error() is not None
  # argument checking that needs no GPU
  assert lib.ixt_create(None, None) == H.lib.IXT_ERR_INVALID
  with pytest.raises(ValueError):
    H.lib.check(lib.ixt_create(None, None))
  # the training-step ABI (include/ixt_train.h) lives in the same library
  thdr = open(os.path.join(H.ROOT, "include", "ixt_train.h")).read()
  tdeclared = set(re.findall(r"\b(ixt_train_[a-z0-9_]+)\s*\(", thdr))
  assert len(tdeclared) >= 10
  for name in tdeclared:
    assert hasattr(lib, name), name
  assert lib.ixt_train_create(None, None) == H.lib.IXT_ERR_INVALID


def test_product_has_no_cpu_fallback_and_no_oracle_import():
  """The product package must never reach into oracle/ and must fail loudly without a GPU."""
  pkg = os.path.join(H.ROOT, "maxtext-indextts2_amd")
  bad = re.compile(r"(from|import)\s+oracle|oracle[./\\]|libixt_oracle|ixt_oracle")
  for dp, _, files in os.walk(pkg):
    for f in files:
      if f.endswith((".py", ".hip", ".h", ".cpp")):
        src = open(os.path.join(dp, f), errors="ignore").read()
        assert not bad.search(src), (dp, f)
  import torch
  if not torch.cuda.is_available():
    maxengine = H.importlib.import_module("maxtext-indextts2_amd.maxengine")
    with pytest.raises(H.lib.IxtError):
      maxengine.MaxEngine(H.make_config())


def test_pyconfig_surface(monkeypatch):
  pc = H.pyconfig
  c = pc.initialize(["x", H.BASE_YML, "model_name=indextts2-1b", "per_device_batch_size=8", "attention=paged", "max_target_length=1280"])
  assert (c.emb_dim, c.num_query_heads, c.num_kv_heads, c.head_dim, c.mlp_dim, c.num_decoder_layers, c.vocab_size) == (2048, 16, 16, 128, 7168, 16, 264192)
  assert c.global_batch_size_to_load == 8 and c.pagedattn_max_pages_per_group == 40 and c.attn_logits_soft_cap is None
  with pytest.raises(ValueError):  # pyconfig.py:437-439
    pc.initialize(["x", H.BASE_YML, "no_such_key=1"])
  with pytest.raises(ValueError):  # read-only, pyconfig.py:1163-1164
    c.vocab_size = 3
  monkeypatch.setenv("M_VOCAB_SIZE", "4096")
  assert pc.initialize(["x", H.BASE_YML]).vocab_size == 4096
  with pytest.raises(ValueError):  # CLI + env conflict, pyconfig.py:441-443
    pc.initialize(["x", H.BASE_YML, "vocab_size=5"])
  monkeypatch.delenv("M_VOCAB_SIZE")
  # example_audio_training.py:54-79 override list is accepted
  c2 = pc.initialize(["x", H.BASE_YML, "dataset_type=emilia_audio", "audio_token_mapping_path=vocab_expansion/audio_token_mapping_adjusted.json",
                      "audio_batch_size=4", "emilia_language=EN", "base_emb_dim=2048", "vocab_size=264191", "global_batch_size_to_load=4",
                      "max_target_length=2048", "steps=10", "learning_rate=1e-4", "per_device_batch_size=4"])
  assert c2.dataset_type == "emilia_audio" and c2.global_batch_size_to_load == 4 and c2.learning_rate == 1e-4
  assert pc.get_individual_scales(8) == (1, 1, 1, 1) and pc.get_individual_scales(2) == (0, 1, 1, 0)


def test_synth_prompt_contract():
  toks, tl = H.synth.synth_prompt(264192, 256, 1234)
  assert toks.shape == (256,) and 248 <= tl <= 256 and toks[0] == 264094 and toks[47] == 264095
  audio = toks[48:tl]
  assert np.all(((audio >= 6) & (audio <= 104)) | ((audio >= 256001) & (audio <= 264093)))
  assert np.all(toks[tl:] == 0)


def test_log_and_logprob_restatement():
  """orc_log (the device's ixt_log: IEEE-only operations) against libm, and log_prob_of_chosen_token (inference_utils.py:56-63) in the
  canonical order against a float64 log_softmax."""
  rng = np.random.default_rng(3)
  x = np.concatenate([np.exp(rng.uniform(-20, 20, 20000)), [1.0, 2.0, 0.5, 1.41421354, 1.4142137, 264192.0, 1e-30, 3e38]]).astype(np.float32)
  got = np.zeros_like(x)
  O.lib().orc_log_vec(O._p(x, O._f32p), O._p(got, O._f32p), x.size)
  ref = np.log(x.astype(np.float64))
  assert np.max(np.abs(got - ref) / np.maximum(1.0, np.abs(ref))) < 2.5e-7
  V = 5000
  lg = O.bf16_to_f32(O.f32_to_bf16(rng.normal(0, 4, (7, V)).astype(np.float32))).reshape(7, V)
  ch = rng.integers(0, V, 7).astype(np.int32)
  lp = O.logprob_rows(lg, ch)
  l64 = lg.astype(np.float64)
  ref = l64[np.arange(7), ch] - (l64.max(1) + np.log(np.exp(l64 - l64.max(1, keepdims=True)).sum(1)))
  assert np.max(np.abs(lp - ref)) < 2e-5
  assert np.all(lp <= 0.0)
