"""The calls this framework is timed by: what a user of it has it do, through its public entry points, over the sizes that its model files, its tests
and its benchmarks use.

  decode      `MaxEngine.insert` of prefilled prompts, then `generate` steps: token generation, from one utterance to a full batch
  prefill     `MaxEngine.prefill` of one prompt (in chunks where it is long), or `prefill_concat` of several prompts in one pass
  utterances  whole utterances through a hybrid decoder: `prefill_concat`, `insert_partial`, `generate`, `release_pages`
  train       `Trainer.train_step`: forward, backward, clipping and AdamW

`exact` restates the models in 64-bit torch.  Weights and inputs are functions of (case, seed), drawn on the device."""
import importlib
import json
import math
import os
import tempfile

import numpy as np
import torch

PAGE = 32
# the model files' sizes (Mixtral with the first layers only: all 32 are 93 GB)
SIZES = {
    "c1-134m": dict(block="llama2", E=768, H=12, KV=12, D=64, F=2048, L=12, V=32000),
    "indextts2-1b": dict(block="llama2", E=2048, H=16, KV=16, D=128, F=7168, L=16, V=264192),
    "gemma2-2b": dict(block="gemma2", E=2304, H=8, KV=4, D=256, F=9216, L=13, V=256128, eps=1e-6),
    "mixtral-8x7b": dict(block="mixtral", E=4096, H=32, KV=8, D=128, F=14336, L=4, V=32000, NE=8, K=2, theta=1e6),
}
# hybrid decoders as the benchmark has them: (width, heads, feed-forward, latent rank, head dims of latent layers, window), eight layers
HYBRID = {"w1024": (1024, 8, 3584, 256, 64, 512), "w2048": (2048, 16, 7168, 512, 128, 1024)}
HYBRID_LAYERS, HYBRID_VOCAB = 8, 32000


def listed():
  return [
      # one utterance: the latency of a token in an interactive session
      {"name": "decode-1", "kind": "decode", "model": "indextts2-1b", "slots": 1, "context": 300, "steps": 32, "quantization": ""},
      # a few utterances at a time
      {"name": "decode-8", "kind": "decode", "model": "indextts2-1b", "slots": 8, "context": 500, "steps": 32, "quantization": ""},
      # a server under ordinary load: neither a few rows nor a full batch
      {"name": "decode-48", "kind": "decode", "model": "indextts2-1b", "slots": 48, "context": 600, "steps": 32, "quantization": ""},
      # the benchmark's full batch in the middle of its utterances
      {"name": "decode-256", "kind": "decode", "model": "indextts2-1b", "slots": 256, "context": 700, "steps": 64, "quantization": ""},
      # routed experts, eight utterances
      {"name": "decode-routed", "kind": "decode", "model": "mixtral-8x7b", "slots": 8, "context": 256, "steps": 32, "quantization": ""},
      # a short text prompt: the time to the first token of an utterance
      {"name": "prefill-short", "kind": "prefill", "model": "indextts2-1b", "prompts": 1, "length": 57, "chunk": 256, "quantization": ""},
      # the benchmark's packed prefill: eight prompts with text and a speaker's audio tokens
      {"name": "prefill-packed", "kind": "prefill", "model": "indextts2-1b", "prompts": 8, "length": 251, "chunk": 256, "quantization": ""},
      # a long conversation or book passage, in the benchmark's larger chunks
      {"name": "prefill-long", "kind": "prefill", "model": "indextts2-1b", "prompts": 1, "length": 3900, "chunk": 1024, "quantization": ""},
      # the fork's other base model family, a long prompt in chunks of the default size
      {"name": "prefill-capped", "kind": "prefill", "model": "gemma2-2b", "prompts": 1, "length": 3000, "chunk": 256, "quantization": ""},
      # a hybrid decoder (latent attention and gated delta rule): eight utterances from prompt to tokens
      {"name": "utterances-hybrid", "kind": "utterances", "model": "vilepel", "size": "w2048", "prompts": 8, "length": 250, "steps": 32, "dtype": "bfloat16"},
      # training steps: the plumbing model on a small batch, and the benchmark's share of one GPU
      {"name": "train-small", "kind": "train", "model": "c1-134m", "batch": 4, "length": 512},
      {"name": "train-1b", "kind": "train", "model": "indextts2-1b", "batch": 8, "length": 2048},
  ]


def _log_int(rng, lo, hi):
  return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
  kind = rng.choice(["decode", "decode", "prefill", "prefill", "utterances", "train"])
  if kind == "decode":
    model = rng.choice(["indextts2-1b", "indextts2-1b", "indextts2-1b", "c1-134m", "mixtral-8x7b"])
    slots = _log_int(rng, 1, 32 if model == "mixtral-8x7b" else 256)
    return {"kind": kind, "model": model, "slots": slots, "context": _log_int(rng, 16, 1000 if slots <= 128 else 700), "steps": 32,
            "quantization": rng.choice(["", "", "fp8"]) if model == "mixtral-8x7b" else ""}
  if kind == "prefill":
    model = rng.choice(["indextts2-1b", "indextts2-1b", "c1-134m", "gemma2-2b", "mixtral-8x7b"])
    if rng.random() < 0.5:
      return {"kind": kind, "model": model, "prompts": rng.randint(2, 8), "length": _log_int(rng, 8, 256), "chunk": 256, "quantization": ""}
    chunk = rng.choice([256, 1024])
    return {"kind": kind, "model": model, "prompts": 1, "length": _log_int(rng, 1, 3000 if model in ("gemma2-2b", "mixtral-8x7b") else 3900), "chunk": chunk,
            "quantization": rng.choice(["", "", "fp8"]) if model in ("gemma2-2b", "mixtral-8x7b") else ""}
  if kind == "utterances":
    return {"kind": kind, "model": rng.choice(["vilepel", "vazilorn"]), "size": rng.choice(sorted(HYBRID)), "prompts": rng.randint(1, 8), "length": _log_int(rng, 8, 512),
            "steps": rng.randint(8, 32), "dtype": rng.choice(["bfloat16", "bfloat16", "bfloat16", "float32"])}
  model = rng.choice(["c1-134m", "c1-134m", "indextts2-1b"])
  return {"kind": kind, "model": model, "batch": rng.randint(1, 8), "length": 8 * _log_int(rng, 16, 256)}


# ------------------------------------------------------------------------------------------------------------------------------ weights and inputs
def _specs(case):
  """[(tensor name, shape, mean, deviation)] of the case's model."""
  if case["kind"] == "utterances":
    return _hybrid_specs(case)
  s = SIZES[case["model"]]
  E, H, KV, D, F, V, out = s["E"], s["H"], s["KV"], s["D"], s["F"], s["V"], []
  dense = lambda name, shape, fan_in: out.append((name, shape, 0.0, fan_in ** -0.5))
  scale = lambda name: out.append((name, (E,), 1.0, 0.1))
  out.append(("params/token_embedder/embedding", (V, E), 0.0, 1.0))
  for i in range(s["L"]):
    p = f"params/decoder/layers_{i}/"
    for sub in ("_local", "_global") if s["block"] == "gemma2" else ("",):
      gemma = s["block"] == "gemma2"
      scale(p + ("pre_self_attention_norm" + sub if gemma else "pre_self_attention_layer_norm") + "/scale")
      a = p + "self_attention" + sub + "/"
      dense(a + "query/kernel", (E, H, D), E * D)          # 1 / sqrt(head size) is part of the query kernel
      dense(a + "key/kernel", (E, KV, D), E)
      dense(a + "value/kernel", (E, KV, D), E)
      dense(a + "out/kernel", (H, D, E), H * D)
      if gemma:
        scale(p + "post_self_attention_norm" + sub + "/scale")
        scale(p + ("mlp_local/mlp_layer_norm/scale" if sub == "_local" else "pre_ffw_norm_global/scale"))
      else:
        scale(p + ("post_self_attention_layer_norm/scale" if s["block"] == "mixtral" else "mlp/mlp_layer_norm/scale"))
      if s["block"] == "mixtral":
        m = p + "MoeBlock_0/"
        dense(m + "gate/kernel", (E, s["NE"]), E / 16)       # wider than the others: tokens differ in their experts
        dense(m + "wi_0", (s["NE"], E, F), E)
        dense(m + "wi_1", (s["NE"], E, F), E)
        dense(m + "wo", (s["NE"], F, E), F)
      else:
        m = p + "mlp" + sub + "/"
        dense(m + "wi_0/kernel", (E, F), E)
        dense(m + "wi_1/kernel", (E, F), E)
        dense(m + "wo/kernel", (F, E), F)
      if gemma:
        scale(p + "post_ffw_norm" + sub + "/scale")
  scale("params/decoder/decoder_norm/scale")
  if s["block"] != "gemma2":
    dense("params/decoder/logits_dense/kernel", (E, V), E)
  return out


def _hybrid_specs(case):
  E, H, F, rank, dim, _ = HYBRID[case["size"]]
  rot, vd, out = 64, 128, []
  lin = lambda name, n, m, f=1.0: out.append((name, (n, m), 0.0, f * m ** -0.5))
  vec = lambda name, n, mean, dev: out.append((name, n, mean, dev))
  vilepel = case["model"] == "vilepel"

  def norm(name, alpha):
    vec(name, (E,), 0.0 if vilepel else 1.0, 0.1)
    if not vilepel:
      vec(name + ".b", (E,), 0.0, 0.1)
      vec(name + ".alpha", (), alpha, 0.0)

  vec("embed", (HYBRID_VOCAB, E), 0.0, 2.0)
  lin("head", HYBRID_VOCAB, E)
  norm("final.norm", 0.6)
  for i in range(HYBRID_LAYERS):
    p, m = f"l{i}.", f"l{i}.mix."
    norm(p + "norm1", 0.6)
    norm(p + "norm2", 0.6)
    if not vilepel:
      norm(p + "norm1b", 1.5)
      norm(p + "norm2b", 1.5)
      for n in ("q", "k", "v"):
        lin(m + n, H * 128, E)
      vec(m + "q.norm", (128,), 1.0, 0.1)
      vec(m + "k.norm", (128,), 1.0, 0.1)
      vec(m + "sink", (H,), 1.0, 0.5)
    elif i % 2 == 0:
      for n in ("q", "k", "v"):
        lin(m + n, H * 128, E)
        vec(m + n + ".conv", (H * 128, 4), 0.0, 0.5)
      lin(m + "b", H, E)
      vec(m + "A_log", (H,), -1.0, 0.5)
      vec(m + "norm", (128,), 1.0, 0.1)
      vec(m + "dt_bias", (H * 128,), -1.0, 0.5)
      for n in ("a", "g"):
        lin(m + n + "1", 128, E)
        lin(m + n + "2", H * 128, 128)
    else:
      lin(m + "q", H * (dim + rot), E)
      lin(m + "dkv", rank + rot, E)
      vec(m + "dkv.norm", (rank,), 1.0, 0.1)
      lin(m + "uk", H * dim, rank)
      lin(m + "uv", H * vd, rank)
    lin(m + "o", E, H * vd)
    lin(p + "mlp.gate", F, E, 0.6)
    lin(p + "mlp.up", F, E, 0.6)
    lin(p + "mlp.down", E, F)
  return out


def _hybrid_config(case):
  E, H, F, rank, dim, window = HYBRID[case["size"]]
  layers = []
  for i in range(HYBRID_LAYERS):
    if case["model"] == "vazilorn":
      mixer = {"heads": H, "kv_heads": H, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": window},
               "rot": {"base": 500000.0, "dims": 128, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
      layers.append({"type": "attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": F}})
    elif i % 2 == 0:
      layers.append({"type": "channel_delta", "mixer": {"heads": H, "kv_heads": H, "dim": 128, "vdim": 128, "conv": 4}, "mlp": {"kind": "dense", "ff": F, "limit": 7.0}})
    else:
      mixer = {"heads": H, "dim": dim, "rot_dim": 64, "vdim": 128, "kv_rank": rank, "scale": (dim + 64) ** -0.5, "mask": {"size": window}, "rot": {"base": 10000.0, "dims": 64}}
      layers.append({"type": "latent_attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": F, "limit": 7.0}})
  out = {"architecture": case["model"].capitalize(), "norm": {"eps": 1e-5}, "vocab": HYBRID_VOCAB, "width": E, "layers": layers}
  return dict(out, embedding={"scale": 1.0}) if case["model"] == "vilepel" else out


class _Tree:
  """{name: bf16 tensor} of a case's model, each tensor drawn when it is asked for."""

  def __init__(self, case, seed):
    self.specs = {n: (i, shape, mean, dev) for i, (n, shape, mean, dev) in enumerate(_specs(case))}
    self.seed, self.g = seed, torch.Generator(device="cuda")

  def __contains__(self, name):
    return name in self.specs

  def __getitem__(self, name):
    i, shape, mean, dev = self.specs[name]
    self.g.manual_seed((self.seed * 1009 + i) % (1 << 62))
    t = torch.empty(shape, dtype=torch.float32, device="cuda")
    return (t.normal_(mean, dev, generator=self.g) if dev else t.fill_(mean)).to(torch.bfloat16)

  def items(self):
    return ((n, self[n]) for n in self.specs)


def _lengths(case, rng):
  """Prompts of one call differ in length: the longest, and others down to half of it."""
  n = case["slots"] if case["kind"] == "decode" else case["prompts"]
  most = case["context"] if case["kind"] == "decode" else case["length"]
  return [most] + [int(v) for v in rng.integers(max(1, most // 2), most + 1, n - 1)]


def _prompts(case, seed):
  rng = np.random.default_rng(seed)
  V = HYBRID_VOCAB if case["kind"] == "utterances" else SIZES[case["model"]]["V"]
  return [rng.integers(1, V, n).astype(np.int32) for n in _lengths(case, rng)]


def _forced(case, seed):
  """The token every sequence continues with (a decoder that starts on a fixed marker); a hybrid pass scores a given continuation."""
  n = case["slots"] if case["kind"] == "decode" else case["prompts"]
  V = HYBRID_VOCAB if case["kind"] == "utterances" else SIZES[case["model"]]["V"]
  return np.random.default_rng(seed + 7919).integers(1, V, (1 if case["kind"] == "decode" else case["steps"], n)).astype(np.int32)


def _batch(case, seed):
  """Rows of audio codes behind a start marker: inputs and targets one apart, the tail of shorter rows padding."""
  rng = np.random.default_rng(seed)
  B, S, V = case["batch"], case["length"], SIZES[case["model"]]["V"]
  n = np.concatenate([[S + 1], rng.integers(S // 2, S + 2, B - 1)])[:B]
  real = (np.arange(S + 1)[None, :] < n[:, None]).astype(np.int32)
  tok = (rng.integers(1, V, (B, S + 1)) * real).astype(np.int32)
  pos = (np.arange(S + 1, dtype=np.int32)[None, :] * real).astype(np.int32)
  return {"inputs": tok[:, :-1].copy(), "inputs_position": pos[:, :-1].copy(), "inputs_segmentation": real[:, :-1].copy(), "targets": tok[:, 1:].copy(),
          "targets_position": pos[:, 1:].copy(), "targets_segmentation": real[:, :-1] * real[:, 1:]}


# ------------------------------------------------------------------------------------------------------------------------------ prepare and run
def _module(name):
  return importlib.import_module("maxtext-indextts2_amd." + name)


def _config(**keys):
  pyconfig = _module("pyconfig")
  return pyconfig.initialize(["cases", os.path.join(pyconfig.PKG_DIR, "configs", "base.yml")], scan_layers=False, run_name="cases", override_model_config=True, **keys)


def _model_keys(case):
  keys = {"model_name": case["model"]}
  if case["model"] == "mixtral-8x7b":
    keys["base_num_decoder_layers"] = SIZES[case["model"]]["L"]
  return keys


def _engine(case, seed, slots, longest, rows, groups, extra):
  """An engine with its weights, for `slots` sequences of at most `longest` tokens, `groups` prompts of `rows` rows in one packed pass."""
  pages = -(-longest // PAGE)
  keys = dict(attention="paged", per_device_batch_size=float(slots), max_prefill_predict_length=rows if groups == 0 else -(-rows // groups), max_target_length=longest,
              pagedattn_tokens_per_page=PAGE, pagedattn_num_pages=(slots + groups) * pages + 1, use_chunked_prefill=True, ixt_staging_groups=groups,
              ixt_max_packed_rows=rows if groups else 0, **extra)
  if case["kind"] == "utterances":
    with tempfile.TemporaryDirectory() as d:
      with open(os.path.join(d, "config.json"), "w", encoding="utf-8") as f:
        json.dump(_hybrid_config(case), f)
      cfg = _config(ixt_model_dir=d, dtype=case["dtype"], **keys)
  else:
    cfg = _config(quantization=case["quantization"], **_model_keys(case), **keys)
  engine = _module("maxengine").MaxEngine(cfg)
  return engine, engine.load_params(params=_Tree(case, seed))


def _packed(prompts):
  lens = np.array([len(p) for p in prompts], np.int32)
  dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
  return {"padded_tokens": dev(np.concatenate(prompts)), "decoder_positions": dev(np.concatenate([np.arange(n) for n in lens])),
          "decoder_segment_ids": dev(np.concatenate([np.full(n, i + 1) for i, n in enumerate(lens)])),
          "start_pos": np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32), "true_lengths": lens, "num_prompts": len(prompts)}


def prepare(case, seed):
  kind = case["kind"]
  if kind == "train":
    cfg = _config(**_model_keys(case), per_device_batch_size=float(case["batch"]), max_target_length=case["length"], dataset_type="synthetic", warmup_steps_fraction=0.0)
    trainer = _module("train").Trainer(cfg)
    trainer.load_params(_Tree(case, seed))
    return {"case": case, "trainer": trainer, "batch": {k: torch.from_numpy(v).cuda() for k, v in _batch(case, seed).items()}}
  prompts = _prompts(case, seed)
  n, most = len(prompts), max(len(p) for p in prompts)
  if kind == "decode":
    engine, params = _engine(case, seed, n, most + case["steps"] + 1, most, 0, {})
    first = torch.from_numpy(_forced(case, seed)).cuda()
    prefixes = []
    for slot, p in enumerate(prompts):
      prefix, _ = engine.prefill(params=params, padded_tokens=torch.from_numpy(p).cuda(), true_length=len(p), slot=slot)
      prefixes.append(dict(prefix, tokens=first[:, slot:slot + 1], logits=None))
    return {"case": case, "engine": engine, "params": params, "prefixes": prefixes, "state": engine.init_decode_state(materialize_logits=True)}
  if kind == "prefill" and n == 1:
    engine, params = _engine(case, seed, 1, most + 1, min(case["chunk"], max(most, 2)), 0, {})
    return {"case": case, "engine": engine, "params": params, "prompt": torch.from_numpy(prompts[0]).cuda()}
  steps = case.get("steps", 0)
  engine, params = _engine(case, seed, n, most + steps + 1, n * most, n, {})
  state = {"case": case, "engine": engine, "params": params, "packed": _packed(prompts)}
  if kind == "utterances":
    state.update(forced=torch.from_numpy(_forced(case, seed)).cuda(), state=engine.init_decode_state(materialize_logits=True))
  return state


def run(s):
  case = s["case"]
  if case["kind"] == "train":
    metrics = s["trainer"].train_step(s["batch"])
    return {"loss": metrics["learning/loss"], "norm": metrics["learning/raw_grad_norm"], "grads": s["trainer"].grads, "params": s["trainer"].params}
  engine, params = s["engine"], s["params"]
  if case["kind"] == "decode":
    state, tokens = s["state"], []
    for slot, prefix in enumerate(s["prefixes"]):
      state = engine.insert(prefix, state, slot)
    for step in range(case["steps"]):
      state, result = engine.generate(params, state)
      tokens.append(result.data)
      if step == 0:
        first = state["logits"].clone()
    return {"first": first, "logits": state["logits"], "tokens": torch.stack(tokens)}
  if case["kind"] == "prefill" and case["prompts"] == 1:
    prompt, done, prefix = s["prompt"], 0, None
    ExistingPrefix = _module("maxengine").ExistingPrefix
    while done < prompt.numel():
      n = min(case["chunk"], prompt.numel() - done)
      old = None if done == 0 else ExistingPrefix(cache=prefix["cache"], common_prefix_tokens=prompt[:done])
      prefix, _ = engine.prefill(params=params, padded_tokens=prompt[done:done + n], true_length=n, slot=0, existing_prefix=old)
      done += n
    return {"logits": prefix["logits"], "tokens": prefix["tokens"]}
  cache, prefix, _ = engine.prefill_concat(params=params, **s["packed"])
  if case["kind"] == "prefill":
    return {"logits": prefix["logits"], "tokens": prefix["tokens"]}
  state, packed = s["state"], s["packed"]
  state = engine.insert_partial(prefix, state, cache, list(range(case["prompts"])), start_indices=packed["start_pos"], num_prompts=case["prompts"], seq_len=int(packed["true_lengths"].max()))
  for step in range(case["steps"]):
    state["tokens"].copy_(s["forced"][step].unsqueeze(1))
    state, _ = engine.generate(params, state)
  for slot in range(case["prompts"]):
    engine.release_pages(slot)
  return {"prefill": prefix["logits"], "logits": state["logits"]}


# ------------------------------------------------------------------------------------------------------------------------------ work and tolerance
def _pairs(n, done=0):
  """Query-key pairs of n causal rows behind `done` earlier ones."""
  return n * done + n * (n + 1) / 2


def work(case):
  rng = np.random.default_rng(0)
  if case["kind"] == "utterances":
    E, H, F, rank, dim, window = HYBRID[case["size"]]
    wide = 4 if case["dtype"] == "float32" else 2
    lens = _lengths(case, rng)
    weights = sum(math.prod(shape) for n, shape, _, _ in _specs(case) if len(shape) == 2 and n != "embed")
    head = HYBRID_VOCAB * E
    rows = sum(lens) + case["steps"] * len(lens)
    pairs = sum(_pairs(min(n + case["steps"], window)) for n in lens)
    passes = 1 + case["steps"]
    per_pair = H * 4 * 128 * HYBRID_LAYERS if case["model"] == "vazilorn" else H * 2 * (2 * rank + 64) * HYBRID_LAYERS // 2
    delta = 0 if case["model"] == "vazilorn" else H * 128 * 128 * HYBRID_LAYERS // 2   # numbers of the recurrent states of one sequence
    state_bytes = 8 * delta * case["steps"] * len(lens)
    cached = wide * (2 * H * 128 * HYBRID_LAYERS if case["model"] == "vazilorn" else (rank + 64) * HYBRID_LAYERS // 2)
    return {"bytes": wide * weights * passes + state_bytes + cached * sum(min(n, window) for n in lens) * case["steps"] + 4 * HYBRID_VOCAB * len(lens) * passes,
            "flops": 2 * (weights - head) * rows + 2 * head * len(lens) * passes + per_pair * pairs + 8 * delta * rows}
  s = SIZES[case["model"]]
  E, H, KV, D, F, V, L = (s[k] for k in ("E", "H", "KV", "D", "F", "V", "L"))
  L *= 2 if s["block"] == "gemma2" else 1
  narrow = 1 if case.get("quantization") == "fp8" else 2
  attn = E * D * (2 * H + 2 * KV)
  experts = s.get("K", 1)
  body = L * (attn + 3 * E * F * experts)
  if case["kind"] == "train":
    T = case["batch"] * case["length"]
    count = L * (attn + 3 * E * F) + 2 * V * E
    return {"bytes": 32.0 * count, "flops": 6.0 * T * (body + E * V) + 3 * 4.0 * H * D * L * case["batch"] * _pairs(case["length"])}
  lens = _lengths(case, rng)

  def touched(rows):      # weights that a pass of so many rows reads
    share = s["NE"] * (1 - (1 - s["K"] / s["NE"]) ** rows) if "NE" in s else 1
    return narrow * L * (attn + 3 * E * F * share) + 2 * E * V

  kv = 4 * KV * D * L
  if case["kind"] == "decode":
    keys = sum((n + case["steps"] / 2) * case["steps"] for n in lens)
    return {"bytes": case["steps"] * (touched(len(lens)) + (kv + 4 * V) * len(lens)) + kv * keys, "flops": 2.0 * len(lens) * case["steps"] * (body + E * V) + 4.0 * H * D * L * keys}
  rows = sum(lens)
  return {"bytes": touched(rows) + kv * rows + 4 * V * len(lens), "flops": 2.0 * rows * body + 2.0 * len(lens) * E * V + 4.0 * H * D * L * sum(_pairs(n) for n in lens)}


def tolerance(case):
  """The engine's llama2, Gemma and Mixtral blocks fix the order of every sum, so their numbers are a function of the inputs.  A training step and a
  hybrid decoder round operands to bf16 on the way; another sound order of sums moves those roundings.  Measured against 64 bits: gradients 0.020 to
  0.022 (largest 0.7 to 1.2 of the root mean square, in the few rows of the embedding that a batch has), hybrid logits 0.015 (0.08), in f32 6e-6 (4e-5)."""
  if case["kind"] in ("decode", "prefill"):
    return "exact"
  if case["kind"] == "train":
    return {"rel": 0.025, "max": 0.95}
  return {"rel": 2e-5, "max": 2e-4} if case["dtype"] == "float32" else {"rel": 0.02, "max": 0.3}


# ------------------------------------------------------------------------------------------------------------------------------ 64 bits
def _rms(x, eps):
  return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _turn_halves(x, pos, theta):
  """[T, heads, D]: feature i turns with feature i + D / 2."""
  half = x.shape[-1] // 2
  a = pos.double()[:, None] * theta ** (-torch.arange(half, device=x.device, dtype=torch.float64) * 2 / x.shape[-1])
  c, s = a.cos()[:, None], a.sin()[:, None]
  u, v = x[..., :half], x[..., half:]
  return torch.cat([u * c - v * s, v * c + u * s], -1)


def _turn_pairs(x, pos, f):
  """[T, heads, dims]: features 2 i and 2 i + 1 turn by position times f[i]."""
  a = pos.double()[:, None] * f
  c, s = a.cos()[:, None], a.sin()[:, None]
  u, v = x[..., 0::2], x[..., 1::2]
  return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)


def _attend(q, k, v, mask, cap=0.0, sink=None):
  """q [T, H, D], k and v [T, KV, D] -> [T, H, D']; mask [T, T] of the pairs that count."""
  T, H, _ = q.shape
  G = H // k.shape[1]
  s = torch.matmul(q.transpose(0, 1).reshape(k.shape[1], G * T, -1), k.permute(1, 2, 0).contiguous()).reshape(H, T, -1)
  if cap:
    s = cap * torch.tanh(s / cap)
  s = s.masked_fill(~mask, -math.inf)
  if sink is not None:
    s = torch.cat([s, sink[:, None, None].expand(H, T, 1)], -1)
  p = torch.softmax(s, -1)[..., :k.shape[0]]
  return torch.matmul(p.reshape(k.shape[1], G * T, -1), v.transpose(0, 1).contiguous()).reshape(H, T, -1).transpose(0, 1)


def _layers(w, s):
  """(names, window, gemma) of every attention layer in order."""
  for i in range(s["L"]):
    p = f"params/decoder/layers_{i}/"
    if s["block"] == "gemma2":
      for sub in ("_local", "_global"):
        yield {"ln1": p + f"pre_self_attention_norm{sub}/scale", "a": p + f"self_attention{sub}/", "pan": p + f"post_self_attention_norm{sub}/scale",
               "ln2": p + ("mlp_local/mlp_layer_norm/scale" if sub == "_local" else "pre_ffw_norm_global/scale"), "m": p + f"mlp{sub}/", "pfn": p + f"post_ffw_norm{sub}/scale"}, 4096 if sub == "_local" else 0
    else:
      yield {"ln1": p + "pre_self_attention_layer_norm/scale", "a": p + "self_attention/", "ln2": p + ("post_self_attention_layer_norm/scale" if s["block"] == "mixtral" else "mlp/mlp_layer_norm/scale"),
             "m": p + ("MoeBlock_0/" if s["block"] == "mixtral" else "mlp/")}, 0


def _silu(x):
  return x * torch.sigmoid(x)


def _logits(case, w, sequences):
  """Logits of the last token of every sequence."""
  s = SIZES[case["model"]]
  E, D, eps, gemma = s["E"], s["D"], s.get("eps", 1e-5), s["block"] == "gemma2"
  lens = [len(t) for t in sequences]
  pos = torch.cat([torch.arange(n, device="cuda") for n in lens])
  emb = w["params/token_embedder/embedding"]
  x = emb[torch.from_numpy(np.concatenate(sequences)).cuda().long()].double()
  cut = lambda n: range(0, n, 16384)
  for names, window in _layers(w, s):
    g = lambda key: w[key].double()
    xn = _rms(x, eps) * g(names["ln1"])
    q, k, v = ((xn @ g(names["a"] + n + "/kernel").reshape(E, -1)).reshape(len(x), -1, D) for n in ("query", "key", "value"))
    q, k = _turn_halves(q, pos, s.get("theta", 1e4)), _turn_halves(k, pos, s.get("theta", 1e4))
    out, at = torch.empty_like(q), 0
    for n in lens:
      i = torch.arange(n, device="cuda")
      mask = (i[:, None] >= i) & ((i[:, None] - i < window) if window else True)
      out[at:at + n] = _attend(q[at:at + n], k[at:at + n], v[at:at + n], mask, 50.0 if gemma else 0.0)
      at += n
    y = out.reshape(len(x), -1) @ g(names["a"] + "out/kernel").reshape(-1, E)
    x = x + (_rms(y, eps) * g(names["pan"]) if gemma else y)
    xn = _rms(x, eps) * g(names["ln2"])
    if s["block"] == "mixtral":
      top, idx = (xn @ g(names["m"] + "gate/kernel")).topk(s["K"])
      share, y = torch.softmax(top, -1), torch.zeros_like(x)
      wi0, wi1, wo = (w[names["m"] + n] for n in ("wi_0", "wi_1", "wo"))
      for e in range(s["NE"]):
        rows, at = (idx == e).nonzero(as_tuple=True)
        if len(rows):
          y[rows] += share[rows, at, None] * ((_silu(xn[rows] @ wi0[e].double()) * (xn[rows] @ wi1[e].double())) @ wo[e].double())
    else:
      wi0, wi1, wo = (g(names["m"] + n + "/kernel") for n in ("wi_0", "wi_1", "wo"))
      act = (lambda t: torch.nn.functional.gelu(t, approximate="tanh")) if gemma else _silu
      y = torch.cat([(act(xn[c:c + 16384] @ wi0) * (xn[c:c + 16384] @ wi1)) @ wo for c in cut(len(x))])
    x = x + (_rms(y, eps) * g(names["pfn"]) if gemma else y)
  last = _rms(x[torch.from_numpy(np.cumsum(lens) - 1).cuda()], eps) * w["params/decoder/decoder_norm/scale"].double()
  if gemma:
    return 30.0 * torch.tanh(last @ emb.double().T.contiguous() / math.sqrt(E) / 30.0)
  return last @ w["params/decoder/logits_dense/kernel"].double()


def _hybrid_logits(case, w, tokens, wanted):
  """Logits [wanted, vocab] of one sequence at the wanted places."""
  E, H, _, rank, dim, window = HYBRID[case["size"]]
  T, eps = len(tokens), 1e-5
  x = w["embed"][torch.from_numpy(tokens).cuda().long()].double()
  pos = torch.arange(T, device="cuda")
  mask = (pos[:, None] >= pos) & (pos[:, None] - pos < window)
  lin = lambda name, h: h @ w[name].double().T
  d = lambda name: w[name].double()

  def norm(name, h):
    if case["model"] == "vilepel":
      return _rms(h, eps) * (1 + d(name))
    return d(name) * torch.tanh(d(name + ".alpha") * h) + d(name + ".b")

  def frequencies(dims, base, scaled):
    f = base ** (-torch.arange(0, dims, 2, device="cuda", dtype=torch.float64) / dims)
    if not scaled:
      return f
    share = ((8192 * f / (2 * math.pi) - 1.0) / 3.0).clamp(0.0, 1.0)
    return share * f + (1 - share) * f / 8.0

  def attention(p, h):
    f = frequencies(128, 500000.0, True)
    q = _turn_pairs(_rms(lin(p + "q", h).reshape(T, H, 128), eps) * d(p + "q.norm"), pos, f)
    k = _turn_pairs(_rms(lin(p + "k", h).reshape(T, H, 128), eps) * d(p + "k.norm"), pos, f)
    return _attend(q * 128 ** -0.5, k, lin(p + "v", h).reshape(T, H, 128), mask, sink=d(p + "sink"))

  def latent(p, h):
    f = frequencies(64, 10000.0, False)
    q, c = lin(p + "q", h).reshape(T, H, dim + 64), lin(p + "dkv", h)
    kr, c = _turn_pairs(c[:, None, rank:], pos, f), _rms(c[:, :rank], eps) * d(p + "dkv.norm")
    k = torch.cat([lin(p + "uk", c).reshape(T, H, dim), kr.expand(T, H, 64)], -1)
    q = torch.cat([q[..., :dim], _turn_pairs(q[..., dim:], pos, f)], -1) * (dim + 64) ** -0.5
    return _attend(q, k, lin(p + "uv", c).reshape(T, H, 128), mask)

  def delta(p, h):
    def conv(n):
      y, taps = torch.nn.functional.pad(lin(p + n, h), (0, 0, 3, 0)), d(p + n + ".conv")
      return _silu(sum(y[j:j + T] * taps[:, j] for j in range(4))).reshape(T, H, 128)
    unit = lambda t: t / torch.sqrt(t.square().sum(-1, keepdim=True) + 1e-6)
    q, k, v = unit(conv("q")) * 128 ** -0.5, unit(conv("k")), conv("v")
    beta = torch.sigmoid(lin(p + "b", h))
    a = (lin(p + "a2", lin(p + "a1", h)) + d(p + "dt_bias")).reshape(T, H, 128)
    decay = torch.exp(-torch.exp(d(p + "A_log"))[:, None] * torch.nn.functional.softplus(a))
    S, out = torch.zeros(H, 128, 128, device="cuda", dtype=torch.float64), torch.empty_like(v)
    for t in range(T):
      S = decay[t][:, :, None] * S
      u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
      S = S + k[t][:, :, None] * u[:, None]
      out[t] = (S * q[t][:, :, None]).sum(1)
    return _rms(out, eps) * d(p + "norm") * torch.sigmoid(lin(p + "g2", lin(p + "g1", h))).reshape(T, H, 128)

  for i in range(HYBRID_LAYERS):
    p = f"l{i}."
    h = x if case["model"] == "vilepel" else norm(p + "norm1", x)
    mixer = attention if case["model"] == "vazilorn" else (delta, latent)[i % 2]
    y = lin(p + "mix.o", mixer(p + "mix.", h).reshape(T, -1))
    x = x + norm(p + ("norm1" if case["model"] == "vilepel" else "norm1b"), y)
    h = x if case["model"] == "vilepel" else norm(p + "norm2", x)
    g, u = lin(p + "mlp.gate", h), lin(p + "mlp.up", h)
    if case["model"] == "vilepel":
      g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
      act = g * torch.sigmoid(1.702 * g) * (u + 1)
    else:
      act = torch.nn.functional.gelu(g, approximate="tanh") * u
    y = lin(p + "mlp.down", act)
    x = x + norm(p + ("norm2" if case["model"] == "vilepel" else "norm2b"), y)
  return lin("head", norm("final.norm", x[wanted]))


def _train(case, seed):
  """One training step in 64 bits by autograd, row by row."""
  s, tree = SIZES[case["model"]], _Tree(case, seed)
  E, H, D, L, S = s["E"], s["H"], s["D"], s["L"], case["length"]
  w = {n: t.double().requires_grad_(True) for n, t in tree.items()}
  dev = {k: torch.from_numpy(v).cuda().long() for k, v in _batch(case, seed).items()}
  i, total, weights = torch.arange(S, device="cuda"), 0.0, 0
  for b in range(case["batch"]):
    seg, pos = dev["inputs_segmentation"][b], dev["inputs_position"][b]
    mask = (seg[:, None] == seg) & (i[:, None] >= i)
    x = w["params/token_embedder/embedding"][dev["inputs"][b]]
    for names, _ in _layers(w, s):
      xn = _rms(x, 1e-5) * w[names["ln1"]]
      q, k, v = ((xn @ w[names["a"] + n + "/kernel"].reshape(E, -1)).reshape(S, -1, D) for n in ("query", "key", "value"))
      y = _attend(_turn_halves(q, pos, 1e4), _turn_halves(k, pos, 1e4), v, mask)
      x = x + y.reshape(S, H * D) @ w[names["a"] + "out/kernel"].reshape(-1, E)
      xn = _rms(x, 1e-5) * w[names["ln2"]]
      x = x + (_silu(xn @ w[names["m"] + "wi_0/kernel"]) * (xn @ w[names["m"] + "wi_1/kernel"])) @ w[names["m"] + "wo/kernel"]
    logits = (_rms(x, 1e-5) * w["params/decoder/decoder_norm/scale"]) @ w["params/decoder/logits_dense/kernel"]
    count = dev["targets_segmentation"][b] != 0
    loss = torch.nn.functional.cross_entropy(logits[count], dev["targets"][b][count], reduction="sum")
    loss.backward()
    total, weights = total + float(loss.detach()), weights + int(count.sum())
    del x, xn, q, k, v, y, logits, loss
  flat = lambda part: torch.cat([part(t).reshape(-1) for t in w.values()])
  grads = flat(lambda t: t.grad)
  norm = float(grads.norm()) / weights
  params = flat(lambda t: t.detach())
  g = grads / weights * min(1.0, 1.0 / norm)          # clipped to a global norm of 1, then the first AdamW update
  params -= 3e-5 * (g / (g.abs() + 1e-8) + 0.1 * params)
  return {"loss": total / weights, "norm": norm, "grads": grads, "params": params}


def exact(case, seed):
  if case["kind"] == "train":
    return _train(case, seed)
  w, prompts = _Tree(case, seed), _prompts(case, seed)
  if case.get("quantization") == "fp8":
    return None                                       # the scheme's own rounding of the weights is part of the result
  with torch.no_grad():
    if case["kind"] == "prefill":
      out = _logits(case, w, prompts)
      return {"logits": out.reshape((len(prompts), 1, 1, -1) if len(prompts) > 1 else (1, 1, -1)), "tokens": None}
    if case["kind"] == "decode":                      # the first step; the later tokens are the framework's own choice
      first = _forced(case, seed)[0]
      out = torch.cat([_logits(case, w, [np.append(p, first[i]) for i, p in list(enumerate(prompts))[at:at + 32]]) for at in range(0, len(prompts), 32)])
      return {"first": out[:, None], "logits": None, "tokens": None}
    forced = _forced(case, seed)
    outs = [_hybrid_logits(case, w, np.concatenate([p, forced[:, i]]), [len(p) - 1, len(p) + len(forced) - 1]) for i, p in enumerate(prompts)]
    return {"prefill": torch.stack([o[0] for o in outs])[:, None, None], "logits": torch.stack([o[1] for o in outs])[:, None]}
