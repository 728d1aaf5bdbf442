"""Several engines on one GPU: passes whose launches have blocks that wait for each other (k_step, k_mid, k_attn_split) beside each other on streams and threads.  Every token is what
a model alone gives, whichever form a pass took."""
import ctypes
import gc
import subprocess
import sys
import threading

import numpy as np
import pytest

import helpers as H
from test_gpu_step import _config

pytestmark = pytest.mark.gpu

STEP, MID, SPLIT = 1, 2, 4
FEW, SOME = (1, 2048, 16, 16, 128, 7168), (20, 512, 4, 4, 64, 1024)      # rows, emb, query heads, kv heads, dim, mlp


def forms(eng):
  out = ctypes.c_int32(-1)
  H.lib.check(eng.lib.ixt_pass_forms(eng._ctx, ctypes.byref(out)))
  return out.value


class Run:
  """One engine with its prompts prefilled and inserted, on a stream of its own."""
  alive = []

  def __init__(self, shape, seed, steps, stream=None, **keys):
    import torch
    self.torch, self.stream, self.tokens = torch, stream or torch.cuda.Stream(), []
    self.cfg = _config(*shape, 12 + steps, 2, **keys)
    self.eng, self.params = H.make_engine(self.cfg, H.synth.synth_weights(self.cfg, seed))
    Run.alive.append(self.eng)
    self.begin()

  def begin(self):
    with self.torch.cuda.stream(self.stream):
      self.state, self.tokens = self.eng.init_decode_state(), []
      for slot in range(self.eng.max_concurrent_decodes):
        prefix, _ = self.eng.prefill(params=self.params, padded_tokens=H.synth.synth_prompt(self.cfg.vocab_size, 12, slot)[0], true_length=1 + slot % 12, slot=slot)
        self.state = self.eng.insert(prefix, self.state, slot)
    self.torch.cuda.synchronize()

  def hold(self):
    """Something in front of the next steps, so that they are still on their way when others are asked for."""
    with self.torch.cuda.stream(self.stream):
      self.torch.cuda._sleep(20_000_000)
    return self

  def step(self):
    with self.torch.cuda.stream(self.stream):
      self.state, result = self.eng.generate(self.params, self.state)
      self.tokens.append(result.data.clone())
    return forms(self.eng)

  def result(self):
    self.torch.cuda.synchronize()
    assert self.eng.exchange_status() == 0
    return self.torch.stack(self.tokens).cpu().numpy()


@pytest.fixture(autouse=True)
def closed():
  """Engines that are still there count: those of earlier tests go first."""
  gc.collect()
  yield
  while Run.alive:
    Run.alive.pop().close()


def test_a_pass_beside_another():
  """While passes of another engine are on their way an engine takes the forms without waits; behind them, and alone, those with."""
  a, b = Run(FEW, 1, 130), Run(SOME, 2, 130)
  a.hold()
  assert [a.step() for _ in range(60)] == [STEP] * 60
  assert b.hold().step() == 0 and a.step() == 0
  a.result()
  b.result()
  b.hold()
  assert [b.step() for _ in range(60)] == [MID] * 60
  assert a.hold().step() == 0 and b.step() == 0
  b.result()
  assert a.step() == STEP
  got = [a.result(), b.result()]
  for r, n, tokens in zip((a, b), (63, 62), got):
    r.begin()
    for _ in range(n):
      r.step()
      r.stream.synchronize()
    assert np.array_equal(tokens, r.result())


def test_engines_on_one_stream():
  """Passes of one stream run one after the other: all with waits, however many are on their way."""
  a = Run(FEW, 1, 130)
  b = Run(SOME, 2, 130, stream=a.stream)
  for _ in range(40):
    assert a.step() == STEP and b.step() == MID
  got = [a.result(), b.result()]
  for r, tokens in zip((a, b), got):
    r.begin()
    for _ in range(40):
      r.step()
      r.stream.synchronize()
    assert np.array_equal(tokens, r.result())


def test_engines_on_threads():
  runs = [Run(FEW, 1, 60), Run(SOME, 2, 60), Run(FEW[:1] + (768, 12, 12, 64, 2048), 3, 60)]
  alone = []
  for r in runs:
    for _ in range(50):
      r.step()
    alone.append(r.result())
    r.begin()
  errors = []

  def work(r):
    try:
      for _ in range(50):
        r.step()
    except Exception as e:  # pylint: disable=broad-except
      errors.append(e)

  threads = [threading.Thread(target=work, args=(r,)) for r in runs]
  for t in threads:
    t.start()
  for t in threads:
    t.join(60)
  assert not errors and not any(t.is_alive() for t in threads)
  for r, want in zip(runs, alone):
    assert np.array_equal(r.result(), want)


@pytest.mark.parametrize("beside", [FEW, SOME])
def test_split_attention_beside_whole_steps(beside):
  """Blocks of the split decode attention all count on being on the chip together; 5 slots of 4 kv heads leave those of a head on several of its parts."""
  split = Run((5, 512, 8, 4, 128, 512), 6, 200, model_name="gemma2-tiny", sliding_window_size=64)
  other = Run(beside, 7, 200)
  alone = []
  for r, form in ((split, SPLIT), (other, STEP if beside is FEW else MID)):
    assert [r.step() for _ in range(60)] == [form] * 60
    alone.append(r.result())
    r.begin()
  seen = {split.hold().step(), other.hold().step()}
  for _ in range(59):
    seen |= {split.step(), other.step()}
  assert 0 in seen
  for r, want in zip((split, other), alone):
    assert np.array_equal(r.result(), want)


def test_an_engine_that_goes_leaves_the_gate_open():
  a, b = Run(FEW, 1, 20), Run(FEW, 2, 20)
  for _ in range(10):
    a.step()
  a.eng.close()
  assert b.step() == STEP
  b.result()


@pytest.mark.parametrize("shape", [FEW, SOME])
def test_a_stream_that_the_caller_captures(shape):
  """Its graph is replayed without a call into the library, so it holds no launch that waits."""
  import torch
  r = Run(shape, 4, 20, ixt_use_hip_graph=False)
  want = []
  for _ in range(6):
    assert r.step() == (STEP if shape is FEW else MID)
  want = r.result()
  r.begin()
  r.step()
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph, stream=r.stream):
    r.state, result = r.eng.generate(r.params, r.state)
  assert forms(r.eng) == 0
  got = [r.tokens[0]]
  for _ in range(5):
    graph.replay()
    got.append(result.data.clone())
    torch.randn(1 << 20, device="cuda").sum().item()
  assert r.eng.exchange_status() == 0
  assert np.array_equal(torch.stack(got).cpu().numpy(), want)


def test_beside_a_capture_of_another_thread():
  """Looking whether another engine's passes have ended does not end a capture that another thread has under way."""
  import torch
  a, b, c = Run(FEW, 1, 40), Run(FEW, 2, 40), Run(SOME, 3, 40)
  alone = []
  for r in (a, b, c):
    for _ in range(24):
      r.step()
    alone.append(r.result())
    r.begin()
  x, graph, errors = torch.zeros(64, device="cuda"), torch.cuda.CUDAGraph(), []

  def work():
    try:
      for _ in range(8):
        for r in (a, a, b, b, c, c, c):
          r.step()
      for r, n in ((a, 8), (b, 8)):
        for _ in range(n):
          r.step()
    except Exception as e:  # pylint: disable=broad-except
      errors.append(e)

  x.add_(0.0)
  torch.cuda.synchronize()
  with torch.cuda.graph(graph):
    x.add_(1.0)
    t = threading.Thread(target=work)
    t.start()
    t.join(60)
    x.add_(1.0)
  assert not errors and not t.is_alive()
  for _ in range(3):
    graph.replay()
  for r, want in zip((a, b, c), alone):
    assert np.array_equal(r.result(), want)
  assert x.cpu().tolist() == [6.0] * 64


HOLD = """
import fcntl, os, sys
fd = os.open(sys.argv[1], os.O_RDWR | os.O_CREAT, 0o666)
fcntl.lockf(fd, fcntl.LOCK_EX | fcntl.LOCK_NB)
print("held", flush=True)
sys.stdin.readline()
"""


def test_beside_another_process():
  """While another process holds the GPU's lock, passes take the forms without waits; they take it when it has gone."""
  import torch
  alone = Run(FEW, 5, 20)
  for _ in range(8):
    alone.step()
  want = alone.result()
  alone.eng.close()                                      # (this process's engines let go of the lock)
  props = torch.cuda.get_device_properties(0)
  lock = f"/tmp/libixt-gpu-{props.pci_domain_id:04x}:{props.pci_bus_id:02x}:{props.pci_device_id:02x}.0.lock"
  with subprocess.Popen([sys.executable, "-c", HOLD, lock], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True) as other:
    assert other.stdout.readline() == "held\n"
    r = Run(FEW, 5, 20)
    assert [r.step() for _ in range(4)] == [0] * 4
    other.stdin.write("\n")
    other.stdin.flush()
    assert other.wait(30) == 0
  assert [r.step() for _ in range(4)] == [STEP] * 4
  assert np.array_equal(r.result(), want)


# ---- waits that give up
def _give_up(r, polls):
  H.lib.check(r.eng.lib.ixt_set_option(r.eng._ctx, b"wait_polls", polls))


GEMMA = dict(model_name="gemma2-tiny", sliding_window_size=64)


@pytest.mark.parametrize("shape,form,keys", [(FEW, STEP, {}), (SOME, MID, {}), ((5, 512, 8, 4, 128, 512), SPLIT, GEMMA)], ids=["step", "mid", "split"])
def test_a_wait_that_gives_up_is_reported(shape, form, keys):
  """No looks at all: what is handed out says so, the next call raises, once, and passes behind it are right again."""
  import torch
  r = Run(shape, 9, 20, **keys)
  for _ in range(5):
    assert r.step() == form
  want = r.result()
  r.begin()
  _give_up(r, 0)
  assert r.step() == form
  torch.cuda.synchronize()
  assert not r.tokens[0][:, 1].any()                     # not valid
  with pytest.raises(H.lib.IxtError, match="gave up"):
    r.step()
  _give_up(r, 1 << 20)
  r.begin()                                              # reported: the prompts again
  for _ in range(5):
    assert r.step() == form
  assert r.tokens[0][:, 1].all()
  assert np.array_equal(r.result(), want)


@pytest.mark.parametrize("late", ["convert", "insert", "prefill", "prefill_concat", "insert_partial", "step"])
def test_where_it_is_reported(late):
  """Whatever the engine is asked for next says what happened to the pass before."""
  import torch
  keys = dict(ixt_staging_groups=2, ixt_max_packed_rows=24, use_chunked_prefill=True) if late in ("prefill_concat", "insert_partial", "step") else {}
  r = Run((2,) + FEW[1:], 10, 20, **keys)
  toks = H.synth.synth_prompt(r.cfg.vocab_size, 12, 3)[0]
  packed = dict(params=r.params, padded_tokens=np.tile(toks[:4], 2), decoder_positions=np.tile(np.arange(4, dtype=np.int32), 2), decoder_segment_ids=np.repeat(np.arange(2) + 1, 4).astype(np.int32),
                start_pos=np.array([0, 4], np.int32), true_lengths=np.array([4, 4], np.int32), num_prompts=2)
  with torch.cuda.stream(r.stream):
    cache, prefix, _ = r.eng.prefill_concat(**packed) if keys else (None, None, None)
    torch.cuda.synchronize()
    _give_up(r, 0)
    if late == "convert":
      prefix, result = r.eng.prefill(params=r.params, padded_tokens=toks, true_length=12, slot=0)
    elif late == "insert":
      prefix, result = r.eng.prefill(params=r.params, padded_tokens=toks, true_length=12, slot=0)
    else:
      r.state, result = r.eng.generate(r.params, r.state)
    if late != "convert":
      torch.cuda.synchronize()
    with pytest.raises(H.lib.IxtError, match="gave up"):
      if late == "convert":
        result.convert_to_numpy()
      elif late == "insert":
        r.eng.insert(prefix, r.state, 0)
      elif late == "prefill":
        r.eng.prefill(params=r.params, padded_tokens=toks, true_length=12, slot=0)
      elif late == "prefill_concat":
        r.eng.prefill_concat(**packed)
      elif late == "insert_partial":
        r.eng.insert_partial(prefix, r.state, cache, [0, 1], num_prompts=2)
      else:
        r.eng.step([(0, 0, toks[:3], [2])])
  assert r.eng.exchange_status() == 0                    # reported once
