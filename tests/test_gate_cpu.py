"""The rule that keeps launches whose blocks wait for each other apart (csrc/ixt_gate.h), built for the host by itself and driven by threads: a pass may take them
only while no other context's pass can be on the GPU, nobody stands still for the answer, and no path of errors leaves the gate shut."""
import os
import shutil
import signal
import subprocess

import pytest

import helpers as H

build = H.importlib.import_module("maxtext-indextts2_amd.build")

PROGRAM = r"""
#include "ixt_gate.h"
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

struct Event { bool ended = true; };
static auto ended = [](void* e) { return static_cast<Event*>(e)->ended; };
static auto mark = [](void* e) { static_cast<Event*>(e)->ended = false; return true; };
static auto broken = [](void*) { return false; };

static const char* file;

static int rules() {
  IxtGate g(file);
  Event a, b, c;
  int settled = 0;
  auto settle = [&] { ++settled; return true; };
  g.join(&a, &a, settle);
  CHECK(g.enter(&a, ended)); g.leave(&a, mark);
  CHECK(a.ended);                                        // alone: no event
  CHECK(g.enter(&a, ended)); g.leave(&a, mark);          // its own passes are in order
  g.join(&b, &b, settle);
  CHECK(settled == 1);                                   // a's last pass has no event: waited for
  CHECK(g.enter(&b, ended)); g.leave(&b, mark);
  CHECK(!b.ended);
  CHECK(!g.enter(&a, ended)); g.leave(&a, mark);         // b's may still run
  CHECK(!g.enter(&b, ended)); g.leave(&b, mark);         // so may a's
  a.ended = true;
  CHECK(g.enter(&b, ended));
  bool other = true;                                     // another thread, while b's pass is being enqueued: refused, at once
  std::thread([&] { other = g.enter(&a, ended); g.leave(&a, mark); }).join();
  CHECK(!other);
  g.leave(&b, mark);
  b.ended = a.ended = true;
  CHECK(g.enter(&b, ended)); g.leave(&b, broken);        // nothing tells when this one has ended
  CHECK(!g.enter(&a, ended)); g.leave(&a, mark);
  a.ended = true;
  CHECK(g.enter(&b, ended)); g.leave(&b, mark);          // until the next one
  b.ended = true;
  CHECK(g.enter(&a, ended)); g.leave(&a, broken);
  g.forget(&a);                                          // or its context goes
  CHECK(g.enter(&b, ended)); g.leave(&b, mark);
  g.join(&c, &c, [&] { return false; });                 // the GPU cannot be waited for: b's pass counts as on its way
  CHECK(!g.enter(&c, ended)); g.leave(&c, mark);
  return 0;
}

// A context comes while another's pass is being enqueued: that pass gets an event.
static int joined_in_between() {
  IxtGate g(file);
  Event a, b;
  auto never = [] { return false; };
  g.join(&a, &a, never);
  CHECK(g.enter(&a, ended));
  g.join(&b, &b, [&] { g.leave(&a, mark); return true; });   // (enqueued while the other waits for the GPU: not covered by that wait)
  CHECK(!a.ended && !g.enter(&b, ended));
  return 0;
}

// contexts on threads of their own; a pass stays on the "GPU" for a while after it was enqueued
static int apart() {
  IxtGate g(file);
  std::atomic<long> until[4], waiting[4];                // ends of the last pass, and of the last one with blocks that wait
  std::atomic<int> running{-1}, bad{0}, in{0};
  auto now = [] { return (long)std::chrono::steady_clock::now().time_since_epoch().count(); };
  auto over = [&](void* e) { return now() >= *static_cast<std::atomic<long>*>(e); };
  for (int k = 0; k < 4; ++k) { until[k] = waiting[k] = 0; g.join(&until[k], &until[k], [] { return true; }); }
  std::vector<std::thread> ts;
  for (int k = 0; k < 4; ++k)
    ts.emplace_back([&, k] {
      for (int i = 0; i < 3000; ++i) {
        const bool may = g.enter(&until[k], over);
        if (may) {
          const int before = running.exchange(k);
          if (before >= 0 && before != k && now() < waiting[before]) ++bad;
          ++in;
        }
        g.leave(&until[k], [&](void*) {
          until[k] = std::max(until[k].load(), now()) + (may ? 20000 : 2000);      // (behind its pass before)
          if (may) waiting[k] = until[k].load();
          return true;
        });
        if (i % 4 == k) std::this_thread::sleep_for(std::chrono::microseconds(30));
      }
    });
  for (auto& t : ts) t.join();
  CHECK(bad == 0 && in > 0);
  return 0;
}
// argv: file, and "hold" to keep the lock until a line comes in, or "ask": may a pass take the waiting forms?
int main(int argc, char** argv) {
  file = argv[1];
  if (argc == 2) return rules() || joined_in_between() || apart();
  IxtGate g(file);
  Event a;
  auto ask = [&] { const bool may = g.enter(&a, ended); g.leave(&a, mark); return may; };
  g.join(&a, &a, [] { return true; });
  std::printf("%d\n", (int)ask());
  std::fflush(stdout);
  if (argv[2][0] == 'h') {
    if (fork() == 0) pause();                            // a child that outlives its parent holds nothing
    std::getchar();
    g.forget(&a);
    std::printf("gone\n");
    std::fflush(stdout);
    std::getchar();
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
  cxx = shutil.which("g++") or shutil.which("c++")
  if cxx is None:
    pytest.skip("no C++ compiler here")
  d = tmp_path_factory.mktemp("gate")
  src, exe = os.path.join(d, "gate.cpp"), os.path.join(d, "gate")
  with open(src, "w", encoding="utf-8") as f:
    f.write(PROGRAM)
  subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I", build.CSRC, src, "-o", exe], check=True)
  return exe


def test_one_context_at_a_time(program, tmp_path):
  done = subprocess.run([program, str(tmp_path / "lock")], capture_output=True, text=True, timeout=60, check=False)
  assert done.returncode == 0, done.stdout


def _ask(program, lock):
  return subprocess.run([program, lock, "ask"], capture_output=True, text=True, timeout=60, check=True).stdout.strip()


def test_one_process_at_a_time(program, tmp_path):
  lock = str(tmp_path / "lock")
  assert _ask(program, lock) == "1" and _ask(program, lock) == "1"         # the first has gone
  with subprocess.Popen([program, lock, "hold"], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True, start_new_session=True) as first:
    try:
      assert first.stdout.readline() == "1\n"
      assert _ask(program, lock) == "0"
      first.stdin.write("\n")
      first.stdin.flush()
      assert first.stdout.readline() == "gone\n"                          # its last context has
      assert _ask(program, lock) == "1"
    finally:
      os.killpg(first.pid, signal.SIGKILL)


def test_a_process_that_dies_lets_go(program, tmp_path):
  lock = str(tmp_path / "lock")
  with subprocess.Popen([program, lock, "hold"], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True, start_new_session=True) as first:
    try:
      assert first.stdout.readline() == "1\n" and _ask(program, lock) == "0"
      first.kill()                                                        # (its child lives on)
      first.wait(30)
      assert _ask(program, lock) == "1"
    finally:
      os.killpg(first.pid, signal.SIGKILL)


def test_no_file_no_waits(program, tmp_path):
  """Where the lock cannot be taken at all, or the file is somebody's link, a pass takes the forms without waits."""
  assert _ask(program, str(tmp_path / "none" / "lock")) == "0"
  os.symlink(tmp_path / "target", tmp_path / "link")
  assert _ask(program, str(tmp_path / "link")) == "0"
