"""The rule that keeps launches whose blocks wait for each other apart (csrc/ixt_gate.h), built for the host by itself and driven by threads: a pass may take them
only while no other context's pass can be on another stream of the GPU, nobody stands still for the answer, and no path of errors leaves the gate shut."""
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
#include <sstream>
#include <string>
#include <thread>
#include <vector>
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

struct Event { bool ended = true; };
static auto ended = [](void* e) { return static_cast<Event*>(e)->ended; };
static auto mark = [](void* e) { static_cast<Event*>(e)->ended = false; return true; };
static auto broken = [](void*) { return false; };

static std::vector<std::string> files;

static IxtGate::Lane lane(long n) { return IxtGate::Lane(reinterpret_cast<void*>(n), std::thread::id()); }
static int settles = 0;
static auto settle = [] { ++settles; return true; };
static auto cannot = [] { return false; };

static int rules() {
  IxtGate g(files);
  Event a, b, c;
  auto in = [&](Event& e, long n) { return g.enter(&e, lane(n), &e, ended, settle); };
  auto out = [&](Event& e) { g.leave(&e, mark); };
  CHECK(in(a, 1)); out(a);
  CHECK(in(a, 2)); out(a);                               // its own passes are in order
  CHECK(in(b, 2)); out(b);                               // so are those of one stream
  CHECK(a.ended && b.ended && settles == 0);             // no event, no look
  CHECK(in(c, 3)); out(c);
  CHECK(settles == 1 && !c.ended);                       // passes without an event on another stream: waited for, once
  CHECK(!in(a, 2)); out(a);                              // c's may still run
  CHECK(!in(c, 3)); out(c);                              // so may a's
  a.ended = true;
  CHECK(in(c, 3));                                       // (b's were waited for)
  bool other = true;                                     // another thread, while c's pass is being enqueued: refused, at once
  std::thread([&] { other = in(a, 2); out(a); }).join();
  CHECK(!other);
  out(c);
  CHECK(in(a, 3)); out(a);                               // behind c's, on its stream
  a.ended = c.ended = true;
  CHECK(in(b, 1)); g.leave(&b, broken);                  // nothing tells when this one has ended
  CHECK(!g.enter(&a, lane(2), &a, ended, cannot)); out(a);
  a.ended = true;
  CHECK(in(c, 3) && settles == 2); out(c);               // but the GPU can be waited for
  c.ended = true;
  CHECK(in(b, 1)); g.leave(&b, broken);
  g.forget(&b);                                          // or its context goes
  CHECK(g.enter(&a, lane(2), &a, ended, cannot)); out(a);
  g.forget(&c);
  CHECK(g.enter(&a, lane(1), &a, ended, cannot));
  a.ended = true; out(a);
  CHECK(a.ended);                                        // alone again: no event
  return 0;
}

// contexts on threads and streams of their own; a pass stays on the "GPU" for a while after it was enqueued
static int apart() {
  IxtGate g(files);
  std::atomic<long> until[4], waiting[4];                // ends of the last pass, and of the last one with blocks that wait
  std::atomic<int> running{-1}, bad{0}, in{0};
  auto now = [] { return (long)std::chrono::steady_clock::now().time_since_epoch().count(); };
  auto over = [&](void* e) { return now() >= *static_cast<std::atomic<long>*>(e); };
  auto all_over = [&] { for (auto& u : until) while (now() < u) {} return true; };
  for (int k = 0; k < 4; ++k) until[k] = waiting[k] = 0;
  std::vector<std::thread> ts;
  for (int k = 0; k < 4; ++k)
    ts.emplace_back([&, k] {
      for (int i = 0; i < 3000; ++i) {
        const bool may = g.enter(&until[k], lane(k), &until[k], over, all_over);
        if (may) {
          const int before = running.exchange(k);
          if (before >= 0 && before != k && now() < waiting[before]) ++bad;
          ++in;
        }
        until[k] = std::max(until[k].load(), now()) + (may ? 20000 : 2000);      // (behind its pass before)
        if (may) waiting[k] = until[k].load();
        g.leave(&until[k], [&](void*) { return i % 16 != 15; });
        if (i % 4 == k) std::this_thread::sleep_for(std::chrono::microseconds(30));
      }
    });
  for (auto& t : ts) t.join();
  CHECK(bad == 0 && in > 0);
  return 0;
}
// argv: files (a colon between them), and "hold" to keep the lock until a line comes in, or "ask": may a pass take the waiting forms?
int main(int argc, char** argv) {
  std::stringstream names(argv[1]);
  for (std::string n; std::getline(names, n, ':');) files.push_back(n);
  if (argc == 2) return rules() || apart();
  IxtGate g(files);
  Event a;
  auto ask = [&] { const bool may = g.enter(&a, lane(1), &a, ended, settle); g.leave(&a, mark); return may; };
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
  assert _ask(program, f"{tmp_path}/none/lock:{tmp_path}/second") == "1" and os.path.exists(tmp_path / "second") and not os.path.exists(tmp_path / "none")
  os.symlink(tmp_path / "target", tmp_path / "link")
  assert _ask(program, str(tmp_path / "link")) == "0"
