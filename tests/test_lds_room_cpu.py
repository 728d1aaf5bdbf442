"""Room for dynamic LDS is asked for once a kernel and device (csrc/ixt_lds_room.h), built for the host by itself: a second GPU of a process is asked too, a refusal is asked again, a
larger size is a question of its own; and no launch helper keeps a flag for all devices in its place."""
import glob
import os
import re
import shutil
import subprocess

import pytest

import helpers as H

build = H.importlib.import_module("maxtext-indextts2_amd.build")

PROGRAM = r"""
#include "ixt_lds_room.h"
#include <cstdio>
#include <thread>
#include <vector>
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
  IxtLdsRoom r;
  int asked = 0, rc = 0;
  auto give = [&] { ++asked; return rc; };
  CHECK(r.ask(0, 96, give) == 0 && asked == 1);
  CHECK(r.ask(0, 96, give) == 0 && r.ask(0, 64, give) == 0 && asked == 1);
  CHECK(r.ask(1, 96, give) == 0 && asked == 2);          // another device
  CHECK(r.ask(0, 128, give) == 0 && asked == 3);         // more
  CHECK(r.ask(0, 96, give) == 0 && asked == 3);
  rc = 7;
  CHECK(r.ask(2, 96, give) == 7 && r.ask(2, 96, give) == 7 && asked == 5);
  rc = 0;
  CHECK(r.ask(2, 96, give) == 0 && asked == 6 && r.ask(2, 96, give) == 0 && asked == 6);
  CHECK(r.ask(64, 96, give) == 0 && r.ask(64, 96, give) == 0 && r.ask(-1, 96, give) == 0 && asked == 9);
  IxtLdsRoom t;
  std::atomic<int> n{0};
  std::vector<std::thread> threads;
  for (int i = 0; i < 8; ++i) threads.emplace_back([&, i] { for (int k = 1; k <= 1000; ++k) t.ask(i & 1, (size_t)k, [&] { ++n; return 0; }); });
  for (auto& x : threads) x.join();
  CHECK(n >= 2000 && t.ask(0, 1000, give) == 0 && t.ask(1, 1000, give) == 0 && asked == 9);
  std::printf("ok\n");
  return 0;
}
"""


def test_room_is_asked_for_on_every_device(tmp_path):
  cxx = shutil.which("g++") or shutil.which("c++")
  if cxx is None:
    pytest.skip("no host C++ compiler")
  src, exe = tmp_path / "room.cpp", tmp_path / "room"
  src.write_text(PROGRAM)
  subprocess.check_call([cxx, "-std=c++17", "-O1", "-Wall", "-pthread", "-I", build.CSRC, str(src), "-o", str(exe)])
  out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
  assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout


def test_no_launch_keeps_a_flag_for_all_devices():
  for path in glob.glob(os.path.join(build.CSRC, "*")):
    with open(path, encoding="utf-8") as f:
      text = f.read()
    calls = len(re.findall(r"hipFuncSetAttribute\(", text))
    assert calls == (1 if os.path.basename(path) == "ixt_device.h" else 0), (path, calls)
