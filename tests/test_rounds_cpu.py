"""How many tiles of prompt attention go by a launch of their own (csrc/ixt_rounds.h), built for the host by itself: whole units, half a round of blocks at most, and nothing behind whole rounds
stays in the launch that they leave -- a unit too few keeps its last round and pays for the other launches, too."""
import shutil
import subprocess

import pytest

import helpers as H

build = H.importlib.import_module("maxtext-indextts2_amd.build")

PROGRAM = r"""
#include "ixt_rounds.h"
#include <cstdio>
#define CHECK(x) do { if (!(x)) { std::printf("%s: %d tiles, %d heads, units of %d, %d keys\n", #x, tiles, heads, unit, keys); return 1; } } while (0)
int main() {
  for (int unit = 1; unit <= 4; unit *= 2)
    for (int heads = 1; heads <= 300; ++heads)
      for (int tiles = 1; tiles <= 300; ++tiles)
        for (int keys = 0; keys <= 3000; keys += 1000) {
          const int over = tiles_split(tiles, heads, unit, keys), blocks = tiles * heads;
          CHECK(over >= 0 && over <= tiles && (over % unit == 0 || over == tiles) && over * heads <= IXT_CUS / 2);
          CHECK((over == tiles) == (blocks <= IXT_CUS / 2));
          if (over == 0 || over == tiles) continue;
          CHECK(keys == 3000 && blocks % IXT_CUS != 0);
          CHECK(((tiles - over) * heads + IXT_CUS - 1) / IXT_CUS == blocks / IXT_CUS);
        }
  std::printf("ok\n");
  return 0;
}
"""


def test_what_is_split_takes_a_round_away(tmp_path):
  cxx = shutil.which("g++") or shutil.which("c++")
  if cxx is None:
    pytest.skip("no host C++ compiler")
  src, exe = tmp_path / "rounds.cpp", tmp_path / "rounds"
  src.write_text(PROGRAM)
  subprocess.check_call([cxx, "-std=c++17", "-O1", "-Wall", "-I", build.CSRC, str(src), "-o", str(exe)])
  out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
  assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
