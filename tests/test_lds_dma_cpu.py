"""The hand-issued LDS-DMA (csrc/ixt_device.h, lds_dma16) in the code that the compiler makes of the kernels that use it: a write of M0 stands at least one
wait state in front of the fetch, and a scalar register that a vector instruction wrote at least five in front of a fetch that addresses with it.  The
compiler keeps these distances for its own instructions and does not look into asm."""
import importlib
import os
import re
import subprocess

import pytest

build = importlib.import_module("maxtext-indextts2_amd.build")
RING = """#include "ixt_kernels.h"
#include "ixt_gemm.h"
template __global__ void k_gemm_ring<2, 4, 4, 2, 2, 4, GEPI_F32, 0, false, false>(const u32x4*, const u32x4*, int, int, int, int, int, int, GemmEpi);
template __global__ void k_gemm_ring<4, 1, 1, 1, 4, 6, GEPI_QKV, 0, false, false>(const u32x4*, const u32x4*, int, int, int, int, int, int, GemmEpi);
template __global__ void k_gemm_ring<2, 2, 2, 2, 2, 4, GEPI_UNEMBED, 0, false, true>(const u32x4*, const u32x4*, int, int, int, int, int, int, GemmEpi);
"""
TRAIN = """#include "ixt_train_gemm.h"
template __global__ void k_tgemm<true, true, 2, 2, 2, 2, 4, true>(TGemm);
template __global__ void k_tgemm<false, false, 8, 4, 2, 4, 4, false>(TGemm);
"""
MID = """#include "ixt_mid.h"
template __global__ void k_mid<2>(MidArgs);
template __global__ void k_mid<3>(MidArgs);
template __global__ void k_mid<4>(MidArgs);
"""


def _registers(operand):
  m = re.match(r"s\[(\d+):(\d+)\]$|s(\d+)$", operand)
  return set() if not m else set(range(int(m[1]), int(m[2]) + 1)) if m[1] else {int(m[3])}


def _distances(asm):
  """(fetches, least distance of M0's write, of a vector instruction's write of the address) in wait states."""
  behind, fetches, m0, address = [], 0, [], []
  for line in asm.splitlines():
    text = line.split(";")[0].strip()
    if re.match(r"^[\w$]+:$", text):                                     # (a kernel's entry; its own labels start with a dot)
      behind = []
    if not text or text.startswith(".") or text.endswith(":"):
      continue
    op, *rest = text.split(None, 1)
    args = [a.split()[0] for a in rest[0].split(",") if a.strip()] if rest else []
    if "load_lds" in op:
      fetches += 1
      uses, states, found = set().union(*(_registers(a) for a in args)), 0, False
      for was, to in reversed(behind[-16:]):
        if not found and was.startswith("s_") and to and to[0] == "m0":
          found = True
          m0.append(states)
        if was.startswith("v_") and to and _registers(to[0]) & uses:
          address.append(states)
        states += int(to[0], 0) + 1 if was == "s_nop" else 1
    behind.append((op, args))
  return fetches, min(m0, default=None), min(address, default=99)


def test_the_scan_sees_both():
  near = "k:\n v_readlane_b32 s4, v1, 0\n s_mov_b32 m0, s2\n global_load_lds_dwordx4 v4, s[4:5]\n"
  assert _distances(near) == (1, 0, 1)
  assert _distances(near.replace(" global", " s_nop 3\n global")) == (1, 4, 5)


@pytest.mark.parametrize("source", [RING, TRAIN, MID], ids=["ring", "train", "mid"])
def test_wait_states(source, tmp_path):
  if not os.path.exists(build.hipcc()):
    pytest.skip("no hipcc here")
  (tmp_path / "k.hip").write_text(source)
  out = tmp_path / "k.s"
  done = subprocess.run([build.hipcc()] + build.HIPCC_FLAGS + ["-I", build.CSRC, "-S", "--offload-device-only", str(tmp_path / "k.hip"), "-o", str(out)], capture_output=True, text=True, timeout=300)
  assert done.returncode == 0, done.stderr
  assert "inline-asm" not in done.stderr
  fetches, m0, address = _distances(out.read_text())
  assert fetches > 20 and m0 is not None and m0 >= 1 and address >= 5, (fetches, m0, address)


def test_barriers_order_the_reads_behind_them():
  """The barrier builtin is no memory operation to the compiler: kernels use lds_barrier, which adds the fence."""
  bare = [n for n in sorted(os.listdir(build.CSRC)) if n != "ixt_device.h" and "__builtin_amdgcn_s_barrier" in open(os.path.join(build.CSRC, n), encoding="utf-8").read()]
  with open(os.path.join(build.CSRC, "ixt_device.h"), encoding="utf-8") as f:
    body = re.search(r"void lds_barrier\(\) \{(.*?)\n\}", f.read(), re.S)
  assert bare == [] and body and re.search(r's_barrier\(\);\s*asm volatile\("" ::: "memory"\);', body[1])


def test_wide_stores_are_followed_by_a_wait_state():
  """A store of more than 8 bytes still reads its registers when the next instruction issues; the compiler keeps a vector instruction that writes them away from its
  own stores and does not look into asm."""
  found = 0
  for n in sorted(os.listdir(build.CSRC)):
    with open(os.path.join(build.CSRC, n), encoding="utf-8") as f:
      for text in re.findall(r'asm(?: volatile)?\s*\(\s*"((?:[^"\\]|\\.)*)"', f.read()):
        for at in re.finditer(r"(?:global|buffer|flat)_store_dwordx[34]", text):
          found += 1
          assert re.search(r"\\n\\ts_nop \d", text[at.end():]), (n, text)
  assert found > 0


def test_no_load_of_memory_into_registers_in_asm():
  """The compiler takes the registers of such a load as written at once: a copy of one, or another use of it, may come ahead of the wait."""
  for n in sorted(os.listdir(build.CSRC)):
    with open(os.path.join(build.CSRC, n), encoding="utf-8") as f:
      for text in re.findall(r'asm(?: volatile)?\s*\(\s*"((?:[^"\\]|\\.)*)"', f.read()):
        assert not re.search(r"(?:global|buffer|flat|scratch)_load_(?!lds)", text), (n, text)


def test_no_vector_arithmetic_in_asm():
  """A matrix product's result may be read only some wait states behind it; the compiler keeps them for the instructions that it knows, and in asm knows none."""
  for n in sorted(os.listdir(build.CSRC)):
    with open(os.path.join(build.CSRC, n), encoding="utf-8") as f:
      for text in re.findall(r'asm(?: volatile)?\s*\(\s*"((?:[^"\\]|\\.)*)"', f.read()):
        assert not re.search(r"\bv_\w+", text), (n, text)
