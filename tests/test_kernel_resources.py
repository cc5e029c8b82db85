"""Register budget of the compiled kernels, read from the metadata of the library's gfx950 code objects.

A kernel that spills keeps a scratch allocation per lane (`.private_segment_fixed_size` in the code object's
kernel metadata, the figure hipcc prints as ScratchSize under -Rpass-analysis=kernel-resource-usage): every tile's
accumulators then make a round trip through memory, and a launch pays for the scratch set-up. No kernel of the
library may have one.
"""

import os
import re
import shutil
import subprocess

import pytest

from tokamax_amd import _lib

LLVM = "/opt/rocm/llvm/bin"
TOOLS = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf", "llvm-objdump")]
TARGET = "hipv4-amdgcn-amd-amdhsa--gfx950"


def _code_objects(tmp_path):
  """The gfx950 code objects bundled into the library, one per source file."""
  fat = tmp_path / "fatbin"
  subprocess.run([TOOLS[0], "-O", "binary", "--only-section=.hip_fatbin", _lib.LIB_PATH, str(fat)], check=True)
  blob = fat.read_bytes()
  starts = [m.start() for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", blob)]  # one bundle per source file
  codes = []
  for n, first in enumerate(starts):
    part, code = tmp_path / f"bundle{n}", tmp_path / f"bundle{n}.co"
    part.write_bytes(blob[first:starts[n + 1] if n + 1 < len(starts) else len(blob)])
    subprocess.run([TOOLS[1], "--unbundle", "--type=o", f"--input={part}", f"--targets={TARGET}", f"--output={code}"], check=True)
    codes.append(code)
  return codes


def _kernel_metadata(tmp_path):
  """[(mangled kernel name, scratch bytes per lane, vgprs)] over every code object bundled into the library."""
  rows = []
  for code in _code_objects(tmp_path):
    notes = subprocess.run([TOOLS[2], "--notes", str(code)], check=True, capture_output=True, text=True).stdout
    name = scratch = None
    for line in notes.splitlines():
      if m := re.match(r"\s+\.name:\s+(\S+)", line):
        name = m.group(1)
      elif m := re.match(r"\s+\.private_segment_fixed_size:\s+(\d+)", line):
        scratch = int(m.group(1))
      elif m := re.match(r"\s+\.vgpr_count:\s+(\d+)", line):
        rows.append((name, scratch, int(m.group(1))))
  return rows


@pytest.mark.skipif(not all(os.path.exists(t) for t in TOOLS), reason="ROCm's LLVM tools are not installed")
def test_no_kernel_of_the_library_uses_scratch_memory(tmp_path):
  assert os.path.exists(_lib.LIB_PATH), "build the library first"
  rows = _kernel_metadata(tmp_path)
  names = [r[0] for r in rows]
  # every source file's kernels were seen: the tiled GEMM entries (plain, quantising, split last round), the
  # streaming small-m kernels and their persistent form, the scheduler
  for piece in ("gemm_entry", "gemm_entry_fp8_out", "gemm_entry_split", "decode_kernel", "decode_persistent_kernel", "schedule"):
    assert any(piece in n for n in names), piece
  assert len(rows) >= 200
  # (The fp8 256 x 256 x 128 tile, 32-byte fragments next to 128 accumulators, keeps a few lane constants of the loops
  # that drain the pipeline in scratch, written and read once per tile, outside the steady-state loop.)
  # (Likewise the two tiles on one row of waves of packed int4 weights with scales per k-block: the 256-row one keeps
  # eight lhs fragments double-buffered next to 128 accumulators, the 128-row one lives in 128 registers so that two
  # workgroups share a CU; five to seven lane constants, stored before the k loop and reloaded after it.)
  # (And the 128 x 256 x 128 tile on one row of waves of fp8 activations over packed int4 weights with scales per k-block:
  # 64 accumulators, 64 partial ones and double-buffered 32-byte lhs fragments; eight lane constants, likewise stored
  # before the k loops and reloaded after them.)
  allowed = lambda name: (24 if "GemmKernelILi0ELi3ELi3ELi256ELi256ELi128E" in name else
                          24 if "GemmKernelILi4ELi1ELi5ELi256ELi256ELi64ELi1ELi8E" in name else
                          32 if "GemmKernelILi4ELi1ELi5ELi128ELi256ELi64ELi1ELi8E" in name else
                          32 if "GemmKernelILi4ELi3ELi5ELi128ELi256ELi128ELi1ELi8E" in name else 0)
  spilling = [(n, s) for n, s, _ in rows if s > allowed(n)]
  if spilling and shutil.which("c++filt"):
    spilling = [(subprocess.run(["c++filt", n], capture_output=True, text=True).stdout.strip(), s) for n, s in spilling]
  assert not spilling, spilling
  # the row quantiser is bound by HBM: the forms that hold a tile in registers leave room for four waves per SIMD
  rows_held = [(n, v) for n, _, v in rows if "quantize_rows_kernel" in n]
  assert rows_held and all(v <= 128 for _, v in rows_held), rows_held
  # the 8-wave tiles run two waves per SIMD: 256 registers each
  headline = [v for n, _, v in rows if "GemmKernelILi0ELi1ELi1ELi256ELi256ELi64ELi2ELi4E" in n]
  assert len(headline) >= 6 and max(headline) <= 256


@pytest.mark.skipif(not all(os.path.exists(t) for t in TOOLS), reason="ROCm's LLVM tools are not installed")
def test_matrix_instruction_of_16_bit_tiles(tmp_path):
  """16x16x32 MFMAs in the forward and dlhs tiles that keep two waves on a SIMD; 32x32x16 where a 4-wave workgroup has
  its CU to itself and in d rhs, which measured up to 30 % slower on the other form."""
  name = lambda mode, *tile: "GemmKernelILi%dELi1ELi1E" % mode + "".join(f"Li{t}E" for t in tile)
  wants = {name(0, 256, 256, 64, 2, 4, 2): "16x16x32", name(1, 128, 256, 64, 2, 4, 3): "16x16x32",
           name(0, 128, 128, 64, 2, 2, 2): "16x16x32", name(3, 128, 256, 64, 2, 4, 3): "16x16x32",
           name(0, 128, 256, 64, 2, 2, 3): "32x32x16", name(1, 128, 128, 64, 2, 2, 4): "32x32x16",
           name(3, 64, 256, 64, 2, 2, 3): "32x32x16", name(2, 128, 128, 64, 2, 2, 4): "32x32x16",
           name(2, 256, 256, 64, 2, 4, 2): "32x32x16"}
  seen = {}
  for code in _code_objects(tmp_path):
    symbols = subprocess.run([TOOLS[2], "--symbols", "--wide", str(code)], check=True, capture_output=True, text=True).stdout
    picked = [w.split()[-1] for w in symbols.splitlines() if "gemm_entryI" in w and not w.endswith(".kd")]
    for tile in wants:
      for symbol in picked:
        if tile in symbol:
          text = subprocess.run([TOOLS[3], "-d", f"--disassemble-symbols={symbol}", str(code)], check=True, capture_output=True, text=True).stdout
          seen[tile] = set(re.findall(r"v_mfma_f32_(\d+x\d+x\d+)_bf16", text))
  assert seen == {tile: {form} for tile, form in wants.items()}
