"""Launches with more than 64 KB of dynamic LDS: every kernel has been allowed that much first.

Runs without a GPU: a small library stands in front of the HIP runtime's launch calls and writes down, in a
process of its own, which kernels were allowed how much and which were launched with it."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

from replisense_rfq_amd import _build

FRONT = r"""
#include <cstddef>
#include <map>
struct D { unsigned x, y, z; };
static std::map<const void*, int> allowed;
static D grid_, block_;
static size_t lds_;
static int launches_, bad_;
extern "C" {
int hipFuncSetAttribute(const void* f, int, int value) { allowed[f] = value; return 0; }
int __hipPushCallConfiguration(D g, D b, size_t lds, void*) { grid_ = g; block_ = b; lds_ = lds; return 0; }
int __hipPopCallConfiguration(D* g, D* b, size_t* lds, void** s) { *g = grid_; *b = block_; *lds = lds_; *s = nullptr; return 0; }
int hipLaunchKernel(const void* f, D, D, void**, size_t lds, void*) {
  ++launches_;
  bad_ += lds > 65536 && (size_t)allowed[f] < lds;
  return 0;
}
int launches() { return launches_; }
int bad() { return bad_; }
}
"""

RUN = """
import ctypes, subprocess, sys
front = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import torch
torch.ops.load_library(sys.argv[2])
lib = ctypes.CDLL(sys.argv[2])
name = next(w for w in subprocess.run(["nm", "-D", "--defined-only", sys.argv[2]], capture_output=True, text=True).stdout.split()
            if w.startswith("_ZN6rfqmix24launch_attn_keep_streams"))
p, i, l, f, b = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_bool
fn = lib[name]
fn.restype = None
fn.argtypes = [p, p, l, p, i, p, p, p, i, i, i, p, p, l, i, p, l, f, i, i, b, i, i, f, f, p, p]
for sigmoid in (False, True):
    for softcap in (0.0, 20.0):
        fn(None, None, 576, None, 22, None, None, None, 4, 4, 2, None, None, 0, 1, None, 32 * 512, 0.1, 0, 0, sigmoid,
           32, 1, softcap, 1.0, None, None)
print("launches", front.launches(), "bad", front.bad())
"""


@pytest.mark.skipif(shutil.which("g++") is None or shutil.which("nm") is None, reason="needs g++ and nm")
def test_streams_launches_are_allowed_their_lds(tmp_path):
    src, so = tmp_path / "front.cpp", tmp_path / "front.so"
    src.write_text(FRONT)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", str(src), "-o", str(so)], check=True)
    if not _build.MIX_SO.exists():
        _build.build_mix_kernels()
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(RUN), str(so), str(_build.MIX_SO)], capture_output=True,
                       text=True, timeout=300, cwd=os.path.dirname(_build.PKG_DIR))
    assert r.returncode == 0, r.stderr[-2000:]
    assert r.stdout.split()[-4:] == ["launches", "8", "bad", "0"], r.stdout
