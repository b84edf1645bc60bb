"""Launches with more than 64 KB of dynamic LDS: every kernel has been allowed that much first.

Runs without a GPU: a small library stands in front of the HIP runtime's launch calls and writes down, in a
process of its own, which kernels were allowed how much and which were launched with it.  The same shows which kernel a step
goes to."""
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
static std::map<const void*, const char*> names;
static const char* last_ = "";
extern "C" {
int hipFuncSetAttribute(const void* f, int, int value) { allowed[f] = value; return 0; }
int __hipPushCallConfiguration(D g, D b, size_t lds, void*) { grid_ = g; block_ = b; lds_ = lds; return 0; }
int __hipPopCallConfiguration(D* g, D* b, size_t* lds, void** s) { *g = grid_; *b = block_; *lds = lds_; *s = nullptr; return 0; }
int hipLaunchKernel(const void* f, D, D, void**, size_t lds, void*) {
  ++launches_;
  last_ = names[f];
  bad_ += lds > 65536 && (size_t)allowed[f] < lds;
  return 0;
}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names[f] = name; }
const char* last() { return last_; }
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
    if not _build.MIX_SO.exists():
        _build.build_mix_kernels()
    out = _run(RUN, _front(tmp_path), _build.MIX_SO)
    assert out.split()[-4:] == ["launches", "8", "bad", "0"], out


def _front(tmp_path):
    src, so = tmp_path / "front.cpp", tmp_path / "front.so"
    src.write_text(FRONT)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", str(src), "-o", str(so)], check=True)
    return so


def _run(program, front, lib, **env):
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(program), str(front), str(lib)], capture_output=True,
                       text=True, timeout=300, cwd=os.path.dirname(_build.PKG_DIR), env={**os.environ, **env})
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout


DECODE = """
import ctypes, subprocess, sys
front = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
front.last.restype = ctypes.c_char_p
import torch
torch.ops.load_library(sys.argv[2])
lib = ctypes.CDLL(sys.argv[2])
name = next(w for w in subprocess.run(["nm", "-D", "--defined-only", sys.argv[2]], capture_output=True, text=True).stdout.split()
            if w.startswith("_ZN3rfq18launch_attn_decodeE"))
p, i, l, f, b = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_bool
fn = lib[name]
fn.restype = None
fn.argtypes = [p, l, p, p, p, i, p, p, p, i, p, p, i, i, p, l, p, p, i, i, f, i, i, p, p, b]
for seqs, items, rows, cols, splits in ((1, 1, 1, 40, 2), (8, 8, 8, 40, 2), (32, 32, 32, 20, 2), (64, 64, 64, 11, 2), (64, 64, 64, 300, 2),
                                        (2, 16, 16, 16, 8), (64, 80, 100, 20, 2), (8, 8, 8, 1, 1)):
    for tiles in (1, 2):
        fn(None, 4096, None, None, None, cols, None, None, None, seqs, None, None, items, rows, None, 4096, None, None, 32, 8, 0.1, splits,
           tiles, None, None, False)
        print(front.last().decode().split("rfq")[1].split("Ev")[0])
print("bad", front.bad())
"""


@pytest.mark.skipif(shutil.which("g++") is None or shutil.which("nm") is None, reason="needs g++ and nm")
def test_which_kernel_a_decode_step_goes_to(tmp_path):
    """attn_decode by its launches: waves by the items that the sequences can need, pages past the caches by the tables' room
    or RFQ_ATTN_NT=1, more rows than items and tables of one page to the general kernel, and all of them allowed their LDS."""
    if not _build.C_SO.exists():
        _build.build_kernels()
    front = _front(tmp_path)
    rows = "23attn_decode_rows_kernelILi%dELi%dELb%dEE"
    # waves by rows, or the items that the sequences can need: two sequences of sixteen rows, six of one tile, four of two
    want = [[(1, 0), (8, 0), (4, 0), (2, 0), (2, 1), (w, 0)] for w in (4, 8)]
    for nt in "", "1":
        out = _run(DECODE, front, _build.C_SO, RFQ_ATTN_NT=nt).split()
        for tiles in (1, 2):
            assert out[tiles - 1:12:2] == [rows % (w, tiles, past or nt == "1") for w, past in want[tiles - 1]], out
        assert all(x.startswith("18attn_decode_kernel") for x in out[12:16]) and out[16:] == ["bad", "0"], out
