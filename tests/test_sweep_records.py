"""Published records of the sync-free sweep lie on 16-byte boundaries.

k_sweep_async polls a record with 16-byte loads and takes a 64-bit word that
no longer reads pending as final.  That holds for words of aligned pieces: a
16-byte load at an odd multiple of 8 bytes may straddle two cache lines.  The
record of each slot, of pub (FP64 and mixed) and of the copy sources' dsrc,
is laid out by kRecord (preprocess.h); the fixtures with supersonic points
(test_gpu_branches.py) run the copies on the GPU.
"""

import ctypes as C
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "3d-mfcfd_amd", "csrc")
SHIM = """
#include "%s/preprocess.h"
extern "C" int record_doubles(int is_float) { return is_float ? mfcfd::kRecord<float> : mfcfd::kRecord<double>; }
""" % CSRC


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    d = tmp_path_factory.mktemp("records")
    src, so = str(d / "records.cpp"), str(d / "librecords.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.run(["g++", "-O1", "-fPIC", "-std=c++17", "-shared", "-o", so, src], check=True)
    return C.CDLL(so)


# (record of floats, bytes of its five values, bytes of the pieces loaded)
@pytest.mark.parametrize("is_float,words,pieces", [(0, 5, (16, 16, 8)), (1, 3, (16, 8))])
def test_every_piece_of_every_record_is_aligned(lib, is_float, words, pieces):
    stride = 8 * lib.record_doubles(is_float)
    assert sum(pieces) == 8 * words <= stride
    for slot in range(33):
        at = slot * stride
        for size in pieces:
            assert at % size == 0
            assert at // 64 == (at + size - 1) // 64
            at += size
        assert slot * stride // 64 == (at - 1) // 64


def test_records_are_addressed_by_the_layout_alone():
    """The kernels index pub and dsrc through record() only; the marks fill both whole."""
    code = "\n".join(line.split("//")[0] for line in open(os.path.join(CSRC, "kernels_sweep.hip")))
    for name in ("a.pub", "a.dsrc"):
        uses = code.count(name)
        marks = code.count(f"reinterpret_cast<u64x2*>({name})[")
        records = code.count(f"record<T>({name}, ") + code.count(f"record<double>({name}, ")
        assert marks == 1 and records >= 2 and marks + records == uses, name
