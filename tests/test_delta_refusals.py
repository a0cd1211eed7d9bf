"""Sizes and empty calls that the delta rule's one-launch kernels leave to the two kernels: decided
on the host, ahead of any launch, so that no GPU is needed.  In a process of its own: a fault there
would end it."""
import json
import subprocess
import sys

import pytest

CALL = """
import ctypes, json, sys
import torch  # libraries of the extension
from omnia_amd.ops import _omnia_kernels as ext
name, args = json.loads(sys.argv[1])
null, wide = ctypes.c_void_p(None), ctypes.c_int64
f = getattr(ctypes.CDLL(ext.__file__), name)
conv = {"p": lambda v: null, "l": wide, "f": ctypes.c_float, "i": ctypes.c_int}
print(f(*[conv[t](v) for t, v in args]))
"""


def call(name, *args):
    pytest.importorskip("omnia_amd.ops._omnia_kernels")
    p = subprocess.run([sys.executable, "-c", CALL, json.dumps([name, args])], capture_output=True,
                       text=True, timeout=300)
    assert p.returncode == 0, (p.returncode, p.stderr[-500:])
    return int(p.stdout.split()[-1])


def ints(*v):
    return [("i", x) for x in v]


P = ("p", 0)


def step_conv(T, KH, H, D, V, Vs, taps=4):
    return call("omnia_delta_step_conv", P, P, P, P, ("i", 0), ("l", 4096), P, P, P, P, P, P,
                *ints(T, KH, H, D, V, Vs, Vs, taps), ("f", 1e-6), P)


# states wider than a block of threads (no row group is left): for the two kernels; of no columns:
# an error
@pytest.mark.parametrize("D,V,Vs,rc", [(64, 1028, 1028, -3), (64, 128, 1028, -3), (8, 4, 4096, -3),
                                       (64, 0, 0, -1)])
def test_step_of_wide_states(D, V, Vs, rc):
    assert step_conv(1, 1, 1, D, V, Vs) == rc


def prep_blocks(T, nseq, KH, H, D, V, taps=4):
    return call("omnia_delta_prep_blocks", P, P, P, P, P, ("i", 0), ("l", 4096), P, P, P, P, P,
                ("i", nseq), P, P, *ints(T, KH, H, D, -(-D // 4) * 4, V, taps), P)


# no rows or no sequences: done only where rows of these sizes would be (the scan then expects records)
@pytest.mark.parametrize("T,nseq", [(0, 3), (0, 0)])
@pytest.mark.parametrize("D,KH,H,taps,rc", [(320, 1, 1, 4, -3), (64, 1, 4, 4, -3), (64, 1, 1, 5, -3),
                                            (64, 1, 2, 4, 0)])
def test_preparation_of_no_rows(T, nseq, D, KH, H, taps, rc):
    assert prep_blocks(T, nseq, KH, H, D, 64, taps) == rc
