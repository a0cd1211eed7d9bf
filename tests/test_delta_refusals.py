"""Sizes and empty calls that the delta rule's one-launch kernels leave to the two kernels: decided
on the host, ahead of any launch, so that no GPU is needed.  In a process of its own, which sees no
GPU: a fault there would end it."""
import json
import os
import subprocess
import sys

import pytest

CALLS = """
import ctypes, json, sys
import torch  # libraries of the extension
from omnia_amd.ops import _omnia_kernels as ext
name, calls = json.loads(sys.argv[1])
conv = {"p": lambda v: ctypes.c_void_p(None), "l": ctypes.c_int64, "f": ctypes.c_float,
        "i": ctypes.c_int}
f = getattr(ctypes.CDLL(ext.__file__), name)
for args in calls:
    print(f(*[conv[t](v) for t, v in args]), flush=True)
"""
P = ("p", 0)


def results(name, calls):
    """What the entry point returns for each of the calls."""
    pytest.importorskip("omnia_amd.ops._omnia_kernels")
    env = os.environ | {"HIP_VISIBLE_DEVICES": "-1", "ROCR_VISIBLE_DEVICES": ""}
    p = subprocess.run([sys.executable, "-c", CALLS, json.dumps([name, calls])], env=env,
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, (p.returncode, p.stdout.split(), p.stderr[-500:])
    return [int(x) for x in p.stdout.split()[-len(calls):]]


def ints(*v):
    return [("i", x) for x in v]


def step_conv(T, KH, H, D, V, Vs, taps=4):
    return [P, P, P, P, ("i", 0), ("l", 4096), P, P, P, P, P, P, *ints(T, KH, H, D, V, Vs, Vs, taps),
            ("f", 1e-6), P]


def test_rows_left_to_two_kernels():
    """-3: states wider than a block of threads (no row group is left); heads past two a key head;
    states of 8 rows a thread at the ends of their rule.  -1: states of no columns."""
    sizes = [(1, 1, 1, 64, 1028, 1028), (1, 1, 1, 64, 128, 1028), (1, 1, 1, 8, 4, 4096),
             (64, 4, 16, 128, 128, 128), (1, 1, 3, 128, 128, 128), (97, 8, 16, 128, 64, 64),
             (112, 8, 16, 64, 128, 128), (1, 1, 1, 64, 0, 0)]
    got = results("omnia_delta_step_conv", [step_conv(*s) for s in sizes])
    assert got == [-3] * (len(sizes) - 1) + [-1]


def prep_blocks(T, nseq, KH, H, D, V, taps):
    return [P, P, P, P, P, ("i", 0), ("l", 4096), P, P, P, P, P, ("i", nseq), P, P,
            *ints(T, KH, H, D, -(-D // 4) * 4, V, taps), P]


def test_preparation_of_no_rows():
    """No rows or no sequences: done (0) only where rows of these sizes would be, since the scan then
    expects records."""
    sizes = [(1, 1, 320, 64, 4), (1, 4, 64, 64, 4), (1, 1, 64, 64, 5), (1, 2, 64, 64, 4)]
    got = results("omnia_delta_prep_blocks",
                  [prep_blocks(0, nseq, *s) for nseq in (3, 0) for s in sizes])
    assert got == [-3, -3, -3, 0] * 2


def test_preparation_in_two_rounds():
    """-3 past two blocks a CU where many sequences are short, and past 640 blocks."""
    sizes = [(33 * 16, 33), (2 * 60, 60), (24 * 31, 24), (1264 + 16, 1), (8 * 1000, 8)]
    got = results("omnia_delta_prep_blocks", [prep_blocks(T, n, 8, R * 8, 128, 128, 4)
                                              for R in (1, 2) for T, n in sizes])
    assert got == [-3] * 10
