"""The local sort's sizes and decisions, which need no GPU: the functions that the
kernels and their launch code use (radix_sort_local_rules.hpp), in a build for
the CPU."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KINDS = [(4, 0), (8, 0), (4, 4), (8, 8)]  # bytes of a key and of a value


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rules") / "librules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-o", out,
                    os.path.join(ROOT, "tests", "cpp", "local_sort_rules.cpp")], check=True)
    lib = ctypes.CDLL(out)
    lib.rule_codes.argtypes = [ctypes.c_int32, ctypes.c_uint64, ctypes.c_uint64, ctypes.c_uint64,
                               ctypes.c_int32]
    lib.rule_codes.restype = ctypes.c_uint32
    return lib


@pytest.mark.parametrize("size", [4, 8])
def test_bins_lie_in_the_stage(rules, size):
    """The bins of a window's keys, and what stands for lanes that hold none: keys behind the
    window's last whole run, and zeros behind the input (0 - low, the largest numbers)."""
    stage = rules.rule_stage_bytes()
    largest = (1 << 8 * size) - 1
    rng = np.random.default_rng(size)
    spans = [0, 1, 2, (1 << 15) - 1, (1 << 18) - 1, 1 << 18, largest >> 1, largest - 1]
    spans += [int(s) for s in rng.integers(0, largest, 200, dtype=np.uint64)]
    outside = 0
    for span in spans:
        inside = sorted([0, span, span // 2, span // 3])
        offsets = []
        for key in inside:
            codes = rules.rule_codes(size, span, key, span - key, 3)
            offsets += [codes & 0xFFFF]
            assert (codes & 0xFFFF) // 4 * 4 + 4 <= stage and (codes >> 16) // 4 * 4 + 4 <= stage
        assert offsets == sorted(offsets)  # larger keys are in later bins
        for key in (span + 1, span + 1 + span // 2, 2 * span + 1, largest):
            if not span < key <= largest:
                continue
            raw = rules.rule_codes(size, span, key, key, 3)
            outside += (raw & 0xFFFF) // 4 * 4 + 4 > stage
            for has_key in (0, 1, 2):
                codes = rules.rule_codes(size, span, key, key, has_key)
                for which in (0, 1):
                    if not has_key >> which & 1:
                        assert (codes >> 16 * which & 0xFFFF) // 4 * 4 + 4 <= stage
    assert outside > 0  # numbers that nothing may be read at
