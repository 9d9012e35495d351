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
    lib.rule_blocks.argtypes = [ctypes.c_int64, ctypes.c_int64]
    lib.rule_blocks.restype = ctypes.c_int64
    lib.rule_deferred.argtypes = [ctypes.c_uint32, ctypes.c_uint32]
    lib.rule_deferred.restype = ctypes.c_uint32
    lib.rule_deferred_bytes.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_uint32]
    lib.rule_deferred_bytes.restype = ctypes.c_int64
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


@pytest.mark.parametrize("key_bytes,value_bytes", KINDS)
def test_a_block_has_room_to_put_off_all_of_its_windows(rules, key_bytes, value_bytes):
    """Windows of whole runs, as a block takes them, for runs that waste the most of a window."""
    window = rules.rule_window(key_bytes, value_bytes)
    rng = np.random.default_rng(key_bytes)
    for part in (1024, window - 1, window, window + 1, 7 * window // 2, 20 * window, 262_144):
        for pattern in ([window // 2 + 1], [1, window], [window], [window + 1], [1, window + 1], [1],
                        [window - 1, 2], list(rng.integers(1, 2 * window, 40))):
            runs, total = [], 0
            while total < part:  # all that start in the part
                runs.append(int(pattern[len(runs) % len(pattern)]))
                total += runs[-1]
            windows, i = 0, 0
            while i < len(runs):
                held = 0
                while i < len(runs) and held + runs[i] <= window:
                    held += runs[i]
                    i += 1
                i += held == 0  # a run longer than a window
                windows += 1
            assert windows <= rules.rule_deferred(part, window)


@pytest.mark.parametrize("key_bytes,value_bytes", KINDS)
def test_what_is_put_off_fits_the_status_words(rules, key_bytes, value_bytes):
    """1 KiB of status per tile and pass, with the longest tiles there are."""
    window = rules.rule_window(key_bytes, value_bytes)
    tile = 1024 * (36 if value_bytes == 0 else 20) // (key_bytes // 4)
    for n in (1 << 14, 18_433, 100_003, 1 << 20, (1 << 22) + 1, 1 << 24, 1 << 28, (1 << 31) - 1):
        for cus in (1, 32, 64, 256, 304, 1024):
            blocks = rules.rule_blocks(n, cus)
            assert rules.rule_deferred_bytes(n, blocks, window) <= key_bytes * 1024 * -(-n // tile)
