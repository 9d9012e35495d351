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
    lib.rule_draws.argtypes = [ctypes.c_int64, ctypes.c_void_p, ctypes.c_void_p]
    lib.rule_limits.argtypes = [ctypes.c_int64, ctypes.c_int32, ctypes.c_int32, ctypes.c_void_p]
    return lib


class Limits(ctypes.Structure):
    _fields_ = [(name, ctypes.c_uint32) for name in
                ("draw_bits", "bin_bits", "parts", "max_equal", "max_pairs", "max_draws", "max_run")]


def draws_of(rules, n):
    """The places of n keys that are drawn, in the order in which the draws are kept."""
    places, slots = np.zeros(1 << 16, np.uint64), np.zeros(1 << 16, np.uint32)
    m = rules.rule_draws(n, places.ctypes.data, slots.ctypes.data)
    assert sorted(slots[:m]) == list(range(m))
    kept = np.zeros(m, np.uint64)
    kept[slots[:m]] = places[:m]
    return kept


def two_digits_are_enough(rules, n, key_bytes, value_bytes, keys_at):
    """What the draws say of keys in their ordered form: the same questions with numpy."""
    limits = Limits()
    rules.rule_limits(n, key_bytes, value_bytes, ctypes.addressof(limits))
    assert limits.max_run == 0 and limits.max_pairs > 0
    keys = keys_at(draws_of(rules, n))
    differ = int(np.bitwise_or.reduce(keys[: rules.rule_chunk_draws()] ^ keys[0]))
    top = (differ.bit_length() - 1) // 8
    if top < 3:
        return False
    prefixes = (keys[: rules.rule_prefix_draws()] >> keys.dtype.type(8 * (top - 1))) & keys.dtype.type(0xFFFF)
    counts = np.bincount(prefixes.astype(np.int64), minlength=1 << 16)
    return counts.max() <= limits.max_draws and (counts * (counts - 1) // 2).sum() <= limits.max_pairs


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


def test_every_chunk_of_draws_is_from_all_over_the_input(rules):
    for n in (1 << 14, (1 << 21) + 1, (1 << 23) + 1, (1 << 25) + 1, 1 << 28, (1 << 31) - 1):
        places = draws_of(rules, n)
        assert places.max() < n and places.size <= n
        assert np.unique(places).size == places.size
        for chunk in places.reshape(-1, min(places.size, rules.rule_chunk_draws())):
            in_64_parts = np.bincount((chunk * np.uint64(64) // np.uint64(n)).astype(np.int64), minlength=64)
            # (A part of the input that is no whole number of elements may give its draw to the next 64th.)
            assert np.abs(in_64_parts - chunk.size // 64).max() <= 2


@pytest.mark.parametrize("n,key_bytes,value_bytes", [
    (1 << 23, 4, 0), ((1 << 25) + 1, 4, 0), (1 << 28, 4, 0), (1 << 26, 4, 4), ((1 << 25) + 1, 8, 0), (1 << 27, 8, 4)])
def test_columns_whose_parts_differ_are_refused_by_the_draws(rules, n, key_bytes, value_bytes):
    """Uniform keys are taken; with a part of the input that is all one value, wherever it
    lies and whatever the value, they are not (a hundredth is ten windows and more here)."""
    kind = np.dtype(f"uint{8 * key_bytes}").type
    largest = (1 << 8 * key_bytes) - 1

    def uniform(places):
        return np.random.default_rng(7).integers(0, largest, places.size, dtype=kind, endpoint=True)

    assert two_digits_are_enough(rules, n, key_bytes, value_bytes, uniform)
    for value in [largest, largest >> 1, largest // 3, 0, 1, 0x3F800000]:
        for first, last in [(0.5, 1), (0, 0.5), (0.75, 1), (0.3, 0.4), (0.9, 1), (0.99, 1), (0, 0.01)]:
            def padded(places):
                return np.where((places >= int(first * n)) & (places < int(last * n)), kind(value), uniform(places))
            assert not two_digits_are_enough(rules, n, key_bytes, value_bytes, padded), (value, first, last)


@pytest.mark.parametrize("n", [18_433, 300_000, 2_000_000, 3_000_000, 10_000_019, 1 << 25, 1 << 26, 1 << 28])
@pytest.mark.parametrize("key_bytes", [4, 8])
def test_columns_of_many_copies_are_refused_by_the_draws(rules, n, key_bytes):
    """Of the draws of the parts of the values that are asked, those that meet an earlier one in
    their bin, for 20 columns of each kind: different keys are taken, and from eight copies of every value on, when
    most windows have a bin of sixteen keys, they are not; long columns of 4-byte keys, where the most draws are
    and the least is saved, from four on."""
    limits = Limits()
    rules.rule_limits(n, key_bytes, 0, ctypes.addressof(limits))
    kind = np.dtype(f"uint{8 * key_bytes}").type
    bins = kind(8 * key_bytes - limits.bin_bits)
    share = limits.parts / rules.rule_parts(limits.draw_bits)
    rng = np.random.default_rng(n)

    def mixed(x):  # a random number for each
        x = (x + np.uint64(1)) * np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ x >> np.uint64(30)) * np.uint64(0xBF58476D1CE4E5B9)
        return x ^ x >> np.uint64(29)

    taken = {0: 0, 8: 0, **({4: 0} if key_bytes == 4 and n >= 1 << 26 else {})}
    for copies in taken:
        for _ in range(20):
            m = 1 << limits.draw_bits
            values = n // copies if copies else 1 << 63
            keys = mixed(rng.integers(0, values, m, dtype=np.uint64)) >> np.uint64(64 - 8 * key_bytes)
            in_bins = keys.astype(kind) >> bins
            asked = in_bins[(mixed(in_bins.astype(np.uint64)) >> np.uint64(40)) < share * (1 << 24)]
            taken[copies] += asked.size - np.unique(asked).size <= limits.max_equal
    assert taken[0] >= 19 and taken[8] <= 1 and taken.get(4, 0) <= 2, taken


@pytest.mark.parametrize("key_bytes,value_bytes", KINDS)
def test_counts_of_two_digits_bound_a_run(rules, key_bytes, value_bytes):
    """The digits' counts of uniform keys pass, with the scatter of 256 of them, as far as the draws let uniform
    keys pass (runs of 0.6 windows); a run of two windows and of n / 2000 keys more does not, nor does
    a digit whose runs are all longer than a window."""
    window = rules.rule_window(key_bytes, value_bytes)
    rng = np.random.default_rng(5)
    for n in (window * 240 + 1, 1 << 23, 1 << 25, int(0.6 * window * 65536)):
        for _ in range(20):
            upper, lower = rng.multinomial(n, [1 / 256] * 256, 2)
            assert rules.rule_counts_allow(n, int(upper.max()), int(lower.max()), window)
            run = 2 * window + n // 2000
            assert not rules.rule_counts_allow(n, int(upper[0]) + run, int(lower[0]) + run, window)
    assert not rules.rule_counts_allow(1 << 30, 256 * window + 1, (1 << 30) // 256, window)
