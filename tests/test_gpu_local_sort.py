"""The local sort: passes over the topmost digits, then windows of whole runs in
LDS.  Against numpy's stable sort, bit for bit, at the lengths of runs and inputs
where another branch takes over."""
import numpy as np
import pytest

from ilgpu_amd import capi
from tests.test_gpu_parity import D, note, sync

pytestmark = pytest.mark.gpu


def order_bits(bits, dtype, descending, total_order):
    """The unsigned bits whose order the sort gives, for keys of these bits."""
    width = bits.dtype.itemsize * 8
    sign = bits.dtype.type(1 << (width - 1))
    kind = np.dtype(dtype).kind
    if kind == "u":
        out = bits
    elif kind == "i":
        out = bits ^ sign
    elif total_order:
        out = np.where(bits & sign, ~bits, bits ^ sign)
    else:  # as the reference writes it: the last bit of positive values is flipped
        out = bits ^ sign ^ (bits.dtype.type(1) - (bits >> bits.dtype.type(width - 1)))
    return ~out if descending else out


def check(bits, dtype, value_dtype=None, descending=False, total_order=False, from_index=True):
    """Sorts keys of these bits; the number of passes that ran."""
    n = bits.size
    expect = np.argsort(order_bits(bits, dtype, descending, total_order), kind="stable")
    keys = D.from_numpy(bits.view(dtype))
    size = 0 if value_dtype is None else np.dtype(value_dtype).itemsize
    temp = capi.temp_buffer(capi.radix_sort_temp_bytes(n, dtype, size))
    if value_dtype is None:
        capi.radix_sort_keys(keys, temp, descending=descending, float_total_order=total_order)
    else:
        places = np.arange(n).astype(value_dtype)
        values = D.zeros(n, value_dtype) if from_index else D.from_numpy(places)
        capi.radix_sort_pairs(keys, values, temp, descending=descending,
                              float_total_order=total_order, values_from_index=from_index)
    sync()
    assert np.array_equal(keys.numpy().view(bits.dtype), bits[expect])
    if value_dtype is not None:
        assert np.array_equal(values.numpy(), places[expect])
    return capi.radix_sort_passes(temp, n, dtype, size)[0]


def random_bits(n, width, seed):
    return np.random.default_rng(seed).integers(0, 1 << width, n, dtype=f"uint{width}", endpoint=False)


# A full window: keys of 4 bytes, of 8, and pairs of either with values of up to 8 bytes.
WINDOWS = {(4, False): 9216, (8, False): 4608, (4, True): 6144, (8, True): 3584}


@pytest.mark.parametrize("dtype,descending,total_order", [
    (np.uint32, False, False), (np.int32, True, False), (np.float32, False, False),
    (np.float32, True, True), (np.uint64, True, False), (np.int64, False, False),
    (np.float64, False, False), (np.float64, True, True)])
@pytest.mark.parametrize("value_dtype", [None, np.uint8, np.uint16, np.uint32, np.uint64])
def test_random_keys_take_one_or_two_passes(dtype, descending, total_order, value_dtype):
    """One pass up to 240 windows, two beyond; at both sides of that and at the shortest."""
    size = np.dtype(dtype).itemsize
    window = WINDOWS[size, value_dtype is not None]
    for n, passes in [(18433, 1), (100_003, 1), (240 * window, 1), (240 * window + 1, 2)]:
        note("local sort", np.dtype(dtype).name, descending, total_order, value_dtype, n)
        ran = check(random_bits(n, 8 * size, n), dtype, value_dtype, descending, total_order,
                    from_index=n % 2 == 0)
        assert ran == passes


@pytest.mark.parametrize("size", [4, 8])
@pytest.mark.parametrize("pairs", [False, True])
def test_runs_of_every_length_around_a_window(size, pairs):
    """One digit's runs of exactly a window, and of one key more (which need all digits or
    two); runs of two digits that are longer than a window, which a block orders through memory."""
    window = WINDOWS[size, pairs]
    width = 8 * size
    kind = np.dtype(f"uint{width}")
    value = np.uint32 if pairs else None
    rng = np.random.default_rng(size)
    for longest in (window, window + 1):
        note("one digit", size, pairs, longest)
        top = np.repeat(np.arange(16), [longest, 1, 2, 63, 64, 65, window // 2] + 9 * [window - 1])
        low = random_bits(top.size, width, 3) >> kind.type(8)
        bits = rng.permutation(top.astype(kind) << kind.type(width - 8) | low)
        ran = check(bits, kind, value)
        assert ran == 1 if longest == window else ran > 1
    # (8-byte keys from 2^21 to 2^23 take the passes over their upper half.)
    for length in (window - 1, window, window + 1, 2 * window + 1):
        note("two digits", size, pairs, length)
        n = 241 * window
        bits = random_bits(n, width, length)
        at = rng.permutation(n)[:length]
        low = random_bits(length, width, 5) & kind.type((1 << (width - 16)) - 1)
        bits[at] = kind.type(0x1234 << (width - 16)) | low
        if length > window:
            low[: length // 2] = low[0]  # copies of one key within the long run
            bits[at] = kind.type(0x1234 << (width - 16)) | low
        check(bits, kind, value, descending=length % 2 == 0)


@pytest.mark.parametrize("size", [4, 8])
@pytest.mark.parametrize("value_dtype", [None, np.uint32, np.uint64])
def test_windows_whose_keys_crowd_are_sorted_by_digits(size, value_dtype):
    """A few runs of one digit hold many copies, or keys side by side: bins of sixteen keys
    and more, and more bins of two than are listed; the other runs are random."""
    width = 8 * size
    kind = np.dtype(f"uint{width}")
    bits = random_bits(200_003, width, 11)
    top = bits >> kind.type(width - 8)
    rng = np.random.default_rng(12)
    low = kind.type((1 << (width - 8)) - 1)
    for run, values in [(3, 1), (7, 15), (8, 17), (9, 300), (10, 380)]:
        inside = np.flatnonzero(top == run)
        few = rng.integers(0, 1 << (width - 8), values, dtype=kind) & low
        bits[inside] = kind.type(run << (width - 8)) | few[rng.integers(0, values, inside.size)]
    inside = np.flatnonzero(top == 200)
    bits[inside] = kind.type(200 << (width - 8)) | rng.permutation(inside.size).astype(kind)
    note("crowded windows", size, value_dtype)
    assert check(bits, kind, value_dtype, from_index=False) == 1
    assert check(bits, kind, value_dtype, descending=True) == 1


def test_inputs_that_would_crowd_most_windows_take_every_digit():
    note("many copies")
    rng = np.random.default_rng(13)
    values = random_bits(10_000, 32, 14)
    assert check(values[rng.integers(0, values.size, 300_000)], np.uint32) == 4
    bits = random_bits(300_000, 64, 15) & np.uint64(0xFFFF00000000FFFF)
    assert check(bits, np.uint64, np.uint32) == 4  # the digits that differ


def check_on_device(bits, dtype, value_dtype=None):
    """`check` for long columns: an int64 or int32 tensor of the keys' bits; ascending integers."""
    import torch
    n, width = bits.numel(), bits.element_size()
    low = torch.iinfo(bits.dtype).min if np.dtype(dtype).kind == "u" else 0
    expect = torch.sort(bits ^ low, stable=True)
    work = bits.clone()
    keys = D(n, dtype, _bytes=work.view(torch.uint8))
    size = 0 if value_dtype is None else np.dtype(value_dtype).itemsize
    temp = capi.temp_buffer(capi.radix_sort_temp_bytes(n, dtype, size))
    if value_dtype is None:
        capi.radix_sort_keys(keys, temp)
    else:
        values = D.zeros(n, value_dtype)
        capi.radix_sort_pairs(keys, values, temp, values_from_index=True)
    sync()
    assert torch.equal(work, expect.values ^ low)
    if value_dtype is not None:
        held = values.bytes.view({4: torch.int32, 8: torch.int64}[size]).to(torch.int64)
        assert torch.equal(held, expect.indices)
    return capi.radix_sort_passes(temp, n, dtype, size)[0]


@pytest.mark.parametrize("dtype,value_dtype", [(np.uint32, None), (np.int32, np.uint32), (np.uint64, None)])
def test_long_columns_whose_parts_differ_take_every_digit(dtype, value_dtype):
    """More draws than are looked at, from a column that is filled in front and padded behind (or the
    other way round): a single run of the padding would be one block's."""
    import torch
    n = (1 << 25) + 3
    width = 8 * np.dtype(dtype).itemsize
    kind = {32: torch.int32, 64: torch.int64}[width]
    uniform = torch.from_numpy(random_bits(n, width, 31).view(f"int{width}")).to("cuda:0")
    note("uniform", np.dtype(dtype).name, n)
    assert check_on_device(uniform, dtype, value_dtype) == 2
    for value in (-1, (1 << (width - 1)) - 1, 0x3F800000):
        for first, last in [(0.5, 1), (0, 0.5), (0.75, 1), (0.99, 1)]:
            note("padded", np.dtype(dtype).name, value, first, last)
            bits = uniform.clone()
            bits[int(first * n):int(last * n)] = torch.tensor(value, dtype=kind)
            assert check_on_device(bits, dtype, value_dtype) == width // 8


@pytest.mark.parametrize("dtype,value_dtype", [
    (np.uint32, None), (np.uint32, np.uint32), (np.uint64, None), (np.uint64, np.uint64)])
def test_a_run_that_the_draws_let_pass_is_told_by_the_counts(dtype, value_dtype):
    """Two windows of keys of one prefix among uniform ones: copies, and different ones, which of 8-byte keys
    the passes over the upper half and the ties order (and of copies, where these are as many as those order)."""
    size = np.dtype(dtype).itemsize
    width = 8 * size
    kind = np.dtype(dtype).type
    window = WINDOWS[size, value_dtype is not None]
    n = (1 << 23) + 1
    uniform = random_bits(n, width, 41)
    at = np.random.default_rng(42).permutation(n)[:2 * window]
    low = random_bits(at.size, width, 43) & kind((1 << (width - 16)) - 1)
    for name, keys, passes in [("copies", low[:1], (4, size)), ("different", low, (4,))]:
        note("two windows", np.dtype(dtype).name, value_dtype, name)
        bits = uniform.copy()
        bits[at] = kind(0x3456 << (width - 16)) | keys
        assert check(bits, dtype, value_dtype) in passes
    note("one window", np.dtype(dtype).name, value_dtype)
    bits[at[window // 2:]] = uniform[at[window // 2:]]
    assert check(bits, dtype, value_dtype) == 2


@pytest.mark.parametrize("size", [4, 8])
@pytest.mark.parametrize("value_dtype", [None, np.uint16, np.uint64])
def test_runs_longer_than_a_window_that_no_count_tells(size, value_dtype):
    """A block orders them through memory: no other key has the run's lower digit.  Different keys, copies,
    and both, of keys whose last digits are the same or not."""
    window = WINDOWS[size, value_dtype is not None]
    width = 8 * size
    kind = np.dtype(f"uint{width}").type
    n = (600 if size == 4 else 450) * window
    assert size == 4 or n < 1 << 21  # where the passes over the upper half come first
    rng = np.random.default_rng(size)
    bits = random_bits(n, width, 51)
    bare = np.flatnonzero((bits >> kind(width - 16) & kind(0xFF)) == 0x34)
    bits[bare] += rng.integers(1, 0x100 - 0x34, bare.size, dtype=kind) << kind(width - 16)
    for length in (window + 1, 3 * window // 2, 7 * window // 4):
        # (Nothing but copies crowd the draws of 4-byte keys alone, and those of longer runs.)
        only_copies = length == window + 1 and (size == 8 or value_dtype is not None)
        for copies, mask in [(0, 0), (4, 0), (0, 0xFF)] + [(1, 0)] * only_copies:
            note("long run", size, value_dtype, length, copies, mask)
            at = rng.permutation(n)[:length]
            low = random_bits(length, width, 52) & kind((1 << (width - 16)) - 1 - mask)
            if copies:
                low[::copies] = low[0]
            keys = bits.copy()
            keys[at] = kind(0x1234 << (width - 16)) | low
            assert check(keys, np.dtype(kind), value_dtype, descending=length % 2 == 0) == 2


def crowded_bits(n, width, seed):
    """Values of every width some 30 times each: neither the local sort nor the ties take them."""
    values = random_bits(n // 30, width, seed)
    return values[np.random.default_rng(seed).integers(0, values.size, n)]


@pytest.mark.parametrize("dtype,descending", [
    (np.uint32, True), (np.int32, False), (np.float32, True), (np.uint64, False), (np.float64, True)])
@pytest.mark.parametrize("value_dtype", [None, np.uint16, np.uint32, np.uint64])
def test_refused_inputs_take_every_pass(dtype, descending, value_dtype):
    """The chains of four and eight passes, at the edges of the short tiles and with every choice of tile."""
    size = np.dtype(dtype).itemsize
    edges = [512 * 6144, 512 * 9216 + 1, 512 * 12288] if size == 4 else [128 * 3072, 128 * 4096 + 1, 128 * 6144 + 1]
    edges = [18_433, 100_003] + (edges if value_dtype is None else [221_261])
    for n in edges:
        for large_block, short_tiles in [(-1, -1), (0, -1), (2**31 - 1, 0)]:
            if n > 400_000 and large_block >= 0:
                continue
            capi.sort_set_parameter(capi.SORT_PARAM_LARGE_BLOCK_MIN_TILES_PER_CU, large_block)
            capi.sort_set_parameter(capi.SORT_PARAM_SHORT_TILE_MAX_TILES, short_tiles)
            note("every pass", np.dtype(dtype).name, value_dtype, n, large_block, short_tiles)
            assert check(crowded_bits(n, 8 * size, n), dtype, value_dtype, descending, total_order=True,
                         from_index=n % 2 == 0) == size


def test_two_refused_sorts_on_two_streams():
    """Chains of four pipelined passes and of eight passes of pairs share the GPU."""
    import torch
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    a, b = crowded_bits((1 << 24) + 11, 32, 71), crowded_bits((1 << 23) + 5, 64, 72)
    d_a = [D.from_numpy(a) for _ in range(3)]
    d_b = [D.from_numpy(b) for _ in range(3)]
    d_v = [D.zeros(b.size, np.uint32) for _ in range(3)]
    t_a = [capi.temp_buffer(capi.radix_sort_temp_bytes(a.size, np.uint32)) for _ in range(3)]
    t_b = [capi.temp_buffer(capi.radix_sort_temp_bytes(b.size, np.uint64, 4)) for _ in range(3)]
    sync()
    note("two refused sorts on two streams")
    for i in range(3):
        with torch.cuda.stream(s1):
            capi.radix_sort_keys(d_a[i], t_a[i])
        with torch.cuda.stream(s2):
            capi.radix_sort_pairs(d_b[i], d_v[i], t_b[i], values_from_index=True)
    sync()
    e_a, order = np.sort(a), np.argsort(b, kind="stable")
    for i in range(3):
        assert capi.radix_sort_passes(t_a[i], a.size, np.uint32)[0] == 4
        assert capi.radix_sort_passes(t_b[i], b.size, np.uint64, 4)[0] == 8
        assert np.array_equal(d_a[i].numpy(), e_a)
        assert np.array_equal(d_b[i].numpy(), b[order]) and np.array_equal(d_v[i].numpy(), order)


@pytest.mark.parametrize("dtype,value_dtype,share", [
    (np.uint32, None, 0.6), (np.int32, None, 0.4), (np.float32, None, 0.6), (np.uint32, np.uint32, 0.6),
    (np.int32, np.uint64, 0.65), (np.float32, np.uint16, 0.65), (np.uint64, None, 0.9), (np.float64, None, 0.95)])
def test_windows_with_more_shared_bins_than_the_list_holds(dtype, value_dtype, share):
    """Full windows, in which a share of the keys comes twice: copies, and neighbours that differ in the last bit."""
    size = np.dtype(dtype).itemsize
    n = 240 * WINDOWS[size, value_dtype is not None]
    rng = np.random.default_rng(size)
    for descending in (False, True):
        for twin in (0, 1):
            note("shared bins", np.dtype(dtype).name, value_dtype, descending, twin)
            bits = random_bits(n, 8 * size, 81)
            twice = int(share * n) // 2
            bits[twice:2 * twice] = bits[:twice] ^ bits.dtype.type(twin)
            bits = bits[rng.permutation(n)]
            assert check(bits, dtype, value_dtype, descending, total_order=True, from_index=twin == 0) == 1


def test_few_copies_of_every_value_take_little_longer_than_none():
    """2 000 000 keys, each value once on average: all windows were sorted by digits, in 1.6 times the time."""
    import torch
    n = 2_000_000
    generator = torch.Generator(device="cuda:0")
    generator.manual_seed(91)
    uniform = torch.randint(-(1 << 31), 1 << 31, (n,), generator=generator, device="cuda:0").to(torch.int32)
    copies = uniform[torch.randint(0, n, (n,), generator=generator, device="cuda:0")]
    temp = capi.temp_buffer(capi.radix_sort_temp_bytes(n, np.int32))
    keys = D(n, np.int32)

    def us(column):
        source = D(n, np.int32, _bytes=column.view(torch.uint8))
        times = []
        for _ in range(15):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(20):
                capi.transform(source, keys)
                capi.radix_sort_keys(keys, temp)
            end.record()
            sync()
            times.append(start.elapsed_time(end) * 50)
        assert capi.radix_sort_passes(temp, n, np.int32)[0] == 1
        return sorted(times)[7]

    us(uniform)
    base, some = us(uniform), us(copies)
    note("copies", base, some)
    assert torch.equal(keys.bytes.view(torch.int32), torch.sort(copies).values)
    assert some < 1.4 * base


def test_digits_that_all_keys_share_do_not_hide_the_topmost():
    """8-byte keys of 40 bits, and of 24 (no two digits to save)."""
    note("forty bits")
    for n, passes in [(100_003, 1), (1_500_001, 2)]:
        assert check(random_bits(n, 64, n) >> np.uint64(24), np.int64, np.uint32) == passes
    assert check(random_bits(100_003, 64, 16) >> np.uint64(40), np.uint64) == 3


def test_local_sorts_can_be_captured_and_replayed():
    """Draws, windows and what is put off are told anew by every replay."""
    import torch
    n = 240 * 9216 + 77
    static = torch.zeros(n, dtype=torch.int32, device="cuda:0")
    work = torch.zeros(n, dtype=torch.int32, device="cuda:0")
    keys = D(n, np.uint32, _bytes=work.view(torch.uint8))
    temp = capi.temp_buffer(capi.radix_sort_temp_bytes(n, np.uint32))

    def calls():
        work.copy_(static)
        capi.radix_sort_keys(keys, temp)

    calls()  # the one-time queries
    sync()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            calls()
    sync()
    few = random_bits(1000, 32, 17)
    inputs = [random_bits(n, 32, 18), few[np.random.default_rng(19).integers(0, 1000, n)], random_bits(n, 32, 20)]
    for replay, (bits, passes) in enumerate(zip(inputs, (2, 4, 2))):
        note("replay", replay)
        static.copy_(torch.from_numpy(bits.view(np.int32)))
        assert torch.rand(1 << 20, device="cuda:0").sum().item() > 0  # eager work between replays
        graph.replay()
        sync()
        assert np.array_equal(keys.numpy(), np.sort(bits))
        assert capi.radix_sort_passes(temp, n, np.uint32)[0] == passes


@pytest.mark.parametrize("dtype,descending,total_order", [
    (np.uint64, False, False), (np.int64, True, False), (np.float64, False, False),
    (np.float64, True, True)])
@pytest.mark.parametrize("value_dtype", [None, np.uint32])
def test_one_tile_sorts_by_the_topmost_digits(dtype, descending, total_order, value_dtype):
    """8-byte keys of one tile: neighbours of one prefix (some hundred of them, in runs of
    two to four), a prefix of as many keys as a key looks at and of one more (all digits), prefixes that
    most keys share (not tried), and keys that are all the same."""
    rng = np.random.default_rng(21)
    for n in (2, 2048, 2049, 9216 if value_dtype is None else 7168):
        for prefix in (0, 2, 24, 25, 26, n):
            note("one tile by prefix", np.dtype(dtype).name, n, prefix)
            bits = random_bits(n, 64, n + prefix)
            shared = rng.permutation(n)[:min(prefix, n)]
            bits[shared] = (bits[shared[:1]] & np.uint64(0xFFFFFFFF00000000)) | random_bits(shared.size, 32, 22)
            for first in range(0, min(n, 300) - 4, 4):  # runs of two to four
                run = slice(first, first + 2 + first // 4 % 3)
                bits[run] = (bits[first] & np.uint64(0xFFFFFFFFFF000000)) | (bits[run] & np.uint64(0xFFFFFF))
            check(bits, dtype, value_dtype, descending, total_order)
    check(np.full(777, 5, np.uint64), np.uint64, np.uint32)


def with_a_cluster(n, length, seed, unasked=False):
    """Random 8-byte keys, `length` of which share their upper half: anywhere, or where the block
    asks no key (it asks the 512 at t * n / 512)."""
    bits = random_bits(n, 64, seed)
    places = np.arange(n)
    if unasked:
        places = np.setdiff1d(places, np.arange(512) * n // 512)
    at = np.random.default_rng(seed).permutation(places)[:length]
    bits[at] = np.uint64(0x12345678 << 32) | random_bits(at.size, 32, seed + 1).astype(np.uint64)
    return bits


@pytest.mark.parametrize("dtype", [np.int64, np.uint64, np.float64])
@pytest.mark.parametrize("value_dtype", [None, np.uint32, np.uint64])
def test_one_tile_whose_keys_cluster(dtype, value_dtype):
    """Prefixes of as many keys as are taken and looked through, of more than a key looks at where none of
    them is asked, of all but the first keys, many prefixes of some 20 keys each, and copies."""
    for n in (500, 2048, 5000, 9216 if value_dtype is None else 5120 if value_dtype is np.uint64 else 7168):
        for length, unasked in [(20, False), (35, False), (90, False), (n // 10, False), (n - 3, False),
                                (257, True), (262, True), (300, True), (n // 3, True)]:
            note("cluster", np.dtype(dtype).name, value_dtype, n, length, unasked)
            check(with_a_cluster(n, length, n + length, unasked), dtype, value_dtype, from_index=False,
                  descending=length % 2 == 0, total_order=True)
        note("forty signed bits", np.dtype(dtype).name, value_dtype, n)
        check((random_bits(n, 64, n).view(np.int64) >> 24).view(np.uint64), dtype, value_dtype, total_order=True)
        few = random_bits(n // 10, 64, n)
        check(few[np.random.default_rng(n).integers(0, few.size, n)], dtype, value_dtype, from_index=False)


def test_one_tile_whose_keys_cluster_takes_no_longer_than_every_digit():
    """9000 keys: a third of the passes more where a prefix says nothing, not passes for nothing and keys that
    look through hundreds of others (five times as long)."""
    import torch
    temp = capi.temp_buffer(capi.radix_sort_temp_bytes(9000, np.uint64))

    def us(bits):
        source, keys = D.from_numpy(bits), D(9000, np.uint64)
        times = []
        for _ in range(15):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(20):
                capi.transform(source, keys)
                capi.radix_sort_keys(keys, temp)
            end.record()
            sync()
            times.append(start.elapsed_time(end) * 50)
        return sorted(times)[7]

    uniform = us(random_bits(9000, 64, 61))
    for name, bits in [("a tenth", with_a_cluster(9000, 900, 62)), ("80", with_a_cluster(9000, 80, 63)),
                       ("forty signed bits", (random_bits(9000, 64, 64).view(np.int64) >> 24).view(np.uint64))]:
        clustered = us(bits)
        note(name, uniform, clustered)
        assert clustered < 2.5 * uniform


def test_one_tile_of_narrow_keys_skips_the_digits_they_share():
    note("narrow keys")
    for n in (18_432, 12_289, 777):
        check(random_bits(n, 32, n) & np.uint32(0x000FF0F0), np.uint32, descending=n % 2 == 0)
        check(random_bits(min(n, 9216), 64, n) & np.uint64(0x00FF00000000FF00), np.int64, np.uint32)
