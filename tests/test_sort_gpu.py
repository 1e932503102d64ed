"""GPU parity of sort / sort! / sortperm / sortperm! (src/kernels/sorting.jl:1-3) against the oracle, through the
C ABI: the sizes and element types of test/hip_rocarray/sorting.jl:5-28 for the default order and rev=true
(values and permutations bit-exact, NaNs compared as equal), plus sizes that span many tiles, special floats,
duplicates (stability) and small-range integers (skipped passes).  The two other forms of that test, `lt=!isless` and
`by=k -> 2k` (:20-26), are native as well: descending order, and map -> sortperm of the keys -> gather."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TYPES = [np.float16, np.float32, np.float64, np.int16, np.int32, np.int64]


def _rand(rng, dtype, n):
    dt = np.dtype(dtype)
    if dt.kind == "f":
        return rng.random(n).astype(dt)                       # rand(T, sz)
    return rng.integers(np.iinfo(dt).min, np.iinfo(dt).max, n, dtype=dt, endpoint=True)


def _check(rk, orc, x):
    xd = rk.ROCArray(x)
    for rev in (False, True):
        want, wperm = orc.sort(x, rev), orc.sortperm(x, rev)
        got = rk.Array(rk.sort(xd, rev=rev))
        assert got.dtype == x.dtype and np.array_equal(got, want, equal_nan=x.dtype.kind == "f"), rev
        if x.dtype.kind == "f":
            assert np.array_equal(np.signbit(got[~np.isnan(got)]), np.signbit(want[~np.isnan(want)]))
        p = rk.Array(rk.sortperm(xd, rev=rev))
        assert p.dtype == np.int64 and np.array_equal(p, wperm), rev
    assert np.array_equal(rk.Array(xd), x, equal_nan=x.dtype.kind == "f")          # sort / sortperm leave x alone
    assert rk.sort_(xd) is xd
    assert np.array_equal(rk.Array(xd), orc.sort(x), equal_nan=x.dtype.kind == "f")


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("sz", [1, 2, 3, 4, 33, 333, 3333, 4096])
def test_reference_sizes_and_types(rk, orc, dtype, sz):
    _check(rk, orc, _rand(np.random.default_rng(sz), dtype, sz))


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("sz", [1, 2, 3, 4, 33, 333, 3333, 4096, 100_003])
def test_reference_lt_and_by(rk, orc, dtype, sz):
    """test/hip_rocarray/sorting.jl:20-26: `sort(xd; lt=!isless)`, `xd[sortperm(xd; lt=!isless)]`, `sort(xd; by=k -> 2k)`,
    `xd[sortperm(xd; by=k -> 2k)]` against the host's sorts (the reference compares values)."""
    x = _rand(np.random.default_rng(1000 + sz), dtype, sz)
    if np.dtype(dtype).kind == "i":
        x = (x // 4).astype(dtype)                              # 2k stays inside the type, as Julia's Int64 product does
    xd = rk.ROCArray(x)
    desc = np.sort(x)[::-1]
    assert np.array_equal(rk.Array(rk.sort(xd, lt=rk.not_isless)), desc)
    p = rk.Array(rk.sortperm(xd, lt=rk.not_isless))
    assert sorted(p.tolist()) == list(range(1, sz + 1)) and np.array_equal(x[p - 1], desc)
    by = lambda k: 2 * k                                        # noqa: E731
    asc = np.sort(x)
    assert np.array_equal(rk.Array(rk.sort(xd, by=by)), asc)
    p = rk.Array(rk.sortperm(xd, by=by))
    assert sorted(p.tolist()) == list(range(1, sz + 1)) and np.array_equal(x[p - 1], asc)
    assert np.array_equal(rk.Array(rk.sort(xd, by=lambda k: -k)), desc)       # a `by` that reverses
    assert np.array_equal(rk.Array(xd), x)
    y = rk.ROCArray(x)
    assert rk.sort_(y, by=by, rev=True) is y and np.array_equal(rk.Array(y), desc)
    with pytest.raises(NotImplementedError):
        rk.sort(xd, lt=lambda a, b: a < b)                      # any other comparator: the stock path


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("n", [4097, 65_537, 1_000_003])
def test_many_tiles(rk, orc, dtype, n):
    _check(rk, orc, _rand(np.random.default_rng(n), dtype, n))


@pytest.mark.parametrize("dtype", [np.float16, np.float32, np.float64])
def test_special_floats_and_stability(rk, orc, dtype):
    rng = np.random.default_rng(5)
    base = np.array([0.0, -0.0, np.nan, np.inf, -np.inf, 1.0, -1.0, 65504.0, -65504.0, 6e-8, -6e-8], dtype=dtype)
    x = rng.choice(base, 50_000)
    x[::7] = -x[::7]
    _check(rk, orc, x)


@pytest.mark.parametrize("dtype", [np.int16, np.int32, np.int64])
def test_small_range_integers_skip_passes(rk, orc, dtype):
    rng = np.random.default_rng(6)
    _check(rk, orc, rng.integers(-10, 11, 300_000).astype(dtype))                  # perf/array.jl:16 rand(-10:10, ...)
    _check(rk, orc, np.full(10_000, 7, dtype=dtype))                               # every pass skipped
    _check(rk, orc, (rng.integers(0, 2, 100_000) * 256).astype(dtype))             # only the second digit varies
    _check(rk, orc, np.arange(100_000, 0, -1).astype(dtype) if dtype != np.int16 else np.arange(30_000, 0, -1).astype(dtype))


def test_perf_suite_size_and_in_place_outputs(rk, orc):
    x = np.random.default_rng(7).random(512 * 1000).astype(np.float32)             # sort(gpu_vec), perf/array.jl:145
    _check(rk, orc, x)
    ix = rk.ROCArray(dims=(x.size,), dtype=np.int64)
    assert rk.sortperm_(ix, rk.ROCArray(x)) is ix
    assert np.array_equal(x[rk.Array(ix) - 1], np.sort(x))                         # y == xd[sortperm(xd)], sorting.jl:14


def test_full_size_sort(rk, orc):
    x = np.random.default_rng(8).standard_normal(1 << 24).astype(np.float32)
    got = rk.Array(rk.sort(rk.ROCArray(x)))
    assert np.array_equal(got, np.sort(x))
    k = np.random.default_rng(9).integers(-2**62, 2**62, 1 << 22, dtype=np.int64)
    p = rk.Array(rk.sortperm(rk.ROCArray(k), rev=True))
    assert np.array_equal(p, orc.sortperm(k, True))


@pytest.mark.parametrize("tiles", [1, 2, 7, 8, 9, 127, 128, 129, 255, 256, 257])
@pytest.mark.parametrize("dtype", [np.int16, np.float16, np.float32, np.int64])
def test_table_of_counts_edges(rk, orc, dtype, tiles):
    # up to 256 tiles of 4096 keys every workgroup of a pass over 2-byte keys sums the columns of the table of counts itself (8
    # groups of rows, 16 rows a round): one key more and less than whole tiles around the edges of the groups and of the dispatch;
    # 4- and 8-byte keys have the edges of the tiles that splitters sort there
    rng = np.random.default_rng(tiles)
    for n in (tiles * 4096 - 1, tiles * 4096, tiles * 4096 + 1):
        x = _rand(rng, dtype, n)
        assert np.array_equal(rk.Array(rk.sort(rk.ROCArray(x))), orc.sort(x))
        assert np.array_equal(rk.Array(rk.sortperm(rk.ROCArray(x), rev=True)), orc.sortperm(x, True))


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32, np.int64])
def test_constant_digits(rk, orc, dtype):
    # digits in which no two keys differ are skipped: low ones (whole numbers as floats, multiples of 65536), high ones, a
    # middle one that only relative keys carry into, none at all
    rng = np.random.default_rng(17)
    for n in (50_000, 300_000):
        _check(rk, orc, rng.integers(-500, 500, n).astype(dtype))
        _check(rk, orc, (rng.integers(-500, 500, n) * 65536).astype(dtype))
        _check(rk, orc, (rng.integers(0, 2, n) * (1 << 24) + 255).astype(dtype))
        _check(rk, orc, np.full(n, 3, dtype=dtype))


def _passes_run(rk, x, perm):
    """The number of passes that a small sort ran, from the control block at the head of its temporary: 256 digit counts
    and three flags for each of 8 passes, the first and the last pass, then their number."""
    import torch
    from amdgpu_jl_amd import _lib as L
    from amdgpu_jl_amd.array import stream_ptr
    d = rk.ROCArray(x)
    out = rk.ROCArray(dims=(x.size,), dtype=np.int64 if perm else x.dtype)
    tmp = torch.empty(int(L.lib.rk_sort_tmp_bytes(d.code, x.size, int(perm))), dtype=torch.uint8, device="cuda")
    f = L.lib.rk_sortperm if perm else L.lib.rk_sort_to
    L.check(f(d.code, d.ptr, out.ptr, x.size, 0, tmp.data_ptr(), tmp.numel(), stream_ptr()), "sort")
    at = 8 * 256 * 4 + 3 * 8 * 4 + 2 * 4
    return int(tmp[at:at + 4].cpu().numpy().view(np.uint32)[0]), rk.Array(out)


@pytest.mark.parametrize("perm", [False, True])
@pytest.mark.parametrize("dtype", [np.int16, np.int32, np.int64])
@pytest.mark.parametrize("n", [2, 4096, 4097, 300_000, 1 << 20])
def test_digits_that_no_two_relative_keys_differ_in_run_no_pass(rk, orc, dtype, n, perm):
    """Small integer sorts: a pass for every digit in which keys minus the smallest one differ, wherever it stands (an id in
    the high digits and a small number, perhaps negative, in the low one; a step; a range that carries), and no other.  More
    than 4096 keys of 4 and 8 bytes are sorted by splitters, in no pass at all."""
    rng = np.random.default_rng(n)
    bits = 8 * np.dtype(dtype).itemsize
    ids, small = rng.integers(0, 100, n).astype(np.int64), rng.integers(-100, 101, n).astype(np.int64)
    wide = np.int64(1) << (bits - 8)
    cases = [(ids - 50) * wide + (small + 100), (ids - 50) * wide + small, (ids - 50) * wide, small, small + 5000, small * 256 // 2,
             np.full(n, -7, dtype=np.int64), rng.integers(-(1 << (bits - 1)), 1 << (bits - 1), n, dtype=np.int64)]
    if bits >= 32:
        cases.append((ids << (bits // 2)) + small * (small > 0))
    for k in cases:
        x = k.astype(dtype)
        rel = np.bitwise_or.reduce(x.astype(np.int64).view(np.uint64) - np.uint64(int(x.min()) & (2 ** 64 - 1)))
        want = sum(1 for p in range(bits // 8) if (int(rel) >> (8 * p)) & 255) if bits == 16 or n <= 4096 else 0
        ran, got = _passes_run(rk, x, perm)
        assert np.array_equal(got, orc.sortperm(x) if perm else orc.sort(x))
        assert ran == want, (ran, want, hex(int(rel)))


# More than 256 tiles of 4096 keys: the sort counts the digits of every tile before each pass (no look-back).
LARGE = 1024 * 4096 + 4096 * 3 + 37


@pytest.mark.parametrize("dtype", TYPES)
def test_large_sorts_all_types(rk, orc, dtype):
    _check(rk, orc, _rand(np.random.default_rng(11), dtype, LARGE))


@pytest.mark.parametrize("dtype", [np.int16, np.int32, np.int64])
def test_large_small_range_integers(rk, orc, dtype):
    rng = np.random.default_rng(12)
    _check(rk, orc, rng.integers(-10, 11, LARGE).astype(dtype))                    # one pass: the range fits a digit
    _check(rk, orc, rng.integers(-300, 70_000 if dtype != np.int16 else 3_000, LARGE).astype(dtype))
    _check(rk, orc, np.full(LARGE, -5, dtype=dtype))                               # every pass skipped
    _check(rk, orc, (rng.integers(0, 2, LARGE) * 256).astype(dtype))               # low digit constant, not skipped


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_large_special_floats(rk, orc, dtype):
    rng = np.random.default_rng(13)
    base = np.array([0.0, -0.0, np.nan, np.inf, -np.inf, 1.0, -1.0, 65504.0, -65504.0, 6e-8, -6e-8], dtype=dtype)
    x = rng.choice(base, LARGE)
    x[::7] = -x[::7]
    _check(rk, orc, x)
    _check(rk, orc, (1.0 + rng.random(LARGE)).astype(dtype))                       # one binade: exponent digits constant


def test_large_unaligned_view(rk, orc):
    x = _rand(np.random.default_rng(14), np.float32, LARGE + 10)
    d = rk.ROCArray(x)
    v = d.view_range(4, LARGE + 6)                                                 # starts 12 bytes into the buffer
    assert np.array_equal(rk.Array(rk.sort(v)), orc.sort(x[3:LARGE + 6]))
    assert np.array_equal(rk.Array(rk.sortperm(v, rev=True)), orc.sortperm(x[3:LARGE + 6], True))
    rk.sort_(v)
    got = rk.Array(d)
    assert np.array_equal(got[3:LARGE + 6], orc.sort(x[3:LARGE + 6]))
    assert np.array_equal(got[:3], x[:3]) and np.array_equal(got[LARGE + 6:], x[LARGE + 6:])


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("n", [2, 4097, (1 << 20) + 1, (1 << 20) + 8191 * 3])
def test_sorted_copy_by_number_of_passes(rk, orc, dtype, n):
    """sort(x) reads x in its first pass and writes another array: keys that differ in no digit (no pass runs: a copy), in
    one, in an odd and an even number, and in all of them; x starts at an odd element and stays as it was."""
    rng = np.random.default_rng(n)
    dt = np.dtype(dtype)
    whole = _rand(rng, dtype, n + 1)
    cases = [np.full(n + 1, whole[0], dtype=dtype), whole]
    if dt.kind == "i":
        cases += [rng.integers(0, 1 << min(bits, 8 * dt.itemsize - 1), n + 1).astype(dtype) for bits in (8, 16, 24)]
    for x in cases:
        for rev in (False, True):
            xd = rk.ROCArray(x)
            got = rk.Array(rk.sort(xd.view_range(2, n + 1), rev=rev))
            assert np.array_equal(got, orc.sort(x[1:], rev))
            assert np.array_equal(rk.Array(xd), x)


@pytest.mark.parametrize("dtype", [np.int16, np.float32, np.float64])
def test_unaligned_views(rk, orc, dtype):
    # keys that start 1 .. 9 elements into a buffer: the vector body of the whole-array reads starts later
    x = _rand(np.random.default_rng(10), dtype, 70_010)
    d = rk.ROCArray(x)
    for first in (2, 3, 4, 6, 10):
        v = d.view_range(first, 70_005)
        want = orc.sort(x[first - 1:70_005])
        assert np.array_equal(rk.Array(rk.sort(v)), want)
        assert np.array_equal(rk.Array(rk.sortperm(v)), orc.sortperm(x[first - 1:70_005]))
    v = d.view_range(3, 70_001)
    rk.sort_(v, rev=True)
    got = rk.Array(d)
    assert np.array_equal(got[2:70_001], orc.sort(x[2:70_001], rev=True))
    assert np.array_equal(got[:2], x[:2]) and np.array_equal(got[70_001:], x[70_001:])      # neighbours untouched


def test_unsupported_forms(rk):
    xd = rk.ROCArray(np.arange(10, dtype=np.float32))
    with pytest.raises(rk.UnsupportedError):
        rk.sort(xd, lt=lambda a, b: a > b)
    with pytest.raises(rk.UnsupportedError):
        rk.sortperm(xd, by=lambda k: k if k > 0 else -k)        # control flow on the value: not traceable
    with pytest.raises(rk.UnsupportedError):
        rk.sort(rk.ROCArray(np.zeros((3, 4), dtype=np.float32)))
    with pytest.raises(rk.UnsupportedError):
        rk.sort(rk.ROCArray(np.zeros(5, dtype=np.uint8)))
    assert len(rk.sort(rk.ROCArray(np.zeros(0, dtype=np.float32)))) == 0


@pytest.mark.parametrize("dtype,utype", [(np.float32, np.uint32), (np.float64, np.uint64), (np.float16, np.uint16)])
@pytest.mark.parametrize("rev", [False, True])
def test_sort_keeps_nan_bit_patterns(rk, dtype, utype, rev):
    # sort!: the result is a permutation of the input bit for bit -- negative NaNs and payloads survive -- with the
    # non-NaN part in isless order and every NaN after it (before it with rev); sortperm: NaNs are equal keys, index order
    rng = np.random.default_rng(99)
    n = 300_000
    h = rng.standard_normal(n).astype(dtype)
    u = h.view(utype)
    nan_bits = {np.float32: [0xffc00001, 0x7fc12345, 0x7f800001, 0xff800001, 0x7fffffff, 0x7fc00000],
                np.float64: [0xfff8000000000001, 0x7ff8000000abcdef, 0x7ff0000000000001, 0xfff0000000000001, 0x7fffffffffffffff, 0x7ff8000000000000],
                np.float16: [0xfe01, 0x7e55, 0x7c01, 0xfc01, 0x7fff, 0x7e00]}[dtype]
    pos = rng.choice(n, 600, replace=False)
    for k, p_ in enumerate(pos):
        u[p_] = nan_bits[k % len(nan_bits)]
    h[rng.choice(n, 50)] = np.inf
    h[rng.choice(n, 50)] = -np.inf
    h[rng.choice(n, 50)] = -0.0
    d = rk.ROCArray(h.copy())
    rk.sort_(d, rev=rev)
    got = rk.Array(d)
    assert np.array_equal(np.sort(got.view(utype)), np.sort(h.view(utype)))            # a permutation of the bits
    nn = int(np.isnan(h).sum())
    body = got[nn:] if rev else got[:n - nn]
    tail = got[:nn] if rev else got[n - nn:]
    assert np.isnan(tail).all() and not np.isnan(body).any()
    want = np.sort(h[~np.isnan(h)])
    want = want[::-1] if rev else want
    assert np.array_equal(body, want) and np.array_equal(np.signbit(body), np.signbit(want))
    perm = rk.Array(rk.sortperm(rk.ROCArray(h), rev=rev)) - 1
    nan_part = perm[:nn] if rev else perm[n - nn:]
    assert np.array_equal(nan_part, np.flatnonzero(np.isnan(h)))                          # stable among the NaNs
    assert np.array_equal(np.sort(perm), np.arange(n))


def _spread(rng, dtype, n, kind):
    """Keys that a bucket of the sorts by splitters does not find evenly spread, and some that it does."""
    dt = np.dtype(dtype)
    if kind == "sorted":
        return np.sort(_rand(rng, dtype, n))
    if kind == "equal":
        return np.full(n, 3, dtype=dt)
    if kind == "few":                                   # a few values, far apart and close together
        return rng.choice(np.array([-70000, -3, -2, 0, 1, 2, 3, 1000, 65536], dtype=dt), n)
    if kind == "hundreds":
        return rng.integers(-500, 500, n).astype(dt)
    if kind == "clusters":                              # narrow clusters and far outliers: what a linear map does not spread
        x = rng.integers(0, 200, n) * 3 + rng.choice(np.array([0, 1 << 20, (1 << 20) + 5000], dtype=np.int64), n)
        x[:: n // 7] = 1 << 30
        return x.astype(dt)
    if kind == "gaps":                                  # a few small numbers, again and again far apart, and those once more: what several
        far, near = (1 << 40, 1 << 20) if dt.itemsize == 8 else (1 << 20, 1 << 10)           # divisions of a bucket take apart
        return (rng.integers(0, 50, n) * far + rng.integers(0, 3, n) * near + rng.integers(0, 3, n)).astype(dt)
    if kind == "steep":                                 # every order of magnitude, both signs
        x = np.exp(rng.uniform(-20, 20, n)) * rng.choice([-1.0, 1.0], n)
        return x.astype(dt)
    return (rng.standard_normal(n) * (1 if dt.kind == "f" else 1 << 24)).astype(dt)


@pytest.mark.parametrize("kind", ["sorted", "equal", "few", "hundreds", "clusters", "gaps", "steep", "normal"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32, np.int64])
def test_sorts_by_splitters(rk, orc, dtype, kind):
    """4096 keys are the last that fit a workgroup, 2^20 the last that take buckets; 512 keys a bucket up to 131072 and more
    beyond; tiles of 4096."""
    rng = np.random.default_rng(31)
    for n in (4095, 4096, 4097, 8193, 66_001, 131_073, (1 << 20) - 1, 1 << 20, (1 << 20) + 1):
        x = _spread(rng, dtype, n, kind)
        for rev in (False, True):
            assert np.array_equal(rk.Array(rk.sort(rk.ROCArray(x), rev=rev)), orc.sort(x, rev)), (n, rev)
            assert np.array_equal(rk.Array(rk.sortperm(rk.ROCArray(x), rev=rev)), orc.sortperm(x, rev)), (n, rev)


def _sampled(n, s):
    """Where a sort of n keys takes its s samples; the constants are those of the source, so that a change there shows here."""
    import pathlib
    text = (pathlib.Path(__file__).parent.parent / "amdgpu.jl_amd" / "csrc" / "rk_sort_buckets.hpp").read_text()
    for line in ("constexpr uint32_t SB_OVER = 16;", "uint32_t h = (j + 1u) * 0x9e3779b1u;", "h ^= h >> 15;", "h *= 0x85ebca77u;", "return a + __umulhi(h, b - a);"):
        assert line in text, line
    j, m = np.arange(s, dtype=np.uint64), np.uint64(0xffffffff)
    a, b = j * np.uint64(n) // np.uint64(s), (j + np.uint64(1)) * np.uint64(n) // np.uint64(s)
    h = (j + np.uint64(1)) * np.uint64(0x9e3779b1) & m
    h ^= h >> np.uint64(15)
    h = h * np.uint64(0x85ebca77) & m
    return (a + (h * (b - a) >> np.uint64(32))).astype(np.int64)


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32, np.int64])
@pytest.mark.parametrize("few", [False, True])
def test_bucket_larger_than_lds(rk, orc, dtype, few):
    """Every key that is sampled is larger than all the others, so these are one bucket: more keys than LDS holds."""
    n, s = 30_000, 16 * 64
    rng = np.random.default_rng(5)
    x = rng.integers(0, 7 if few else 1 << 20, n).astype(dtype)
    x[_sampled(n, s)] = (1 << 24) + rng.integers(0, 1 << 20, s)
    _check(rk, orc, x)


@pytest.mark.parametrize("kind", ["sorted", "equal", "few", "hundreds", "clusters", "gaps", "steep", "normal"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int64])
def test_sorts_by_two_levels_of_splitters(rk, orc, dtype, kind):
    """More than 2^20 keys; tiles of 4096 keys below 2^22 and of 8192 from there on, of which the last is full, or holds one key."""
    rng = np.random.default_rng(32)
    for n, rev in (((1 << 20) + 1, False), ((1 << 21) - 5, True), ((1 << 22) - 1, False), (1 << 22, True), ((1 << 22) + 8193, False)):
        x = _spread(rng, dtype, n, kind)
        assert np.array_equal(rk.Array(rk.sort(rk.ROCArray(x), rev=rev)), orc.sort(x, rev)), (n, rev)
        assert np.array_equal(rk.Array(rk.sortperm(rk.ROCArray(x), rev=rev)), orc.sortperm(x, rev)), (n, rev)


@pytest.mark.parametrize("digits", [(), (2,), (3, 4), (2, 3, 4), (0, 7), (1, 3, 6), (0, 2, 3, 5), (0, 1, 2, 3, 4, 5, 6, 7)])
def test_large_int64_by_varying_digits(rk, orc, digits):
    """Keys take radix passes if there are three digits at most from the lowest that varies to the top of their range, others
    splitters; sort! in place and into another array."""
    rng = np.random.default_rng(33)
    n = (1 << 20) + 4097
    x = np.full(n, 1 << 40, dtype=np.int64)
    for d in digits:
        x ^= rng.integers(0, 256, n).astype(np.int64) << (8 * d)
    _check(rk, orc, x)
    y = rk.ROCArray(x)
    rk.sort_(y)
    assert np.array_equal(rk.Array(y), orc.sort(x, False))
    for perm in (False, True):
        planned, got = _passes_run(rk, x, perm)
        assert np.array_equal(got, orc.sortperm(x) if perm else orc.sort(x))
        assert planned == (max(digits) - min(digits) + 1 if digits else 0)


@pytest.mark.parametrize("dtype", [np.float64, np.int64])
@pytest.mark.parametrize("n", [(1 << 23) - 1, 1 << 23, (1 << 24) + 1, 1 << 26])
def test_long_sorts_by_two_levels_of_splitters(rk, dtype, n):
    """From 2^23 keys on an XCD takes neighbouring buckets; 2^26 keys are the most that are sorted this way.  Against torch's sort."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    x = torch.randn(n, device="cuda", generator=g, dtype=torch.float64) if dtype == np.float64 else \
        torch.randint(-2**62, 2**62, (n,), device="cuda", generator=g, dtype=torch.int64)
    xd = rk.ROCArray(buf=x.view(torch.uint8), dims=(n,), dtype=dtype)
    want = torch.sort(x, stable=True)
    assert torch.equal(rk.sort(xd).buf[:8 * n].view(x.dtype), want.values)
    assert torch.equal(rk.sortperm(xd).buf[:8 * n].view(torch.int64) - 1, want.indices)


@pytest.mark.parametrize("dtype", [np.float64, np.int64])
def test_part_whose_keys_lie_far_apart(rk, dtype):
    """The smallest keys stand in the first and the last six tiles of 2048: a tile of their part collects runs on both sides of
    more empty ones than LDS holds at a time."""
    import torch
    rng = np.random.default_rng(34)
    n, tile = 1 << 24, 8192
    x = (1 << 50) + rng.integers(0, 1 << 40, n)
    for part in (slice(0, 6 * tile), slice(n - 6 * tile, n)):
        x[part] = rng.integers(0, 1 << 40, 6 * tile)
    x = torch.from_numpy(x.astype(dtype)).cuda()
    xd = rk.ROCArray(buf=x.view(torch.uint8), dims=(n,), dtype=dtype)
    want = torch.sort(x, stable=True)
    assert torch.equal(rk.sort(xd).buf[:8 * n].view(x.dtype), want.values)
    assert torch.equal(rk.sortperm(xd).buf[:8 * n].view(torch.int64) - 1, want.indices)


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int64])
@pytest.mark.parametrize("few", [False, True])
def test_part_and_buckets_larger_than_lds(rk, orc, dtype, few):
    """Every key that is sampled first is larger than all the others: these are one part of more tiles than a bucket's workgroup
    holds the runs of, and its 256 buckets are larger than LDS."""
    n, s = (1 << 20) + 300_000, 4096
    rng = np.random.default_rng(6)
    x = (rng.integers(0, 7, n) if few else rng.integers(0, 1 << 20, n)).astype(dtype)
    if dtype == np.int64:
        x += rng.integers(0, 7, n) << 40                     # (four digits and more)
    x[_sampled(n, s)] = (1 << 50) + rng.integers(0, 1 << 20, s)
    _check(rk, orc, x)


def _device_sort_check(rk, x, revs=(False, True)):
    """sort and sort! of a vector against torch's sort, bit for bit (no -0.0 beside 0.0 and no NaN among the keys)."""
    import torch
    xt = torch.from_numpy(x).cuda()
    want = torch.sort(xt).values.view(torch.int32)
    for rev in revs:
        xd = rk.ROCArray(buf=xt.clone().view(torch.uint8), dims=(x.size,), dtype=x.dtype.type)
        assert torch.equal(rk.sort(xd, rev=rev).buf[:4 * x.size].view(torch.int32), want.flip(0) if rev else want), rev
        assert torch.equal(xd.buf[:4 * x.size].view(torch.int32), xt.view(torch.int32))
        rk.sort_(xd, rev=rev)
        assert torch.equal(xd.buf[:4 * x.size].view(torch.int32), want.flip(0) if rev else want), rev


QUANTILES = {np.float32: (1 << 22) + 1, np.int32: (1 << 23) + 1}         # from so many keys on sorts of 4-byte keys move them into buckets once


@pytest.mark.parametrize("kind", ["sorted", "equal", "few", "hundreds", "clusters", "gaps", "steep", "normal", "zeros", "quantized", "two in a bin"])
@pytest.mark.parametrize("dtype", [np.float32, np.int32])
def test_sorts_by_quantiles(rk, dtype, kind):
    """One key more than sorts by other ways take, and tiles of 24576 keys of which the last is full, lacks a key or holds one; keys
    that the buckets hold, and that send the call to the radix passes, over all digits or some, or none at all."""
    rng = np.random.default_rng(41)
    n0 = QUANTILES[dtype]
    for n in (n0, 24576 * 343, 24576 * 343 + 1, 24576 * 344 - 1):
        if n < n0:
            continue
        if kind == "zeros":
            x = np.maximum(rng.standard_normal(n) - 1.3, 0) * (1 if dtype == np.float32 else 1 << 24)
        elif kind == "quantized":
            x = rng.standard_normal(n).astype(np.float16).astype(np.float32) * (1 if dtype == np.float32 else 1 << 24)
            x[x == 0] = 0
        elif kind == "two in a bin":                     # 3000 values, many times over, each with its neighbour
            v = rng.standard_normal(1500).astype(np.float32) * (1 if dtype == np.float32 else 1 << 24)
            x = rng.choice(np.concatenate([v, np.nextafter(v, np.float32(np.inf)) if dtype == np.float32 else v + 1]), n)
        else:
            x = _spread(rng, dtype, n, kind)
        _device_sort_check(rk, np.ascontiguousarray(x.astype(dtype)), (False, True) if n == n0 else (False,))


def _moved_into_buckets(rk, x):
    """Whether a sort of the keys went through buckets: it leaves a number of passes that none has."""
    return _passes_run(rk, x, False)[0] == 0xffffffff


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("near,width", [(1000, 1), (9000, 1), (15000, 64), (20000, 1), (18000, 8192), (60000, 1)])
def test_bucket_with_a_cluster(rk, dtype, near, width):
    """`near` keys among `width` times the values of a bin: many rounds of merges, bins that are sorted in memory, and a cluster that is larger than
    a bucket may be, which a value of its own or the radix passes take."""
    rng = np.random.default_rng(near)
    n = QUANTILES[dtype] + 12345
    span = 1 << 30 if dtype == np.int32 else 1 << 22     # of Float32: of the bits of one binade, so that cells are lines of equal slope
    x = rng.integers(0, span, n)
    bucket = span // 256 if dtype == np.float32 else span // 512
    at = span // 3
    x[rng.choice(n, near, replace=False)] = at + rng.integers(0, max(2, min(bucket // 8192 * width, bucket)), near)
    x = (x + (127 << 23)).astype(np.uint32).view(np.float32) if dtype == np.float32 else x.astype(np.int32)
    _device_sort_check(rk, x, (False,))


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("near,values", [(36000, 40), (40000, 40), (36000, 20000), (40000, 200)])
def test_bucket_that_does_not_fit_one_window(rk, dtype, near, values):
    """A cluster inside one cell, of more keys than lie in LDS at a time (31920) and fewer than a bucket's workgroup holds (49152), none of its values
    frequent: 20000 neighbours spread over many bins are sorted a window after the other; of 40 in one bin or two, or 200 in few, a bin exceeds half a window,
    and the bucket is sorted in memory."""
    rng = np.random.default_rng(near + values)
    n = QUANTILES[dtype] + 12345
    span = 1 << 30 if dtype == np.int32 else 1 << 27     # (of Float32: of their bits, 16 binades)
    x = rng.integers(0, span, n)
    at = span // 4096 * 1365 + span // 16384             # in the middle of a cell, away from a bucket's end
    x[rng.choice(n, near, replace=False)] = at + rng.integers(0, values, near)
    x = (x + (120 << 23)).astype(np.uint32).view(np.float32) if dtype == np.float32 else x.astype(np.int32)
    assert _moved_into_buckets(rk, x)
    _device_sort_check(rk, x)


SENTINELS = {                                            # keys around a number, a share of them replaced
    "zeros": (1000, 1, 0.001, (0,)), "few zeros": (300, 10, 0.0001, (0,)), "missing": (20, 5, 0.03, (-9999,)), "nine in ten": (0, 1, 0.9, (0,)),
    "four": (20, 5, 0.3, (-9999, 0, 1e6, 2e6)), "half": (0, 1, 0.5, (0.25,)), "nothing else": (0, 1, 1.0, (7, 70_000, 1 << 20))}


@pytest.mark.parametrize("dtype,kind", [(t, k) for t in (np.float32, np.int32) for k in SENTINELS] + [(np.float32, "NaN"), (np.float32, "infinities")])
def test_sorts_of_keys_with_a_value_in_large_numbers(rk, orc, dtype, kind):
    """A few values that stand for many keys, or that lie far from all the others: they have buckets of their own, the table covers the rest, and
    the keys are moved once."""
    rng = np.random.default_rng(43)
    for n in (QUANTILES[dtype], 24576 * 344 + 1):
        mean, width, share, values = SENTINELS.get(kind, (1013, 10, 0.03, (np.nan,) if kind == "NaN" else (np.inf, -np.inf, np.nan)))
        x = mean + width * rng.standard_normal(n)
        if dtype == np.int32:
            x *= 100_000                                 # (three digits and more)
        at = rng.random(n) < share
        x[at] = rng.choice(np.array(values), int(at.sum()))
        x = x.astype(dtype)
        x[x == 0] = 0
        assert _moved_into_buckets(rk, x), n
        if kind not in ("NaN", "infinities"):
            _device_sort_check(rk, x, (False, True))
            continue
        for rev in (False, True):
            want = orc.sort(x, rev)
            y = rk.ROCArray(x)
            assert np.array_equal(rk.Array(rk.sort(y, rev=rev)).view(np.uint32), want.view(np.uint32))
            rk.sort_(y, rev=rev)
            assert np.array_equal(rk.Array(y).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
def test_sorts_by_quantiles_with_a_sample_that_misleads(rk, dtype):
    """The keys that are sampled are spread and larger than nearly all the others, which go to the first bucket: the sample says that the buckets
    fit, the count that they do not, and nothing has been moved yet.  The rule of the sample is that of the source, so that a change there shows here."""
    import pathlib
    text = (pathlib.Path(__file__).parent.parent / "amdgpu.jl_amd" / "csrc" / "rk_sort_quantiles.hpp").read_text()
    for line in ("constexpr uint32_t SQ_GROUP = 16;", "uint32_t h = (g + 1u) * 0x9e3779b1u;", "h ^= h >> 15;", "h *= 0x85ebca77u;",
                 "keys[a + __umulhi(h, b - a - (SQ_GROUP - 1u)) + s % SQ_GROUP]", "return n <= (int64_t)1 << 25 ? 512u : 256u;", "constexpr uint32_t SQ_SAMPLES_EACH = 4;", "constexpr int64_t SQ_MEAN = 26624;"):
        assert line in text, line
    rng = np.random.default_rng(44)
    n = QUANTILES[dtype] + 54321
    groups = -(-n // (256 * 26624)) * 256 * 512 // 16
    g, m = np.arange(groups, dtype=np.uint64), np.uint64(0xffffffff)
    a, b = g * np.uint64(n) // np.uint64(groups), (g + np.uint64(1)) * np.uint64(n) // np.uint64(groups)
    h = (g + np.uint64(1)) * np.uint64(0x9e3779b1) & m
    h ^= h >> np.uint64(15)
    h = h * np.uint64(0x85ebca77) & m
    at = ((a + (h * (b - a - np.uint64(15)) >> np.uint64(32)))[:, None] + np.arange(16, dtype=np.uint64)).reshape(-1).astype(np.int64)
    x = rng.integers(0, 1 << 20, n)
    x[at] = (1 << 24) + rng.integers(0, 1 << 24, at.size)
    x = (x * 1.5).astype(np.float32) if dtype == np.float32 else x.astype(np.int32)
    assert not _moved_into_buckets(rk, x)
    _device_sort_check(rk, x)


@pytest.mark.parametrize("n", [1 << 24, 1 << 25, (1 << 26) - 24575, 1 << 26, (1 << 26) + 1])
def test_long_sorts_of_floats(rk, n):
    """2^26 keys are the most that go into buckets; the next length takes radix passes."""
    x = np.random.default_rng(n).standard_normal(n, dtype=np.float32)
    x[x == 0] = 0                                        # (some are -0.0)
    _device_sort_check(rk, x, (False,))


def test_sorts_by_quantiles_keep_special_floats_and_neighbours(rk, orc):
    """NaNs of every bit pattern, infinities, zeros of both signs, at both ends of a view that starts at an odd element."""
    n = QUANTILES[np.float32] + 77
    rng = np.random.default_rng(42)
    x = rng.standard_normal(n + 8).astype(np.float32)
    u = x.view(np.uint32)
    bits = np.array([0xffc00001, 0x7fc12345, 0x7f800001, 0xff800001, 0x7fffffff, 0x7f800000, 0xff800000, 0x80000000, 0, 1, 0x80000001, 0x7f7fffff], dtype=np.uint32)
    u[rng.choice(n, 6000, replace=False)] = rng.choice(bits, 6000)
    for rev in (False, True):
        d = rk.ROCArray(x.copy())
        rk.sort_(d.view_range(4, n + 3), rev=rev)
        whole = rk.Array(d)
        got, src = whole[3:n + 3], x[3:n + 3]
        assert np.array_equal(whole[:3].view(np.uint32), u[:3]) and np.array_equal(whole[n + 3:].view(np.uint32), u[n + 3:])
        assert np.array_equal(np.sort(got.view(np.uint32)), np.sort(src.view(np.uint32)))
        want = orc.sort(src, rev)
        assert np.array_equal(got, want, equal_nan=True) and np.array_equal(np.signbit(got[~np.isnan(got)]), np.signbit(want[~np.isnan(want)]))
