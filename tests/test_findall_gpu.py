"""GPU parity of findall / logical indexing masks (src/kernels/indexing.jl:8-36, test/hip_rocarray/indexing.jl:5-18)
against the oracle, through the C ABI: the one-pass stream compaction (rk_findall) and the reference's own
cumsum + scatter sequence (rk_accumulate + rk_findall_scatter).  Indices are bit-exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(rk, orc, m):
    from amdgpu_jl_amd.indexing import findall_two_pass
    want = orc.findall(m)
    d = rk.ROCArray(m)
    for fn in (rk.findall, findall_two_pass):
        got = rk.Array(fn(d))
        assert got.dtype == np.int64
        assert np.array_equal(got if m.ndim == 1 else got.T, want), fn.__name__


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 1000, 65535, 65536, 65537, 131072, 1_000_003, (1 << 22) + 5])
@pytest.mark.parametrize("density", [0.0, 0.03, 0.5, 1.0])
def test_findall_vector(rk, orc, n, density):
    _check(rk, orc, np.random.default_rng(n).random(n) < density)


@pytest.mark.parametrize("shape", [(16,), (1, 16), (3, 1, 16), (33, 65), (257, 300, 7), (2, 3, 4, 5, 6, 7), (70000, 3), (1, 1, 200_000)])
def test_findall_shapes(rk, orc, shape):
    # test/hip_rocarray/indexing.jl:5-18 shapes first
    _check(rk, orc, np.random.default_rng(7).random(shape) < 0.5)


def test_findall_unaligned_view_and_patterns(rk, orc):
    b = np.random.default_rng(3).random(200_001) < 0.4
    d = rk.ROCArray(b)
    v = d.view_range(2, 200_001)                               # byte offset 1: the scalar load path
    assert np.array_equal(rk.Array(rk.findall(v)), orc.findall(b[1:]))
    for pat in (np.arange(300_000) % 64 == 63, np.arange(300_000) % 1024 < 3, np.arange(300_000) >= 299_999):
        _check(rk, orc, pat)


def test_findall_repeated_calls_share_the_workspace_with_scans(rk, orc):
    rng = np.random.default_rng(11)
    for it in range(8):
        n = int(rng.integers(70_000, 900_000))
        b = rng.random(n) < rng.random()
        assert np.array_equal(rk.Array(rk.findall(rk.ROCArray(b))), orc.findall(b)), it
        x = rng.integers(-100, 100, n, dtype=np.int32)
        assert np.array_equal(rk.Array(rk.cumsum(rk.ROCArray(x))), orc.cumsum(x)), it


def test_findall_full_size_and_count_out(rk, orc):
    import torch
    from amdgpu_jl_amd import _lib as L
    from amdgpu_jl_amd.array import workspace, stream_ptr
    n = 1 << 26
    b = np.random.default_rng(5).random(n) < 0.25
    d = rk.ROCArray(b)
    total = int(b.sum())
    ys = rk.ROCArray(dims=(total,), dtype=np.int64)
    cnt = rk.ROCArray(dims=(1,), dtype=np.int64)
    shape = L.shape_array((n,))
    ws, ws_bytes = workspace(L.lib.rk_workspace_bytes(L.RK_KIND_FINDALL, L.RK_U8, 1, shape, 0))
    L.check(L.lib.rk_findall(d.ptr, 1, shape, ys.ptr, cnt.ptr, ws, ws_bytes, stream_ptr()), "rk_findall")
    assert int(rk.Array(cnt)[0]) == total
    assert np.array_equal(rk.Array(ys), np.nonzero(b)[0] + 1)
    # selection x[m] == x[findall(m)] (test/hip_rocarray/indexing.jl:8)
    x = np.random.default_rng(6).integers(-2**31, 2**31 - 1, 1 << 20, dtype=np.int32)
    m = np.random.default_rng(7).random(1 << 20) < 0.5
    idx = rk.Array(rk.findall(rk.ROCArray(m)))
    assert np.array_equal(x[idx - 1], x[m])


@pytest.mark.parametrize("dtype", [np.int32, np.float64, np.int16, np.bool_, np.complex128])
def test_selection_by_mask(rk, orc, dtype):
    # test/hip_rocarray/indexing.jl:5-18: x[m], x[:, m], x[:, :, m]
    rng = np.random.default_rng(12)
    def rand(shape):
        return (rng.random(shape) * 1000).astype(dtype) if np.dtype(dtype).kind != "b" else rng.random(shape) < 0.5
    for n in (16, 100_003):
        m = rng.random(n) < 0.5
        md = rk.ROCArray(m)
        for shape in ((n,), (1, n), (3, 1, n), (7, n)):
            x = rand(shape)
            got = rk.Array(rk.getindex_mask(rk.ROCArray(x), md))
            assert np.array_equal(got, x[..., m])
    x = rand((33, 65))
    m2 = rng.random((33, 65)) < 0.3
    got = rk.Array(rk.getindex_mask(rk.ROCArray(x), rk.ROCArray(m2)))
    assert np.array_equal(got, x.reshape(-1, order="F")[m2.reshape(-1, order="F")])        # column-major order of the hits
    with pytest.raises(IndexError):
        rk.getindex_mask(rk.ROCArray(x), rk.ROCArray(np.ones(5, dtype=bool)))
    assert rk.getindex_mask(rk.ROCArray(x), rk.ROCArray(np.zeros((33, 65), dtype=bool))).dims == (0,)


@pytest.mark.parametrize("n", [1, 15, 63, 4095, 4096, 4097, 65535, 65536, 65537, 16 * 65536 + 5, (1 << 24) + 3, (1 << 26) + 4097])
def test_mask_select_edges(rk, n):
    # tile (4096), group (16 or 64 tiles) and completion-ticket edges of the count; every density class of the list in LDS
    rng = np.random.default_rng(n)
    x = rng.integers(0, 1 << 31, n).astype(np.uint32).view(np.float32)
    dx = rk.ROCArray(x)
    for dens in (0.0, 0.01, 0.5, 1.0) if n < 1 << 26 else (0.4,):
        m = rng.random(n) < dens
        if dens == 0.5:
            m[n // 2:] = True                                       # a full stretch behind a mixed one
        got = rk.Array(rk.getindex_mask(dx, rk.ROCArray(m)))
        assert np.array_equal(got.view(np.uint32), x[m].view(np.uint32))


@pytest.mark.parametrize("dtype", [np.int8, np.int16, np.int32, np.int64])
def test_mask_select_unaligned(rk, dtype):
    # mask and x that start at odd addresses (views), element sizes 1 to 8
    rng = np.random.default_rng(3)
    n = 200_003
    x, m = rng.integers(-100, 100, n).astype(dtype), rng.random(n) < 0.3
    dx, dm = rk.ROCArray(x), rk.ROCArray(m)
    for a, b in ((2, n), (8, n - 1), (17, n - 70_000)):
        got = rk.Array(rk.getindex_mask(dx.view_range(a, b), dm.view_range(a, b)))
        assert np.array_equal(got, x[a - 1:b][m[a - 1:b]])


def _mask_calls(rk, mask, x, y, elsize, n, nsel=None, between=None):
    """rk_mask_count and rk_mask_select on raw addresses; `between` runs after the count.  Returns the count."""
    import torch
    from amdgpu_jl_amd import _lib as L
    from amdgpu_jl_amd.array import stream_ptr, workspace
    tmp = torch.empty(int(L.lib.rk_mask_tmp_bytes(n)), dtype=torch.uint8, device="cuda")
    total = torch.full((1,), -1, dtype=torch.int64, device="cuda")
    ws, ws_bytes = workspace()
    L.check(L.lib.rk_mask_count(mask, n, total.data_ptr(), tmp.data_ptr(), tmp.numel(), ws, ws_bytes, stream_ptr()), "count")
    cnt = int(total.item())
    if between is not None:
        between()
    L.check(L.lib.rk_mask_select(mask, n, x, y, elsize, cnt if nsel is None else nsel, tmp.data_ptr(), tmp.numel(), stream_ptr()), "select")
    torch.cuda.synchronize()
    return cnt


@pytest.mark.parametrize("xoff,yoff", [(0, 0), (8, 0), (0, 8), (8, 24)])
def test_mask_select_16_byte_elements(rk, xoff, yoff):
    """Elements of 16 bytes need 8-byte alignment only (ComplexF64, pairs of Int64)."""
    import torch
    rng = np.random.default_rng(xoff + 3 * yoff)
    n = 70_003
    x, m = rng.integers(-2**62, 2**62, (n, 2)), rng.random(n) < 0.4
    dx = torch.zeros(16 * n + 64, dtype=torch.uint8, device="cuda")
    dx[xoff:xoff + 16 * n] = torch.from_numpy(x.view(np.uint8).reshape(-1).copy()).cuda()
    dm, want = torch.from_numpy(m.view(np.uint8).copy()).cuda(), x[m]
    dy = torch.full((16 * len(want) + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    assert dx.data_ptr() % 16 == 0 and dy.data_ptr() % 16 == 0
    assert _mask_calls(rk, dm.data_ptr(), dx.data_ptr() + xoff, dy.data_ptr() + yoff, 16, n) == len(want)
    got = dy.cpu().numpy()
    assert np.array_equal(got[yoff:yoff + 16 * len(want)].view(np.int64).reshape(-1, 2), want)
    assert (got[:yoff] == 0xA5).all() and (got[yoff + 16 * len(want):] == 0xA5).all()


@pytest.mark.parametrize("n", [100, 70_003, (1 << 24) + 5])
def test_mask_bytes_and_the_bound_of_the_result(rk, n):
    """Only bit 0 of a Bool byte counts, and no element is written past nsel: neither with a smaller one than the count nor
    for a mask that gains entries between the two calls."""
    import torch
    rng = np.random.default_rng(n)
    x = rng.integers(0, 1 << 31, n, dtype=np.int32)
    m = rng.choice(np.array([0, 1, 2, 3, 254, 255], dtype=np.uint8), n)
    dx, dm, want = torch.from_numpy(x).cuda(), torch.from_numpy(m).cuda(), x[(m & 1) == 1]
    for nsel in (len(want), len(want) // 2):
        dy = torch.full((len(want) + 16,), -7, dtype=torch.int32, device="cuda")
        assert _mask_calls(rk, dm.data_ptr(), dx.data_ptr(), dy.data_ptr(), 4, n, nsel) == len(want)
        got = dy.cpu().numpy()
        assert np.array_equal(got[:nsel], want[:nsel]) and (got[nsel:] == -7).all()
    dy = torch.full((len(want) + 16,), -7, dtype=torch.int32, device="cuda")
    _mask_calls(rk, dm.data_ptr(), dx.data_ptr(), dy.data_ptr(), 4, n, between=lambda: dm.fill_(1))
    assert (dy.cpu().numpy()[len(want):] == -7).all()


@pytest.mark.parametrize("n", [1, 3, 255, 1023, 1025, 4095, 4097, 70_003, 16 * 4096 + 2])
@pytest.mark.parametrize("elsize", [4, 8])
@pytest.mark.parametrize("xoff,moff", [(0, 0), (0, 4), (0, 1), (8, 0)])
def test_mask_select_of_most_elements(rk, n, elsize, xoff, moff):
    """Masks that select three quarters and more read x whole when x is aligned to 16 bytes and the mask to 4: ends of steps and
    tiles, elements in front of the result and behind it, a result that ends early and a mask that grows."""
    import torch
    rng = np.random.default_rng(n + elsize + moff)
    dt = np.int32 if elsize == 4 else np.int64
    x, m = rng.integers(0, 1 << 30, n).astype(dt), rng.random(n) < 0.85
    m[: n // 2] |= rng.random() < 0.5                              # now and then lanes whose every element is selected
    m[0] = True
    dx = torch.zeros(elsize * n + 64, dtype=torch.uint8, device="cuda")
    dx[xoff:xoff + elsize * n] = torch.from_numpy(x.view(np.uint8).copy()).cuda()
    dm = torch.zeros(n + 64, dtype=torch.uint8, device="cuda")
    dm[moff:moff + n] = torch.from_numpy(m.view(np.uint8).copy()).cuda()
    want = x[m]
    for nsel in (len(want), len(want) - len(want) // 50):
        dy = torch.from_numpy(np.full(len(want) + 16, -7, dtype=dt)).cuda()
        assert _mask_calls(rk, dm.data_ptr() + moff, dx.data_ptr() + xoff, dy.data_ptr(), elsize, n, nsel) == len(want)
        got = dy.cpu().numpy()
        assert np.array_equal(got[:nsel], want[:nsel]) and (got[nsel:] == -7).all()
    dy = torch.from_numpy(np.full(len(want) + 16, -7, dtype=dt)).cuda()
    _mask_calls(rk, dm.data_ptr() + moff, dx.data_ptr() + xoff, dy.data_ptr(), elsize, n, between=lambda: dm.fill_(1))
    assert (dy.cpu().numpy()[len(want):] == -7).all()


@pytest.mark.parametrize("n", [1, 63, 4095, 4096, 4097, (1 << 24) - 1, (1 << 24) + 4097, (1 << 25) + 1])
@pytest.mark.parametrize("elsize", [1, 4, 8])
@pytest.mark.parametrize("share", [0.05, 0.45, 0.55])
def test_mask_bits_of_the_count(rk, n, elsize, share):
    """What the count leaves of a mask at an odd address with bytes other than 0 and 1, one, two and four tiles a wave, shares
    around the lines between the two kernels, and the first and last element of every tile."""
    import torch
    from amdgpu_jl_amd import _lib as L
    from amdgpu_jl_amd.array import stream_ptr, workspace
    gen = torch.Generator(device="cuda").manual_seed(n + elsize)
    dx = torch.randint(0, 256, (n * elsize,), dtype=torch.uint8, device="cuda", generator=gen)
    mask = torch.randint(0, 128, (n + 1,), dtype=torch.uint8, device="cuda", generator=gen) * 2
    m = torch.rand(n, device="cuda", generator=gen) < share
    m[::4096] = True
    m[4095::4096] = True
    mask[1:] += m.to(torch.uint8)
    want = dx.view(n, elsize)[m].reshape(-1)
    tmp = torch.randint(0, 256, (int(L.lib.rk_mask_bits_tmp_bytes(n)),), dtype=torch.uint8, device="cuda", generator=gen)
    total = torch.full((1,), -1, dtype=torch.int64, device="cuda")
    ws, ws_bytes = workspace()
    L.check(L.lib.rk_mask_count_bits(mask.data_ptr() + 1, n, total.data_ptr(), tmp.data_ptr(), tmp.numel(), ws, ws_bytes, stream_ptr()), "count")
    nsel = int(total.item())
    assert nsel * elsize == want.numel()
    for short in (0, nsel // 3):                                   # a result that ends early
        dy = torch.full((want.numel() + 16,), 0xA5, dtype=torch.uint8, device="cuda")
        L.check(L.lib.rk_mask_select_bits(n, dx.data_ptr(), dy.data_ptr(), elsize, nsel - short, tmp.data_ptr(), tmp.numel(), stream_ptr()), "select")
        end = (nsel - short) * elsize
        assert torch.equal(dy[:end], want[:end]) and bool((dy[end:] == 0xA5).all())


@pytest.mark.parametrize("dtype", [np.float32, np.int64])
@pytest.mark.parametrize("hits", ["random", "runs of 10", "first quarter", "every second tile", "last element"])
def test_mask_select_beyond_the_cache(rk, dtype, hits):
    """x beyond 128 MiB is read 16 bytes a lane from an eighth of the elements on, lanes and tiles without a hit left out: hits
    evenly spread, in runs that begin and end inside a lane's elements, in tiles that are full beside empty ones; mask bytes
    other than 0 and 1, of which bit 0 counts."""
    import torch
    rng = np.random.default_rng(5)
    n = (1 << 27) // np.dtype(dtype).itemsize + 4099
    x, i = rng.integers(-1000, 1000, n).astype(dtype), np.arange(n)
    m = {"random": lambda: rng.random(n) < 0.25, "runs of 10": lambda: i % 37 < 10, "first quarter": lambda: i < n // 4,
         "every second tile": lambda: i // 4096 % 2 == 1, "last element": lambda: (i < n // 8 + 1) | (i == n - 1)}[hits]()
    mask = (m + 2 * rng.integers(0, 128, n)).astype(np.uint8)
    dx, dm, want = torch.from_numpy(x).cuda(), torch.from_numpy(mask).cuda(), x[m]
    assert len(want) >= n // 8
    dy = torch.full((len(want) + 16,), -7, dtype=dx.dtype, device="cuda")
    assert _mask_calls(rk, dm.data_ptr(), dx.data_ptr(), dy.data_ptr(), x.itemsize, n) == len(want)
    got = dy.cpu().numpy()
    assert np.array_equal(got[:len(want)], want) and (got[len(want):] == -7).all()


def test_the_paths_the_tunables_select():
    """RK_SELECT_ORDERED=0 (persistent workgroups fed by a tile counter) and RK_SCAN_DYNAMIC_IDS=1 (the same for the
    long scans) are read once per process, so they are exercised in a child process: findall and a long cumsum against
    numpy, several calls on one workspace."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = r'''
import sys
sys.path.insert(0, %r)
import numpy as np
from __graft_entry__ import load_package
rk = load_package()
rng = np.random.default_rng(5)
for n, dens in ((1 << 21) + 77, 0.3), ((1 << 22), 0.01), (300_000, 1.0), (5, 0.5):
    m = rng.random(n) < dens
    got = rk.Array(rk.findall(rk.ROCArray(m)))
    assert np.array_equal(got, np.flatnonzero(m) + 1), (n, dens)
m = rng.random((257, 3001)) < 0.4
got = rk.Array(rk.findall(rk.ROCArray(m)))
want = np.argwhere(m.T)[:, ::-1] + 1                  # column-major order of the hits
assert np.array_equal(got.T, want)
x = rng.integers(-100, 100, size=(1 << 22) + 3).astype(np.int32)
for _ in range(3):
    assert np.array_equal(rk.Array(rk.cumsum(rk.ROCArray(x))), np.cumsum(x, dtype=np.int32))
print("child ok")
''' % root
    env = dict(os.environ, RK_SELECT_ORDERED="0", RK_SCAN_DYNAMIC_IDS="1")
    out = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=110)
    assert out.returncode == 0 and "child ok" in out.stdout, out.stdout[-2000:] + out.stderr[-2000:]
