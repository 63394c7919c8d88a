"""The one-item kernel with every run in 16-byte pairs (FACES_OPT_FLOW 4) at the
edges of its ranges: one element per row, rows one shorter and one longer than
its item length and than twice that, a lone row and plane, every element size it
is compiled for (n = 2 to 16), periodic, open with and without neighbours, the
staged step and the 6-message tree.  Every sum is one fixed tree, so results are
bit-equal to the oracle's."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests import _brute as brute

pytestmark = pytest.mark.gpu

import faces_amd as fa  # noqa: E402

# longest default item per n (elements): fields of this size take the second
SMALL = {2: 64, 3: 32, 4: 16, 5: 10, 6: 8, 7: 5, 8: 4, 9: 3, 10: 2, 11: 2, 12: 2, 13: 2, 14: 1, 15: 1, 16: 1}
LARGE = {2: 64, 3: 32, 4: 24, 5: 10, 6: 12, 7: 8, 8: 6, 9: 4, 10: 3, 11: 2, 12: 2, 13: 2, 14: 1, 15: 1, 16: 1}


def step(torch, u, shape, boundary, rank, lgrid, path, seg, ps=0, sblocks=None, shares=2):
    n, mx, my, mz = shape
    d = torch.from_numpy(u.copy()).to("cuda")
    f = fa.Faces(rank, *lgrid, mx, my, mz, n, boundary=boundary, plane_stride=ps)
    f.set_path(path)
    f.set_option(fa.OPT_FLOW, 4)
    f.set_option(fa.OPT_SEG, seg)
    if sblocks is not None:
        f.set_option(fa.OPT_SURFACE_BLOCKS, sblocks)
    for _ in range(shares):
        f.share(d)
    torch.cuda.synchronize()
    got = d.cpu().numpy()
    f.close()
    return got


@pytest.mark.parametrize("n", range(2, 17))
def test_pairs_edges_bitexact(torch_cuda, n):
    for seg in sorted({SMALL[n], LARGE[n], max(1, LARGE[n] - 1)}):
        for mx in sorted({1, 2, max(1, seg - 1), seg, seg + 1, 2 * seg + 1, 4 * seg + 1}):
            shape = (n, mx, 2, 3) if mx % 2 else (n, mx, 1, 1)
            ps = (n ** 3 * mx * shape[2] + 7) if mx % 3 == 0 else 0
            print("case pairs", shape, seg, ps, flush=True)
            u = oracle.new_field(*shape, fa.FILL_RAND, seed=11 * n + mx, ps=ps)
            want = u.copy()
            for _ in range(2):
                oracle.share_sweep(want, *shape, periodic=True, ps=ps)
            assert np.array_equal(step(torch_cuda, u, shape, fa.PERIODIC, 0, (1, 1, 1), fa.PATH_AUTO, seg, ps), want)
            for rank, path in ((0, fa.PATH_AUTO), (22, fa.PATH_AUTO), (13, fa.PATH_STAGED), (5, fa.PATH_STAGED_DIRECT),
                               (4, fa.PATH_SIX)):
                mask = brute.mask_for_rank(rank, 3, 3, 3)
                want = u.copy()
                for _ in range(2):
                    (oracle.share_six if path == fa.PATH_SIX else oracle.share_staged)(want, *shape, nbr_mask=mask, ps=ps)
                got = step(torch_cuda, u, shape, fa.OPEN, rank, (3, 3, 3), path, seg, ps)
                assert np.array_equal(got, want), (rank, path)


@pytest.mark.parametrize("sblocks", [1, 2, 0, 3])
@pytest.mark.parametrize("n", range(6, 17))
def test_pairs_surface_blocks_bitexact(torch_cuda, n, sblocks):
    """The staged step's surface sums before and after items of every block
    size (256 to 768 threads), as a launch of their own, by the items."""
    for seg in sorted({SMALL[n], LARGE[n]}):
        shape = (n, 2 * seg + 1, 4, 3)
        for rank, path in ((13, fa.PATH_STAGED_DIRECT), (0, fa.PATH_STAGED), (22, fa.PATH_STAGED_DIRECT)):
            print("case pairs surface blocks", shape, seg, rank, path, sblocks, flush=True)
            u = oracle.new_field(*shape, fa.FILL_RAND, seed=90 + n + rank)
            want = u.copy()
            for _ in range(2):
                oracle.share_staged(want, *shape, nbr_mask=brute.mask_for_rank(rank, 3, 3, 3))
            got = step(torch_cuda, u, shape, fa.OPEN, rank, (3, 3, 3), path, seg, sblocks=sblocks)
            assert np.array_equal(got, want), (shape, rank, path)


@pytest.mark.parametrize("sblocks", [1, 2])
@pytest.mark.parametrize("shape", [(7, 48, 40, 32), (13, 30, 20, 14)])
def test_pairs_surface_blocks_large_field(torch_cuda, shape, sblocks):
    """Fields of 128 MiB and more, whose surface blocks run beside items of
    512 and 768 threads: three staged steps of an interior rank."""
    print("case pairs surface blocks large", shape, sblocks, flush=True)
    u = oracle.new_field(*shape, fa.FILL_RAND, seed=95)
    got = step(torch_cuda, u, shape, fa.OPEN, 13, (3, 3, 3), fa.PATH_STAGED_DIRECT, 0, sblocks=sblocks, shares=3)
    for _ in range(3):
        oracle.share_staged(u, *shape, nbr_mask=63)
    assert np.array_equal(got, u)


def test_pairs_special_values(torch_cuda):
    """Infinities, NaN, signed zeros and subnormals go through as the oracle's
    sums give them."""
    shape = (7, 9, 2, 2)
    u = oracle.new_field(*shape, fa.FILL_RAND, seed=3)
    u[::17], u[5::29], u[3::31], u[1::37] = np.inf, -0.0, 5e-324, -np.inf
    u[2::97] = np.nan
    want = u.copy()
    for _ in range(2):
        oracle.share_sweep(want, *shape, periodic=True)
    got = step(torch_cuda, u, shape, fa.PERIODIC, 0, (1, 1, 1), fa.PATH_AUTO, 8)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.array_equal(got[ok].view(np.uint64), want[ok].view(np.uint64))


@pytest.mark.parametrize("shape", [(2, 3, 2, 2), (5, 1, 1, 1), (7, 4, 1, 3), (8, 5, 4, 3), (13, 2, 2, 1), (17, 2, 1, 2)])
def test_surface_open_ranks(torch_cuda, shape):
    """compute = 0 on every rank position of a 3x3x3 grid: the surface sums of
    an open rank in one launch, dense and padded planes, two shares."""
    n, mx, my, mz = shape
    for rank in range(27):
        ps = n ** 3 * mx * my + 5 if rank % 2 else 0
        print("case surface open", shape, rank, ps, flush=True)
        u = oracle.new_field(*shape, fa.FILL_RAND, seed=40 + rank, ps=ps)
        d = torch_cuda.from_numpy(u.copy()).to("cuda")
        f = fa.Faces(rank, 3, 3, 3, mx, my, mz, n, boundary=fa.OPEN, plane_stride=ps)
        for _ in range(2):
            f.share(d, compute=False)
            oracle.share_staged(u, *shape, nbr_mask=brute.mask_for_rank(rank, 3, 3, 3), compute=False, ps=ps)
        torch_cuda.cuda.synchronize()
        got = d.cpu().numpy()
        f.close()
        assert np.array_equal(got, u), rank


@pytest.mark.parametrize("shape", [
    (8, 16, 8, 8), (8, 25, 41, 1),      # 1024 and 1025 one-element items
    (9, 16, 8, 12), (9, 29, 53, 1),     # 1536 and 1537
    (11, 16, 16, 8), (11, 3, 683, 1),   # 2048 and 2049
    (6, 9, 18, 19), (5, 11, 18, 19),    # 1026 items of 4 and of 5
    (4, 13, 6, 5),                      # own runs in pairs, 8 and 5 elements
    (7, 12, 60, 60), (7, 25, 40, 30),   # 6 and 6 elements by the 8-element kernel; 7, 7, 7 and 4
    (8, 37, 41, 22), (9, 30, 23, 34), (10, 16, 26, 30),  # 64 MiB and more: other lengths on open ranks
])
def test_default_item_lengths_bitexact(torch_cuda, shape):
    """The plan's own item lengths on both sides of where their rule changes
    them: periodic, an open rank without and with neighbours, the staged step."""
    n, mx, my, mz = shape
    u = oracle.new_field(*shape, fa.FILL_RAND, seed=77)
    for boundary, rank, lgrid, path in ((fa.PERIODIC, 0, (1, 1, 1), fa.PATH_AUTO), (fa.OPEN, 0, (1, 1, 1), fa.PATH_AUTO),
                                        (fa.OPEN, 4, (3, 3, 3), fa.PATH_AUTO), (fa.OPEN, 22, (3, 3, 3), fa.PATH_STAGED_DIRECT)):
        print("case default lengths", shape, boundary, rank, path, flush=True)
        d = torch_cuda.from_numpy(u.copy()).to("cuda")
        f = fa.Faces(rank, *lgrid, mx, my, mz, n, boundary=boundary)
        f.set_path(path)
        f.share(d)
        torch_cuda.cuda.synchronize()
        f.close()
        want = u.copy()
        if boundary == fa.PERIODIC:
            oracle.share_sweep(want, *shape, periodic=True)
        else:
            oracle.share_staged(want, *shape, nbr_mask=brute.mask_for_rank(rank, *lgrid))
        assert np.array_equal(d.cpu().numpy(), want), (boundary, rank, path)
