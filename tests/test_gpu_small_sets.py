"""GPU tests of the one-launch neighbour map and plan order that coord sets of
at most 4,096 rows take: the map against the oracle's scan (lowest row of
duplicated coords), the order against numpy, on both sides of the limit."""
import numpy as np
import pytest
import torch

from bevy_synth_amd import flex_gmm as F
from bevy_synth_amd import synth
from tests.test_gpu_plan import check_plan, dev, ocfg

pytestmark = pytest.mark.gpu

LIMIT = 4096


def make(kind, n, seed=0):
    """Coords [n, 4] of the given kind, and the plan's ordering mode for them."""
    rng = np.random.default_rng(seed + n)
    base = synth.sphere_shell_coords(48, 20.0, 1.0, (24.0,) * 3)[:n]
    assert len(base) == n
    if kind == "sorted":
        return base, 3 if n > 1 else 2
    if kind == "shuffled":
        return base[rng.permutation(n)], 1 if n > 1 else 2
    if kind == "duplicates":  # about a third of the rows repeat another, in any order
        c = base[rng.integers(0, max(1, n // 2), n)].copy()
        c[:, 0] = rng.integers(0, 2, n)
        return c, 1
    if kind == "wide":  # a box beyond the grid: the sort by bricks, duplicates included
        c = base.copy()
        c[:, 1] += rng.integers(0, 4, n).astype(np.int32) * 5000
        c[: n // 8] = c[n - n // 8:] if n >= 8 else c[: n // 8]
        return c[rng.permutation(n)], 0
    if kind == "clump":  # every row in one brick but one far away
        c = np.zeros((n, 4), np.int32)
        c[:, 1:] = rng.integers(0, 8, (n, 3))
        c[-1, 1:] = 1 << 20
        return c, 0
    if kind == "sorted_past_lds":  # sorted, 1-2 M cells: more than the LDS bitmap holds
        c = base.copy()
        c[n // 2:, 1] += 390
        return c, 3
    levels = synth.sphere_shell_coords(16, 6.0, 1.0, (8.0,) * 3)
    for _ in range(3):
        levels = synth.child_expand(levels, (rng.random((len(levels), 8)) < 0.3).astype(np.uint8))
    return levels[:n], 2


def expected_order(c, mode):
    n = len(c)
    if mode == 2:
        return np.arange(n)
    q = c.astype(np.int64) - c.min(0)
    shift = 3
    if mode == 0:
        cap = (max(2 * n, 4096) + 1023) // 1024 * 1024
        ext = q.max(0) + 1
        while ext[0] * np.prod(((ext[1:] - 1) >> shift) + 1, dtype=object) > cap:
            shift += 1
    nb = np.r_[q[:, 0].max() + 1, (q[:, 1:].max(0) >> shift) + 1]
    brick = ((q[:, 0] * nb[1] + (q[:, 1] >> shift)) * nb[2] + (q[:, 2] >> shift)) * nb[3] + (q[:, 3] >> shift)
    if mode == 0:
        return np.lexsort((np.arange(n), brick))
    cell = brick * 512 + (q[:, 1] & 7) * 64 + (q[:, 2] & 7) * 8 + (q[:, 3] & 7)
    by = np.lexsort((np.arange(n), cell))
    first = np.r_[True, cell[by][1:] != cell[by][:-1]]
    return np.concatenate([by[first], np.sort(by[~first])])


@pytest.mark.parametrize("kind", ["sorted", "shuffled", "duplicates", "wide", "clump", "sorted_past_lds", "octree"])
@pytest.mark.parametrize("n", [1, 60, 257, 1025, LIMIT - 1, LIMIT, LIMIT + 1])
def test_small_order_and_map(oracle, kind, n):
    if n < 16 and kind in ("wide", "clump", "sorted_past_lds", "duplicates"):
        pytest.skip("needs a box of its own")
    coords, mode = make(kind, n)
    n = len(coords)
    cfg = F.SparseSubmConvConfig(32, 32)
    cd = dev(coords)
    ws = F.NeighborMapWorkspace()
    nbr = F.neighbor_rows_tensor_from_coords_tensor(cfg, cd, workspace=ws)
    assert F.neighbor_map_one_launch(ws.get(n)) == (n <= LIMIT)
    assert np.array_equal(nbr.cpu().numpy(), oracle.build_neighbor_rows_scan(ocfg(oracle, cfg), coords))
    h = check_plan(F.build_conv_plan(cfg, cd, nbr), nbr.cpu().numpy(), n)
    assert h["grid_mode"] == mode
    # past the limit, a brick of more than 512 rows keeps the scatter's order
    if not (n > LIMIT and kind == "clump"):
        assert np.array_equal(h["order"].ravel()[:n], expected_order(coords, mode))
    if mode == 1:
        assert h["n_unique"] == len(np.unique(coords, axis=0)) == n - h["n_extras"]


@pytest.mark.parametrize("kernel,order,sign,n,q", [
    ((3, 3, 1), (2, 0, 1), (1, -1, 1), 700, 300), ((1, 1, 1), (0, 1, 2), (1, 1, 1), 65, 64),
    ((2, 4, 4), (1, 2, 0), (-1, 1, -1), LIMIT, 4000), ((3, 3, 3), (0, 1, 2), (1, 1, 1), 500, 0)])
def test_small_map_kernels(oracle, kernel, order, sign, n, q):
    cfg = F.SparseSubmConvConfig(1, 1, *kernel, axis_order=order, axis_sign=sign)
    coords, _ = make("duplicates", n)
    got = F.neighbor_rows_tensor_from_coords_tensor(cfg, dev(coords), query_rows=q).cpu().numpy()
    assert np.array_equal(got, oracle.build_neighbor_rows_scan(ocfg(oracle, cfg), coords)[:q])


def test_small_map_edges_of_the_coord_range(oracle):
    """Coords at 0 and at INT_MAX (a step past either is absent), and a set
    with a negative coord: reported, and mapped to -1 everywhere."""
    top = 2**31 - 1
    c = np.array([[0, 0, 0, 0], [0, 0, 0, 1], [0, top, top, top], [0, top, top, top - 1], [top, 0, 0, 0]], np.int32)
    cfg = F.SparseSubmConvConfig(1, 1)
    got = F.neighbor_rows_tensor_from_coords_tensor(cfg, dev(c)).cpu().numpy()
    assert np.array_equal(got, oracle.build_neighbor_rows_scan(ocfg(oracle, cfg), c))
    c[1, 3] = -1
    ws = F.NeighborMapWorkspace().get(len(c))
    out = torch.zeros((len(c), 27), dtype=torch.int32, device="cuda")
    F.neighbor_map_build_into(cfg, dev(c), out, ws)
    assert (out == -1).all() and F.neighbor_map_table_mode(ws) == "none"
    with pytest.raises(F.SparseConvError):
        F.neighbor_map_check(ws)


def test_status_words_of_several_threads():
    """The checks of concurrent calls read their own status: only the threads
    whose coords are negative are refused, on every repetition."""
    import threading

    cfg = F.SparseSubmConvConfig(32, 32)
    wrong = []

    def work(i):
        c = torch.randint(0, 20, (500 + i, 4), dtype=torch.int32)
        c[:, 0] = 0
        if i % 2:
            c[i, 1] = -1
        with torch.cuda.stream(torch.cuda.Stream()):
            c = c.cuda()
            for _ in range(20):
                try:
                    F.neighbor_rows_tensor_from_coords_tensor(cfg, c)
                    refused = False
                except Exception:
                    refused = True
                if refused != bool(i % 2):
                    wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
