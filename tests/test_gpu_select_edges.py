"""Selection at the sizes where its kernels change course, against a sort on the host.

With a one-hot query a block's bound is one metadata value, so the selected ids are known exactly: the
k largest, ties towards the lower id."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bounds(kind: str, n: int, rng: np.random.Generator) -> np.ndarray:
    if kind == "normal":  # few candidates share a value
        return rng.normal(100.0, 20.0, size=n)
    if kind == "cluster":  # the boundary bin holds hundreds of candidates, with ties, beside two outliers
        b = 1.0 + rng.integers(0, 400, size=n) / 1024.0
        b[[n // 3, n // 2]] = (60000.0, -60000.0)
        return b
    if kind == "one value":
        return np.full(n, -0.25)
    return np.sort(rng.normal(0.0, 1.0, size=n))  # "sorted": one thread's run is taken whole


def _metadata(kind: str, h: int, n: int, seed: int):  # noqa: ANN202
    rng = np.random.default_rng(seed)
    values = np.stack([_bounds(kind, n, rng) for _ in range(h)]).astype(np.float16)
    kmax = torch.zeros((1, h, n, 64), dtype=torch.float16)
    kmax[0, :, :, 0] = torch.from_numpy(values)
    q = torch.zeros((h * 4, 64), dtype=torch.float16)
    q[:, 0] = 1.0
    return values.astype(np.float64), kmax.cuda(), q.cuda()


# n around whole runs of 4 to 16 keys a thread (one key left over among them), and k around one and two keys
# a thread of 512 and of 1,024 threads, where the first range starts at another value.
SIZES = [(5, 1), (5, 5), (64, 63), (509, 200), (2045, 511), (2048, 512), (2046, 513), (4093, 1023), (4094, 1024), (4096, 1025), (8185, 1024), (8189, 2047), (8192, 8192)]


@pytest.mark.parametrize("kind", ["normal", "cluster", "one value", "sorted"])
@pytest.mark.parametrize(("n", "k"), SIZES)
def test_selection_in_one_workgroup_takes_the_best_k(n: int, k: int, kind: str) -> None:
    from lazykv_amd import kernels

    h = 2
    values, kmax, q = _metadata(kind, h, n, n + k)
    want = np.stack([np.sort(np.lexsort((np.arange(n), -values[j]))[:k]) for j in range(h)])
    idx = kernels.bound_topk(q, kmax, kmax, k)
    store = torch.zeros((n, h, 2, 16, 64), dtype=torch.float16, device="cuda")
    fused = torch.full((h, k), -1, dtype=torch.int32, device="cuda")
    kernels.select_decode(q, kmax, kmax, k, cand_offset=0, n_cand=n, block_size=16, scale=0.125, sel=kernels.pool_source(store), out_idx=fused)
    assert np.array_equal(idx.cpu().numpy(), want)
    assert np.array_equal(fused.cpu().numpy(), want)


# Around a wave's run of 256 candidates, the in-workgroup limit, and the largest count; k around whole powers
# of two, the sort's own edges.
# Beyond 16,384 candidates in parts of 8,192 while the parts' picks are at most 12,288 (a last part of one candidate, and of
# fewer than k, among them), else in one pass over the row.
LONG = [(3, 2), (255, 64), (257, 65), (4097, 1025), (8193, 700), (12289, 2048), (16385, 2000), (16640, 1), (24577, 2048), (65535, 1024), (65537, 1365), (262144, 384), (262144, 2047)]


@pytest.mark.parametrize("kind", ["normal", "cluster", "one value", "sorted"])
@pytest.mark.parametrize(("n", "k"), LONG)
def test_long_and_sorted_selections_take_the_best_k(n: int, k: int, kind: str) -> None:
    """Ascending and descending, from the workspace's rows and from a caller's dense bounds."""
    from lazykv_amd import kernels

    h = 2
    values, kmax, q = _metadata(kind, h, n, n + k)
    order = [np.lexsort((np.arange(n), -values[j]))[:k] for j in range(h)]
    for sorted_ in (False, True):
        want = np.stack([o if sorted_ else np.sort(o) for o in order])
        got = kernels.bound_topk(q, kmax, kmax, k, sorted_=sorted_)
        dense = torch.empty((h, n), dtype=torch.float32, device="cuda")
        got_dense = kernels.bound_topk(q, kmax, kmax, k, sorted_=sorted_, out_bound=dense)
        assert np.array_equal(got.cpu().numpy(), want), sorted_
        assert np.array_equal(got_dense.cpu().numpy(), want), sorted_
        assert np.array_equal(dense.cpu().numpy().astype(np.float64), values)


@pytest.mark.parametrize(("n", "k"), [(20000, 5000), (20000, 20000), (30001, 29999)])
def test_long_selections_of_many_blocks(n: int, k: int) -> None:
    from lazykv_amd import kernels

    values, kmax, q = _metadata("normal", 2, n, n + k)
    want = np.stack([np.sort(np.lexsort((np.arange(n), -values[j]))[:k]) for j in range(2)])
    assert np.array_equal(kernels.bound_topk(q, kmax, kmax, k).cpu().numpy(), want)


@pytest.mark.parametrize("kind", ["normal", "one value"])
@pytest.mark.parametrize(("n", "k"), [(1, 1), (6, 5), (509, 200), (2045, 511), (4093, 1023), (8189, 2047), (8193, 1025), (12285, 2048), (12287, 3), (12289, 700)])
def test_selection_from_dense_rows_of_any_alignment(n: int, k: int, kind: str) -> None:
    """Rows that are not whole 16-byte vectors, up to the in-workgroup limit and past it; three heads, so that each row starts at another
    alignment."""
    from lazykv_amd import kernels

    h = 3
    values, kmax, q = _metadata(kind, h, n, n + k)
    order = [np.lexsort((np.arange(n), -values[j]))[:k] for j in range(h)]
    dense = torch.empty((h, n), dtype=torch.float32, device="cuda")
    for sorted_ in (False, True):
        want = np.stack([o if sorted_ else np.sort(o) for o in order])
        got = kernels.bound_topk(q, kmax, kmax, k, sorted_=sorted_, out_bound=dense)
        assert np.array_equal(got.cpu().numpy(), want), sorted_
