"""Routes that once cost more than another the library has for the same bytes: one call's time against its neighbour's,
both replayed in graphs, in turn, the least of several. The bars lie midway between what the route took and what it takes."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _us(*routes, calls: int = 10) -> list[float]:  # noqa: ANN002
    """Microseconds per call of each route, replayed in turn: the least of 12 runs."""
    graphs = []
    for call in routes:
        for _ in range(2):
            call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(calls):
                call()
        graphs.append(graph)
    best = [float("inf")] * len(graphs)
    for _ in range(12):
        for i, graph in enumerate(graphs):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            start.record()
            for _ in range(4):
                graph.replay()
            end.record()
            torch.cuda.synchronize()
            best[i] = min(best[i], start.elapsed_time(end) / (4 * calls) * 1e3)
    return best


def _records(h: int, n: int, bs: int, d: int, dt: torch.dtype):  # noqa: ANN202
    from lazykv_amd import kernels
    from lazykv_amd.quant import pack

    pool = torch.randn((n, h, 2, bs, d), device="cuda").to(dt)
    return kernels.record_source(pack(pool), dt)


@pytest.mark.parametrize(("h", "g", "bs", "tokens", "k"), [(8, 1, 256, 4096, 6), (32, 1, 256, 4096, 6), (4, 2, 64, 16384, 60), (8, 1, 16, 2000, 20)])
def test_a_model_query_attends_a_remainder_of_records_no_slower_than_a_float32_one(h: int, g: int, bs: int, tokens: int, k: int) -> None:
    """The matrix-core launch (a query of the model's dtype) against the vector one (a float32 query): 41.7 us against 24.5 where a
    wave held whole 256-token blocks, in four slots whatever it had; now 20.9."""
    from lazykv_amd import kernels

    d, dt, n = 64, torch.float16, tokens // bs
    src = _records(h, n, bs, d, dt)
    idx = torch.stack([torch.randperm(n - 1, device="cuda")[:k].sort().values + 1 for _ in range(h)]).to(torch.int32)
    q = torch.randn((h * g, d), device="cuda")
    lse = torch.empty(h * g, device="cuda")

    def route(qq):  # noqa: ANN001, ANN202
        out, ws = torch.empty_like(qq), kernels.Workspace()
        return lambda: kernels.sparse_decode(qq, n_kv=h, block_size=bs, scale=d**-0.5, sel=src, idx=idx, rem=src, rem_range=(0, n), out=out, lse=lse, ws=ws)

    times = _us(route(q.to(dt)), route(q))
    print(f"remainder of records h={h} g={g} bs={bs}: model query {times[0]:.1f} us, float32 {times[1]:.1f}", flush=True)
    assert times[0] < 1.25 * times[1]


@pytest.mark.parametrize(("records", "bar"), [(False, 0.61), (True, 0.475)])
def test_small_blocks_pay_for_their_own_rows(records: bool, bar: float) -> None:
    """Blocks of 4 tokens fill a quarter of the matrix cores' 16-row chunks: the value rows that a block does not have cost nothing.
    Against a float32 query on the vector path, which skips them too: 38.1 us against 55.6 (pairs) and 54.6 against 100.9 (records)
    with the rows masked; now 29.6 and 41.6."""
    from lazykv_amd import kernels

    h, g, d, bs, n, k, dt = 8, 4, 128, 4, 4096, 600, torch.bfloat16
    pool = torch.randn((n, h, 2, bs, d), device="cuda").to(dt)
    src = _records(h, n, bs, d, dt) if records else kernels.pool_source(pool)
    idx = torch.stack([torch.randperm(n - 1, device="cuda")[:k].sort().values + 1 for _ in range(h)]).to(torch.int32)
    q = torch.randn((h * g, d), device="cuda")
    lse = torch.empty(h * g, device="cuda")

    def route(qq):  # noqa: ANN001, ANN202
        out, ws = torch.empty_like(qq), kernels.Workspace()
        return lambda: kernels.sparse_decode(qq, n_kv=h, block_size=bs, scale=d**-0.5, sel=src, idx=idx, rem=src, rem_range=(0, n), out=out, lse=lse, ws=ws)

    times = _us(route(q.to(dt)), route(q))
    print(f"4-token blocks, records={records}: model query {times[0]:.1f} us, float32 {times[1]:.1f}", flush=True)
    assert times[0] < bar * times[1]


@pytest.mark.parametrize("h", [32])
def test_a_model_query_of_one_head_decodes_records_no_slower_than_a_float32_one(h: int) -> None:
    """600 records of 4 tokens a head: 20.2 us on the matrix cores, 15.3 on the vector path that both queries take."""
    from lazykv_amd import kernels

    d, bs, n, k, dt = 64, 4, 4096, 600, torch.float16
    src = _records(h, n, bs, d, dt)
    idx = torch.stack([torch.randperm(n, device="cuda")[:k].sort().values for _ in range(h)]).to(torch.int32)
    q = torch.randn((h, d), device="cuda")
    lse = torch.empty(h, device="cuda")

    def route(qq):  # noqa: ANN001, ANN202
        out, ws = torch.empty_like(qq), kernels.Workspace()
        return lambda: kernels.sparse_decode(qq, n_kv=h, block_size=bs, scale=d**-0.5, sel=src, idx=idx, out=out, lse=lse, ws=ws)

    times = _us(route(q.to(dt)), route(q))
    print(f"records of one head: model query {times[0]:.1f} us, float32 {times[1]:.1f}", flush=True)
    assert times[0] < 1.15 * times[1]


@pytest.mark.parametrize(("d", "bar"), [(64, 2.0), (128, 2.1)])
def test_packing_small_blocks_costs_about_their_bytes(d: int, bar: float) -> None:
    """A layer of 4-token blocks packed with its metadata against the same tokens in 16-token blocks (1.2 times the bytes written): 98 us
    against 35 at d 64 and 157 against 55 at d 128 where every block paid for 16 rows; now 41 and 76."""
    from lazykv_amd import kernels
    from lazykv_amd.quant import packed_pair_bytes

    h, tokens, dt = 8, 32768, torch.float16

    def route(bs: int):  # noqa: ANN202
        n = tokens // bs
        src = kernels.pool_source(torch.randn((n, h, 2, bs, d), device="cuda").to(dt))
        dst = kernels.record_source(torch.empty((n, h, packed_pair_bytes(bs, d)), dtype=torch.uint8, device="cuda"), dt)
        kmin = torch.empty((1, h, n, d), dtype=dt, device="cuda")
        kmax = torch.empty_like(kmin)
        return lambda: kernels.store_blocks(src, dst=dst, n_kv=h, head_dim=d, block_size=bs, first_block=0, n_blocks=n, kmin=kmin, kmax=kmax)

    times = _us(route(4), route(16))
    print(f"packing at d {d}: 4-token blocks {times[0]:.1f} us, 16-token {times[1]:.1f}", flush=True)
    assert times[0] < bar * times[1]


def test_copying_float32_rows_costs_their_bytes() -> None:
    """Blocks of 64 float32 channels against 128 float16 ones, the same bytes: 7.3 us against 6.1 where a lane's two accesses left gaps;
    now 6.1."""
    from lazykv_amd import kernels

    h, n, bs = 8, 256, 16

    def route(d: int, dt: torch.dtype):  # noqa: ANN202
        src = kernels.pool_source(torch.randn((n, h, 2, bs, d), device="cuda").to(dt))
        dst = kernels.dense_source(torch.empty((1, h, n * bs, d), dtype=dt, device="cuda"), torch.empty((1, h, n * bs, d), dtype=dt, device="cuda"), bs)
        return lambda: kernels.store_blocks(src, dst=dst, n_kv=h, head_dim=d, block_size=bs, first_block=0, n_blocks=n)

    times = _us(route(64, torch.float32), route(128, torch.float16))
    print(f"copies: float32 {times[0]:.2f} us, float16 {times[1]:.2f}", flush=True)
    assert times[0] < 1.08 * times[1]


@pytest.mark.parametrize("n", [12286])
def test_selection_from_dense_bounds_reads_them_once(n: int) -> None:
    """Bounds written to the caller's dense rows (not whole 16-byte vectors) against the workspace's padded ones: 18.5 us against 11.3
    where dense rows were read three times; now 13.4."""
    from lazykv_amd import kernels

    h, d, k, dt = 8, 64, n // 16, torch.float16
    a, b = torch.randn((1, h, n, d), device="cuda").to(dt), torch.randn((1, h, n, d), device="cuda").to(dt)
    kmin, kmax = torch.minimum(a, b), torch.maximum(a, b)
    q = torch.randn((4 * h, d), device="cuda").to(dt)
    idx = torch.empty((h, k), dtype=torch.int32, device="cuda")
    dense, ws = torch.empty((h, n), device="cuda"), kernels.Workspace()
    times = _us(lambda: kernels.bound_topk(q, kmin, kmax, k, out_idx=idx, out_bound=dense, ws=ws),
                lambda: kernels.bound_topk(q, kmin, kmax, k, out_idx=idx, ws=ws))
    print(f"selection of {k} of {n}: dense rows {times[0]:.1f} us, padded {times[1]:.1f}", flush=True)
    assert times[0] < 1.4 * times[1]
