"""The calls whose speed is watched: decode steps, selection, the tier's stores and a dense decode.

Every case is one call (or one replayed step) of the public entry points with the inputs a decoding
program has in hand. Shapes are the 1B and 8B ones of the benchmark (32 query heads over 8 KV heads,
head_dim 64 in float16 or 128 in bfloat16, 16-token blocks), and, for drawn cases, sizes around them:
other groups of query heads, block sizes, budgets and odd context lengths.

The cases that read or write mapped host memory (host, hybrid, exact, build) are bound by the host
link, not by HBM; `work` counts their bytes all the same.
"""

from __future__ import annotations

import math

import torch

from lazykv_amd import kernels
from lazykv_amd.attention import attend
from lazykv_amd.cache import FullGPUCache
from lazykv_amd.quant import pack, packed_pair_bytes, unpack
from lazykv_amd.selection import QuestView, blocks_for_budget, top_blocks
from lazykv_amd.tiered import DenseScratch, TieredLayer, allocate_host_pools

DEV = "cuda"
TYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
HYBRID_STEPS = 4
HYBRID_DRIFT = 0.3  # of the query's size, per step


def _case(name: str, kind: str, dtype: str, d: int, tokens: int, k: int, layers: int = 1, h: int = 8, g: int = 4, bs: int = 16, **more) -> dict:
    return {"name": name, "kind": kind, "dtype": dtype, "d": d, "tokens": tokens, "k": k, "layers": layers, "h": h, "g": g, "bs": bs, **more}


def listed() -> list[dict]:
    return [
        # A short chat over a dense HBM cache: one layer's selection and attention, called eagerly as
        # a model's attention function calls it. Launches and host time are most of it.
        _case("select_4k", "select", "f16", 64, 4099, 62),
        # The 1B-shaped decode step at 32K tokens, all KV in HBM, all 16 layers in one replayed graph.
        _case("step_1b_32k", "step", "f16", 64, 32768, 512, layers=16),
        # The 1B-shaped step at 64K tokens with the sealed blocks as int8 records in HBM.
        _case("step_1b_64k_int8", "step", "f16", 64, 65536, 1024, layers=16, int8=True),
        # The 8B-shaped step at 128K tokens and a 6.25% budget, all KV in HBM.
        _case("step_8b_128k", "step", "bf16", 128, 131072, 512, layers=4),
        # The same step of one layer with every block in mapped host memory, read in place.
        _case("host_8b_128k", "host", "bf16", 128, 131072, 512),
        # Four steps of the hybrid tier (a slot in HBM for each selected block) under a drifting query.
        _case("hybrid_8b_64k", "hybrid", "bf16", 128, 65536, 256),
        # Exact attention: the selected blocks from HBM, all the others as int8 records in host memory.
        _case("exact_8b_32k_int8", "exact", "bf16", 128, 32768, 128, int8=True),
        # A dense layer's decode (the first two layers of a model, or no selection at all).
        _case("dense_8b_128k", "dense", "bf16", 128, 131065, 0),
        # Block ids in descending order of their bound over a context of a million tokens.
        _case("rank_8b_1m", "rank", "bf16", 128, 1048560, 1024),
        # A 64K-token layer packed into int8 records and unpacked again.
        _case("int8_1b_64k", "int8", "f16", 64, 65536, 0),
        # A user's turn of 200 tokens over a tier kept in HBM: the layer's KV assembled densely.
        _case("turn_8b_64k", "turn", "bf16", 128, 65541, 256, turn=200),
        # The end of a prefill: a layer's KV into int8 records in host memory, with its metadata.
        _case("build_8b_32k_int8", "build", "bf16", 128, 32775, 128, int8=True),
    ]


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(("select", "step", "step", "step", "host", "hybrid", "exact", "dense", "dense", "rank", "int8", "int8", "turn", "build"))
    dtype = rng.choice(("f16", "bf16"))
    d = rng.choice((64, 128))
    bs = rng.choice((16, 16, 16, 32, 64))
    h, g = rng.choice(((8, 4), (8, 4), (8, 4), (8, 8), (8, 1), (4, 4), (16, 2)))
    top = {"select": 32768, "step": 131072, "host": 65536, "hybrid": 32768, "exact": 16384, "dense": 131072, "rank": 1048560, "int8": 65536,
           "turn": 32768, "build": 16384}[kind]
    tokens = _log(rng, 2048, top)
    if h == 16:
        tokens = max(2048, tokens // 2)
    n = tokens // bs
    budget = rng.choice((0.0625, 0.125, 0.25))
    k = max(1, min(blocks_for_budget(budget, tokens, bs), n - 4, 2048))
    more = {}
    layers = 1
    if kind == "step":
        layers = rng.choice((2, 4))
        if rng.random() < 0.4:
            more["int8"] = True
    if kind == "rank":
        k = min(k, 2048)
    if kind in ("exact", "build"):
        more["int8"] = True
    if kind == "hybrid" and rng.random() < 0.5:
        more["int8"] = True
    if kind == "turn":
        more["turn"] = _log(rng, 2, 512)
    if kind == "dense":
        k = 0
        bs = 16
    return _case("drawn", kind, dtype, d, tokens, k, layers=layers, h=h, g=g, bs=bs, **more)


# -- inputs -----------------------------------------------------------------------------------------


def _generator(seed: int, layer: int, what: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed((seed * 64 + layer) * 8 + what)


def _kv(case: dict, seed: int, layer: int = 0) -> tuple[torch.Tensor, torch.Tensor]:
    """Keys and values [1, h, tokens, d]: normal, with a scale per channel in [0.5, 2]."""
    h, t, d = case["h"], case["tokens"], case["d"]
    got = []
    for what in (0, 1):
        g = _generator(seed, layer, what)
        scale = torch.rand((1, h, 1, d), generator=g, device=DEV) * 1.5 + 0.5
        x = torch.randn((1, h, t, d), generator=g, device=DEV)
        got.append(x.mul_(scale).to(TYPES[case["dtype"]]))
        del x
    return got[0], got[1]


def _query(case: dict, seed: int, layer: int = 0) -> torch.Tensor:
    n_q, d = case["h"] * case["g"], case["d"]
    return torch.randn((n_q, d), generator=_generator(seed, layer, 2), device=DEV).to(TYPES[case["dtype"]])


def _queries(case: dict, seed: int) -> list[torch.Tensor]:
    """The hybrid tier's queries: one step's is the base plus a fresh drift."""
    base = torch.randn((case["h"] * case["g"], case["d"]), generator=_generator(seed, 0, 2), device=DEV)
    g = _generator(seed, 0, 3)
    return [(base + HYBRID_DRIFT * torch.randn(base.shape, generator=g, device=DEV)).to(TYPES[case["dtype"]]) for _ in range(HYBRID_STEPS)]


def _extent(case: dict) -> tuple[int, int]:
    """(sealed blocks, tokens in the current block). In a decode a block that has just filled is still
    current; a tier built from a prompt seals every full block of it."""
    n, fill = divmod(case["tokens"], case["bs"])
    return (n - 1, case["bs"]) if fill == 0 and case["kind"] in ("select", "step") else (n, fill)


# -- prepare and run --------------------------------------------------------------------------------


def prepare(case: dict, seed: int) -> dict:
    st = {"case": case, "kind": case["kind"]}
    return {"select": _prepare_select, "step": _prepare_step, "host": _prepare_layer, "hybrid": _prepare_layer, "exact": _prepare_layer,
            "dense": _prepare_dense, "rank": _prepare_rank, "int8": _prepare_int8, "turn": _prepare_turn, "build": _prepare_build}[case["kind"]](case, seed, st)


def _prepare_select(case: dict, seed: int, st: dict) -> dict:
    k, v = _kv(case, seed)
    full = FullGPUCache.from_kv([(k, v)], case["tokens"] + 64)
    st["view"] = QuestView(full, case["k"], case["bs"], dense_layers=0, bound_dtype=torch.float32)
    st["q"] = _query(case, seed).view(1, -1, 1, case["d"])
    return st


def _prepare_step(case: dict, seed: int, st: dict) -> dict:
    """Every layer's sealed blocks in an HBM pool, the sink and the current block in a slot pool, and
    the layers' prepared calls captured once."""
    h, d, bs, L = case["h"], case["d"], case["bs"], case["layers"]
    dt = TYPES[case["dtype"]]
    n_q = h * case["g"]
    n, fill = _extent(case)
    out = torch.empty((L, n_q, d), dtype=dt, device=DEV)
    lse = torch.empty((L, n_q), dtype=torch.float32, device=DEV)
    ws = kernels.Workspace(torch.device(DEV, torch.cuda.current_device()))
    calls, keep = [], []
    for layer in range(L):
        keys, values = _kv(case, seed, layer)
        src = kernels.dense_source(keys, values, bs)
        kmin = torch.zeros((1, h, n, d), dtype=dt, device=DEV)
        kmax = torch.zeros_like(kmin)
        if case.get("int8"):
            pool = torch.empty((n, h, packed_pair_bytes(bs, d)), dtype=torch.uint8, device=DEV)
            sel = kernels.record_source(pool, dt)
        else:
            pool = torch.empty((n, h, 2, bs, d), dtype=dt, device=DEV)
            sel = kernels.pool_source(pool)
        kernels.store_blocks(src, dst=sel, n_kv=h, head_dim=d, block_size=bs, first_block=0, n_blocks=n, kmin=kmin, kmax=kmax)
        slots = torch.zeros((2, h, 2, bs, d), dtype=dt, device=DEV)
        for i, x in enumerate((keys, values)):
            slots[0, :, i] = x[0, :, :bs]
            slots[1, :, i, :fill] = x[0, :, n * bs : n * bs + fill]
        two = kernels.pool_source(slots)
        q = _query(case, seed, layer)
        calls.append(kernels.PreparedSelectDecode(q, kmin, kmax, case["k"], cand_offset=1, n_cand=n - 1, block_size=bs, scale=d**-0.5, sel=sel, sink=two, sink_block=0,
                                                  cur=two, cur_block=1, fill=fill, out=out[layer], lse=lse[layer], ws=ws))
        keep.append((kmin, kmax, pool, slots, q))
        del keys, values, src
    for call in calls:
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for call in calls:
            call()
    st.update(graph=graph, out=out, lse=lse, keep=(calls, keep, ws))
    return st


def _prepare_layer(case: dict, seed: int, st: dict) -> dict:
    """One tiered layer built from a prompt's KV: zero-copy ("host"), the reference's slotted fetch
    ("hybrid"), or the exact split over an HBM store ("exact")."""
    keys, values = _kv(case, seed)
    more = {"host": {"fetch": "zerocopy"}, "hybrid": {"fetch": "runs"}, "exact": {"fetch": "resident", "exact": True}}[case["kind"]]
    st["layer"] = TieredLayer(keys, values, case["k"], case["bs"], case["tokens"] + 64, quant="int8" if case.get("int8") else None, **more)
    st["q"] = _queries(case, seed) if case["kind"] == "hybrid" else [_query(case, seed)]
    st["q"] = [q.view(1, -1, 1, case["d"]) for q in st["q"]]
    st["ws"] = kernels.Workspace(torch.device(DEV, torch.cuda.current_device()))
    return st


def _prepare_dense(case: dict, seed: int, st: dict) -> dict:
    keys, values = _kv(case, seed)
    full = FullGPUCache.from_kv([(keys, values)], case["tokens"] + 64)
    layer = full.layers[0]
    st["full"] = full
    st["kv"] = (layer.keys[:, :, : case["tokens"]], layer.values[:, :, : case["tokens"]])
    st["q"] = _query(case, seed).view(1, -1, 1, case["d"])
    return st


def _rank_metadata(case: dict, seed: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Block minima and maxima [1, h, n, d] of a context that is not kept: n normal channel ranges."""
    shape = (1, case["h"], case["tokens"] // case["bs"], case["d"])
    g = _generator(seed, 0, 4)
    scale = torch.rand((1, case["h"], 1, case["d"]), generator=g, device=DEV) * 1.5 + 0.5
    a = torch.randn(shape, generator=g, device=DEV).mul_(0.5).sub_(1.75).mul_(scale)
    b = torch.randn(shape, generator=g, device=DEV).mul_(0.5).add_(1.75).mul_(scale)
    dt = TYPES[case["dtype"]]
    return torch.minimum(a, b).to(dt), torch.maximum(a, b).to(dt)


def _prepare_rank(case: dict, seed: int, st: dict) -> dict:
    st["meta"] = _rank_metadata(case, seed)
    st["q"] = _query(case, seed).view(1, -1, 1, case["d"])
    return st


def _prepare_int8(case: dict, seed: int, st: dict) -> dict:
    h, d, bs = case["h"], case["d"], case["bs"]
    n = case["tokens"] // bs
    keys, values = _kv(case, seed)
    pairs = torch.stack([x[0, :, : n * bs].reshape(h, n, bs, d) for x in (keys, values)], dim=2)  # [h, n, 2, bs, d]
    st["pairs"] = pairs.transpose(0, 1).contiguous()
    return st


def _prepare_turn(case: dict, seed: int, st: dict) -> dict:
    keys, values = _kv(case, seed)
    st["layer"] = TieredLayer(keys, values, case["k"], case["bs"], case["tokens"] + 64, fetch="resident")
    new = dict(case, tokens=case["turn"])
    st["new"] = _kv(new, seed, 1)
    st["scratch"] = DenseScratch()
    return st


def _prepare_build(case: dict, seed: int, st: dict) -> dict:
    st["kv"] = _kv(case, seed)
    st["host"] = allocate_host_pools(1, case["h"], case["d"], case["bs"], case["tokens"] + 64, TYPES[case["dtype"]], quant="int8" if case.get("int8") else None)[0]
    st["host"].zero_()  # touched once, as a pool that has served a session
    return st


def run(st: dict):
    case, kind = st["case"], st["kind"]
    if kind == "select":
        got = st["view"].select(0, st["q"])
        return [got.out, got.lse]
    if kind == "step":
        st["graph"].replay()
        return [st["out"], st["lse"]]
    if kind in ("host", "hybrid", "exact"):
        return [st["layer"].decode(q, None, ws=st["ws"]) for q in st["q"]]
    if kind == "dense":
        return [attend(st["q"], *st["kv"], None)]
    if kind == "rank":
        return [top_blocks(st["q"], *st["meta"], case["k"], dtype=torch.float32)]
    if kind == "int8":
        records = pack(st["pairs"])
        flat = records.view(-1, records.shape[-1])
        return [records, unpack(flat, case["bs"], case["d"], st["pairs"].dtype)]
    if kind == "turn":
        k, v, _ = st["layer"].dense_kv(*st["new"], st["scratch"])
        return [k, v]
    layer = TieredLayer(*st["kv"], case["k"], case["bs"], case["tokens"] + 64, host=st["host"], quant="int8" if case.get("int8") else None, fetch="zerocopy")
    return [layer.host, layer.kmin, layer.kmax, layer.pool]


# -- the work, the tolerance, the exact values --------------------------------------------------------


def work(case: dict) -> dict:
    h, g, d, bs, t, k, L = (case[x] for x in ("h", "g", "d", "bs", "tokens", "k", "layers"))
    es = 4 if case["dtype"] == "f32" else 2
    n, fill = _extent(case)
    pair = 2 * bs * d * es
    record = 2 * bs * d + 4 * d + 4 * bs
    stored = record if case.get("int8") else pair
    ends = h * (pair + 2 * fill * d * es)  # the sink and the current block
    io = 2 * h * g * d * es + 4 * h * g
    meta = 2 * h * (n - 1) * d * es
    score = 4 * h * g * d * (n - 1)
    kind = case["kind"]
    if kind in ("select", "step", "host", "hybrid"):
        steps = HYBRID_STEPS if kind == "hybrid" else L
        return {"bytes": steps * (meta + h * k * stored + ends + io), "flops": steps * (score + 4 * h * g * d * ((k + 1) * bs + fill))}
    if kind == "exact":
        return {"bytes": meta + h * k * pair + h * (n - 1 - k) * stored + ends + io, "flops": score + 4 * h * g * d * t}
    if kind == "dense":
        return {"bytes": 2 * h * t * d * es + io, "flops": 4 * h * g * d * t}
    if kind == "rank":
        c = t // bs
        return {"bytes": 2 * h * c * d * es + 8 * h * k, "flops": 4 * h * g * d * c}
    if kind == "int8":
        m = h * (t // bs)
        return {"bytes": m * 2 * (pair + record), "flops": m * 2 * bs * d * 6}
    if kind == "turn":
        return {"bytes": 2 * 2 * h * (t + case["turn"]) * d * es, "flops": 0}
    return {"bytes": 2 * h * t * d * es + h * (t // bs) * stored + 2 * h * (t // bs) * d * es, "flops": h * (t // bs) * 2 * bs * d * 6}


def tolerance(case: dict):
    if case["kind"] in ("int8", "turn", "build"):
        return "exact"
    if case["kind"] == "rank":
        return {"rel": 1e-5, "differ": 0.01}  # two bounds equal to float32's last places may change places
    # Outputs in the model's 16 bits: another order of the float32 sums flips a last place here and there.
    return {"rel": 2e-3 if case["dtype"] == "bf16" else 4e-4, "max": 0.05 if case["dtype"] == "bf16" else 0.01}


def _through_int8(x: torch.Tensor, axis: int) -> torch.Tensor:
    """x through 8-bit codes over `axis` with a float16 scale and zero: what a record holds, widened."""
    f = x.float()
    lo, hi = f.amin(axis, keepdim=True), f.amax(axis, keepdim=True)
    scale = ((hi - lo) / 255.0).clamp_min(torch.finfo(torch.float32).tiny)
    codes = torch.round((f - lo) / scale).clamp(0.0, 255.0)
    return (codes * scale.half().float() + lo.half().float()).to(x.dtype)


def _bound(q: torch.Tensor, kmin: torch.Tensor, kmax: torch.Tensor, g: int) -> torch.Tensor:
    """Quest's bound [h, n] in 64 bits of q [n_q, d] over kmin / kmax [h, n, d]."""
    q = q.double()
    rows = []
    for j in range(kmin.shape[0]):
        qh = q[j * g : (j + 1) * g]
        up, down = qh.clamp_min(0.0), qh.clamp_max(0.0)
        rows.append((kmax[j].double() @ up.T.contiguous() + kmin[j].double() @ down.T.contiguous()).amax(1))
    return torch.stack(rows)


def _attend(q: torch.Tensor, keys: list, values: list, g: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Attention in 64 bits of q [n_q, d] over each KV head's keys and values [t, d]."""
    outs, lses = [], []
    for j, (k, v) in enumerate(zip(keys, values)):
        s = (q[j * g : (j + 1) * g].double() @ k.double().T.contiguous()) * q.shape[-1] ** -0.5
        lses.append(torch.logsumexp(s, 1))
        outs.append(torch.softmax(s, 1) @ v.double())
    return torch.cat(outs), torch.cat(lses)


def _exact_step(case: dict, seed: int, layer: int, queries: list) -> list:
    h, g, d, bs, k = (case[x] for x in ("h", "g", "d", "bs", "k"))
    n, fill = _extent(case)
    keys, values = (x[0] for x in _kv(case, seed, layer))
    blocks = [x[:, : n * bs].reshape(h, n, bs, d) for x in (keys, values)]
    stored = [_through_int8(blocks[0], 2), _through_int8(blocks[1], 3)] if case.get("int8") else blocks
    exact = case["kind"] == "exact"
    ranked = blocks[0] if exact else stored[0]  # the exact tier ranks and reads what its HBM store holds
    kmin, kmax = ranked.amin(2), ranked.amax(2)
    got = []
    for q in queries:
        ids = _bound(q, kmin[:, 1:], kmax[:, 1:], g).topk(k, dim=1).indices + 1
        ks, vs = [], []
        for j in range(h):
            parts = []
            for whole, kept, end in ((blocks[0], stored[0], keys), (blocks[1], stored[1], values)):
                mine = [whole[j, 0], (whole if exact else kept)[j, ids[j]].reshape(-1, d), end[j, n * bs : n * bs + fill]]
                if exact:
                    rest = torch.ones(n, dtype=torch.bool, device=DEV)
                    rest[0] = False
                    rest[ids[j]] = False
                    mine.append(kept[j, rest].reshape(-1, d))
                parts.append(torch.cat(mine))
            ks.append(parts[0])
            vs.append(parts[1])
        got.append(_attend(q, ks, vs, g))
    return got


def exact(case: dict, seed: int):
    kind, n_q, d = case["kind"], case["h"] * case["g"], case["d"]
    if kind == "select":
        out, lse = _exact_step(case, seed, 0, [_query(case, seed)])[0]
        return [out.view(1, n_q, 1, d), lse.view(1, n_q)]
    if kind == "step":
        got = [_exact_step(case, seed, layer, [_query(case, seed, layer)])[0] for layer in range(case["layers"])]
        return [torch.stack([o for o, _ in got]), torch.stack([s for _, s in got])]
    if kind == "hybrid":
        return _exact_step(case, seed, 0, _queries(case, seed))
    if kind in ("host", "exact"):
        return _exact_step(case, seed, 0, [_query(case, seed)])
    if kind == "dense":
        keys, values = (x[0] for x in _kv(case, seed))
        return [_attend(_query(case, seed), list(keys), list(values), case["g"])[0].view(1, n_q, 1, d)]
    if kind == "rank":
        kmin, kmax = _rank_metadata(case, seed)
        return [_bound(_query(case, seed), kmin[0], kmax[0], case["g"]).topk(case["k"], dim=1).indices.unsqueeze(0)]
    return None  # bytes and copies: the same to the bit
