"""The tier's decode path on the GPU: TieredLayer / TieredCache counterparts of lazykv/tiered.py.

What a selecting layer does per decode step, with no host synchronisation anywhere:

1. `append` writes the token into the current block's slot; a full block is sealed first by one
   kernel that stores it into the host pool (as model-dtype bytes or as an int8 record) and
   writes its key min/max metadata (lazykv/tiered.py:306-314,353-375).
2. `rank` scores every candidate block (1 .. n_sealed-1) with the Quest bound and selects the top
   K per KV head on the device (lazykv/tiered.py:383-387, without the `.cpu()`).
3. `decode` attends sink + selected + current[:fill] in one block-sparse kernel that reads each
   selected pair where it lives: in place from the mapped host pool over PCIe (`fetch="zerocopy"`,
   lazykv/tiered.py:489-511), from an HBM store (`fetch="resident"`, all blocks on the GPU as
   in rung 5, lazykv/selection.py:147-183), or from HBM slots holding the k most recently selected
   blocks per head, the misses read in place and admitted as they are attended (`fetch="hybrid"`,
   the device-side form of rung 6's admit/gather, lazykv/tiered.py:389-487; bit-identical to the
   zero-copy result). With `exact=True` the same kernel also attends every
   other sealed block from the host tier and merges the two partials by log-sum-exp
   (lazykv/exact.py:225-264), so the result is full attention.

Layouts follow the reference: GPU slot pool [2, h, 2, bs, d] holding the sink (slot 0) and the
current block (slot 1) (`n_slots=0`, lazykv/tiered.py:250,261); host pool [cap, h, 2, bs, d] in
the model dtype or [cap, h, P] int8 records (:265); metadata [1, h, cap, d] in the model dtype
(:262), taken over the dequantised keys for an int8 tier (:182-194). Rung 7's speculative
prefetch and the host-side residency tables of rung 6 are not part of this path.
"""

from __future__ import annotations

from dataclasses import dataclass, field
from typing import Any

import numpy as np
import torch

from transformers.cache_utils import Cache

from lazykv_amd import _lib, kernels
from lazykv_amd.cache import CacheStats, Decoded, FullGPUCache  # Decoded: what select returns
from lazykv_amd.pinned import pinned_empty
from lazykv_amd.quant import packed_pair_bytes
from lazykv_amd.selection import QUEST_DENSE_LAYERS

FETCH_MODES = ("zerocopy", "resident", "hybrid")  # how a tier reads its selected pairs, in this library's terms
RUNG6_FETCHES = ("runs", "gather")  # the reference's host-driven fetches into HBM slots (lazykv/tiered.py:420-487)
FETCH_NAMES = FETCH_MODES + RUNG6_FETCHES
MAX_SLOTS = 4096  # HBM slots per KV head of a hybrid tier (the residency launch's limit)


def device_fetch(fetch: str) -> str:
    """The read a fetch name stands for. "zerocopy", "resident" and "hybrid" are this library's own.
    The reference's rung-6 names, "runs" and "gather", copy each step's missed pairs into n_slots HBM
    slots per head from the host, one transfer per run of pairs or one staged gather
    (lazykv/tiered.py:420-487). Both name the device-side hybrid here: the same slots and the same
    least-recently-used victims, but the residency tables live on the device and a miss is read in
    place over the link and written into its slot by the decode itself, so nothing is staged and
    nothing returns to the host."""
    if fetch in RUNG6_FETCHES:
        return "hybrid"
    if fetch in FETCH_MODES:
        return fetch
    raise ValueError(f"unknown fetch mode {fetch!r}; expected one of {FETCH_NAMES}")


@dataclass
class TierCounters:
    """Work counters of the tier, with the reference's field names (lazykv/tiered.py:76-109).

    Counted here: selections, selected pairs, zero-copy bytes, seals, the boundary and multi-token
    ingestion, and the remainder pairs of the exact tier. The reference's host-time fields
    (host_*_s) time host work this path does not do -- ranking, residency bookkeeping and copy
    launches are device work with no host sync -- and stay 0. So do its residency outcomes
    (hit_pairs, fetched_pairs, fetch_*, thrash_pairs) and its prefetch fields: a hybrid tier decides
    hits and misses on the device, and counting them on the host would need the sync the path
    removes; `TieredLayer.resident_pairs` reads the tables when a caller wants them.
    """

    host_select_s: float = 0.0
    host_rank_s: float = 0.0
    host_fetch_s: float = 0.0
    host_prefetch_s: float = 0.0
    host_seal_s: float = 0.0
    boundary_d2h_s: float = 0.0
    boundary_d2h_bytes: int = 0
    selections: int = 0
    selected_pairs: int = 0
    hit_pairs: int = 0
    fetched_pairs: int = 0
    fetch_transfers: int = 0
    fetch_bytes: int = 0
    thrash_pairs: int = 0
    prefetched_pairs: int = 0
    prefetch_transfers: int = 0
    prefetch_bytes: int = 0
    prefetch_used_pairs: int = 0
    seals: int = 0
    seal_bytes: int = 0
    # Dense ingestion of multi-token forwards (lazykv/tiered.py:101-104,649-663).
    ingest_forwards: int = 0
    ingest_tokens: int = 0
    ingest_h2d_bytes: int = 0
    host_ingest_s: float = 0.0
    zerocopy_bytes: int = 0
    # The exact tier: sealed pairs attended as the remainder, summed over selections.
    remainder_pairs: int = 0
    fetched_pairs_per_step: list[int] = field(default_factory=list)


def _renumbered(src: kernels.Source, first: int, elem_bytes: int) -> kernels.Source:
    """`src` with its block 0 addressed as block `first`: a store of blocks [first, first + n)
    then reads the source's blocks [0, n). The base addresses move back by `first` blocks; the
    kernel only addresses blocks from `first` on, which lie inside the source."""
    back = first * src.block_stride * (1 if src.dtype == _lib.INT8_RECORD else elem_bytes)
    return kernels.Source(src.k - back, src.v - back if src.v else 0, src.block_stride, src.head_stride, src.dtype, src.deq_dtype,
                          first + src.n_blocks, src.owners, src.flags)


class DenseScratch:
    """One HBM buffer pair [1, h, T, d] that a multi-token forward's dense keys and values are
    assembled in (`TieredLayer.dense_kv`). A cache's selecting layers run one after another on one
    stream, so they share it; it grows to the longest forward seen and is never shrunk."""

    def __init__(self) -> None:
        self.k: torch.Tensor | None = None
        self.v: torch.Tensor | None = None

    def take(self, h: int, tokens: int, d: int, dtype: torch.dtype, device: torch.device) -> tuple[torch.Tensor, torch.Tensor]:
        k = self.k
        if k is None or k.shape[1] != h or k.shape[2] < tokens or k.shape[3] != d or k.dtype != dtype or k.device != device:
            # Whole blocks of 256 tokens, so a turn that grows the context by a few tokens reuses it.
            cap = -(-tokens // 256) * 256
            self.k = torch.empty((1, h, cap, d), dtype=dtype, device=device)
            self.v = torch.empty_like(self.k)
        assert self.k is not None and self.v is not None
        return self.k, self.v


def allocate_host_pools(n_layers: int, heads: int, head_dim: int, block_size: int, capacity_tokens: int, dtype: torch.dtype = torch.bfloat16, quant: str | None = None, coherent: bool = False) -> list[torch.Tensor]:
    """Mapped pinned host pools, one per selecting layer (lazykv/tiered.py:874-882)."""
    blocks = -(-capacity_tokens // block_size)
    if quant is None:
        shape, dt = (blocks, heads, 2, block_size, head_dim), dtype
    elif quant == "int8":
        shape, dt = (blocks, heads, packed_pair_bytes(block_size, head_dim)), torch.uint8
    else:
        raise ValueError(f"unknown tier precision {quant!r}")
    return [pinned_empty(shape, dt, coherent=coherent) for _ in range(n_layers)]


class TieredLayer:
    """One selecting layer: slot pool (sink + current), host pool, optional HBM store, metadata."""

    def __init__(
        self,
        keys: torch.Tensor,
        values: torch.Tensor,
        k_blocks: int,
        block_size: int,
        capacity_tokens: int,
        host: torch.Tensor | None = None,
        n_slots: int | None = None,
        quant: str | None = None,
        fetch: str = "zerocopy",
        exact: bool = False,
        rank_dtype: torch.dtype | None = torch.float32,
    ) -> None:
        """Build the tier from a prompt's KV [1, h, L, d] on the GPU (lazykv/tiered.py:153-206).

        Every full block is stored to the host pool once and its metadata written, by one kernel;
        the tail goes to the current slot.
        """
        _lib.require_cuda(keys, values)
        _, h, length, d = keys.shape
        n_blocks = length // block_size
        self._allocate(h, d, n_blocks, k_blocks, block_size, capacity_tokens, keys.device, keys.dtype, host, n_slots, quant, fetch, exact, rank_dtype)
        self._open_prompt()
        self.seal_prompt_blocks(keys, values, 0, n_blocks)
        self.close_prompt(keys, values)

    @classmethod
    def opened(
        cls,
        h: int,
        d: int,
        prompt_tokens: int,
        k_blocks: int,
        block_size: int,
        capacity_tokens: int,
        device: torch.device,
        dtype: torch.dtype,
        host: torch.Tensor | None = None,
        n_slots: int | None = None,
        quant: str | None = None,
        fetch: str = "zerocopy",
        exact: bool = False,
        rank_dtype: torch.dtype | None = torch.float32,
    ) -> TieredLayer:
        """A layer for a prompt of `prompt_tokens` tokens whose KV arrives in pieces: the caller seals
        the prompt's full blocks as they become available (`seal_prompt_blocks`, in any grouping) and
        then `close_prompt` sets the sink and the current block. The result is the constructor's."""
        self = cls.__new__(cls)
        self._allocate(h, d, prompt_tokens // block_size, k_blocks, block_size, capacity_tokens, torch.device(device), dtype, host, n_slots, quant, fetch, exact, rank_dtype)
        self._open_prompt()
        return self

    def _open_prompt(self) -> None:
        self.n_sealed, self.fill, self.length = 0, 0, 0
        self.boundary_d2h_bytes = 0
        self._prompt_sealed = 0  # prompt blocks [0, _prompt_sealed) are in the tier

    def seal_prompt_blocks(self, keys: torch.Tensor, values: torch.Tensor, first: int, n: int) -> None:
        """Store prompt blocks [first, first + n) of the dense KV [1, h, >= (first + n) * bs, d] into
        the tier (host pool and/or HBM store) with their metadata: one kernel launch. Blocks must
        arrive in order; the launch goes to the current stream."""
        if first != self._prompt_sealed:
            raise ValueError(f"prompt blocks must be sealed in order: expected block {self._prompt_sealed}, got {first}")
        if n <= 0:
            return
        src = kernels.dense_source(keys, values, self.bs)
        if first + n > src.n_blocks:
            raise ValueError(f"blocks {first}..{first + n} are not all in the given KV ({src.n_blocks} full blocks)")
        self._store(src, first, n, with_store=True)
        self._prompt_sealed = first + n
        if self.host is not None:
            self.boundary_d2h_bytes += n * self.h * self.pair_bytes

    def close_prompt(self, keys: torch.Tensor, values: torch.Tensor) -> None:
        """Finish a prompt of L = keys.shape[2] tokens whose full blocks are sealed: the sink slot
        takes block 0 and the current slot the L % bs tokens past the last full block."""
        length = keys.shape[2]
        n_blocks, tail = divmod(length, self.bs)
        if self._prompt_sealed != n_blocks:
            raise ValueError(f"{self._prompt_sealed} of the prompt's {n_blocks} full blocks are sealed")
        # The sink never leaves VRAM and stays exact even under an int8 tier (lazykv/tiered.py:200-202).
        ends = [(self.pool[0, :, 0], keys[0, :, : self.bs]), (self.pool[0, :, 1], values[0, :, : self.bs])]
        if tail:
            ends += [(self.pool[1, :, 0, :tail], keys[0, :, n_blocks * self.bs : length]), (self.pool[1, :, 1, :tail], values[0, :, n_blocks * self.bs : length])]
        kernels.copy_rows(ends)
        self.n_sealed, self.fill, self.length = n_blocks, tail, length
        self._seed_slots()

    def _seed_slots(self) -> None:
        """A hybrid tier's residency at the end of the prompt (lazykv/tiered.py:165-168,274-287): the
        min(n_slots, n_sealed - 1) most recent sealed blocks in slots 0, 1, ..., read back from the tier
        as a decode reads them (an int8 record dequantised), so a later hit attends exactly what a miss
        would; the other slots stay empty and come first in the use order. One store launch and a few
        table fills, all on the current stream."""
        if self.res is None:
            return
        seed = min(self.n_slots, self.n_sealed - 1)
        if seed <= 0:
            return
        first = self.n_sealed - seed
        slots = kernels.pool_source(self.res.slots)
        # Block `first + j` of the tier lands in slot j: the slot pool addressed from block `first` on.
        dst = _renumbered(slots, first, self.res.slots.element_size())
        kernels.store_blocks(self._host_src, dst=dst, n_kv=self.h, head_dim=self.d, block_size=self.bs, first_block=first, n_blocks=seed)
        self.res.seed(first, seed)

    @classmethod
    def from_state(
        cls,
        h: int,
        d: int,
        k_blocks: int,
        block_size: int,
        capacity_tokens: int,
        device: torch.device,
        dtype: torch.dtype,
        host: torch.Tensor | None = None,
        quant: str | None = None,
        fetch: str = "zerocopy",
        exact: bool = False,
        rank_dtype: torch.dtype | None = torch.float32,
    ) -> TieredLayer:
        """An empty layer whose pools the caller fills (`load_blocks`, `set_current`), e.g. a restore."""
        self = cls.__new__(cls)
        self._allocate(h, d, capacity_tokens // block_size, k_blocks, block_size, capacity_tokens, device, dtype, host, None, quant, fetch, exact, rank_dtype, check_budget=False)
        self.n_sealed, self.fill, self.length = 0, 0, 0
        self.boundary_d2h_bytes = 0
        return self

    @classmethod
    def from_store(
        cls,
        host: torch.Tensor,
        n_sealed: int,
        tail: torch.Tensor,
        k_blocks: int,
        block_size: int,
        capacity_tokens: int,
        device: torch.device,
        n_slots: int | None = None,
        fetch: str = "zerocopy",
        exact: bool = False,
        rank_dtype: torch.dtype | None = torch.float32,
    ) -> TieredLayer:
        """A layer over a host pool whose first `n_sealed` blocks already hold the sealed KV
        (lazykv/tiered.py:226-236): a snapshot restore reads them straight into the pool.

        The metadata is rebuilt on the GPU by reading the pool in place (and, for the exact tier,
        copying it into the HBM store in the same pass); the sink slot is block 0 of the pool and the
        current slot is `tail` [h, 2, fill, d]. Nothing is written back to the host.
        """
        _, h, two, bs, d = host.shape
        if two != 2 or bs != block_size:
            raise ValueError(f"host pool {tuple(host.shape)} is not [blocks, h, 2, {block_size}, d]")
        fill = tail.shape[2]
        if tuple(tail.shape) != (h, 2, fill, d) or not 0 <= fill <= bs:
            raise ValueError(f"tail must be [{h}, 2, fill <= {bs}, {d}], got {tuple(tail.shape)}")
        self = cls.__new__(cls)
        self._allocate(h, d, n_sealed, k_blocks, bs, capacity_tokens, torch.device(device), host.dtype, host, n_slots, None, fetch, exact, rank_dtype)
        if n_sealed > 0:
            src = kernels.pool_source(host)  # read in place over PCIe
            kernels.store_blocks(src, dst=self._store_src, n_kv=h, head_dim=d, block_size=bs, first_block=0, n_blocks=n_sealed, kmin=self.kmin, kmax=self.kmax)
            self.pool[0].copy_(host[0])
        if fill:
            self.pool[1, :, :, :fill].copy_(tail)
        self.n_sealed, self.fill, self.length = n_sealed, fill, n_sealed * bs + fill
        self.boundary_d2h_bytes = 0
        self._seed_slots()
        return self

    def _allocate(self, h, d, n_blocks, k_blocks, bs, capacity_tokens, dev, dt, host, n_slots, quant, fetch, exact, rank_dtype, check_budget=True) -> None:  # noqa: ANN001
        if check_budget and n_blocks - 1 <= k_blocks:
            raise ValueError(f"budget of {k_blocks} blocks covers all {n_blocks - 1} candidate blocks; the tier needs selection")
        mode = device_fetch(fetch)
        if quant not in (None, "int8"):
            raise ValueError(f"unknown tier precision {quant!r}")
        if mode == "hybrid":
            # The reference's rule for n_slots (lazykv/tiered.py:249-252): K by default, never fewer.
            n_slots = k_blocks if n_slots is None else n_slots
            if n_slots < k_blocks:
                raise ValueError(f"{n_slots} slots cannot hold a selection of {k_blocks} blocks")
            if n_slots > MAX_SLOTS:
                raise ValueError(f"{n_slots} slots per head exceed the hybrid tier's limit of {MAX_SLOTS}")
        elif mode == "resident" and n_slots not in (None, 0):
            raise ValueError("the resident tier keeps every block in its HBM store and no slots (n_slots=0)")
        else:
            n_slots = 0  # zero-copy: VRAM holds the sink and the current block (lazykv/tiered.py:573-578)
        if exact and mode == "zerocopy":
            raise ValueError("the exact tier attends its selected blocks from HBM: fetch 'resident', or a slotted fetch ('runs', 'gather', 'hybrid')")
        if dt not in (torch.float16, torch.bfloat16):
            raise ValueError(f"KV dtype {dt} unsupported: float16 or bfloat16")
        self.h, self.d, self.bs, self.k = h, d, bs, k_blocks
        self.n_slots, self.tail_slot = n_slots, 1
        self.quant, self.fetch, self.exact = quant, mode, exact
        self.fetch_name = fetch
        self.rank_mode = _lib.RANK_F32 if rank_dtype == torch.float32 else _lib.RANK_MODEL
        self.dtype = dt
        self.cap_blocks = -(-capacity_tokens // bs)
        # Zeroed: the current block's unfilled rows are masked (lazykv/tiered.py:259-261).
        self.pool = torch.zeros((2, h, 2, bs, d), dtype=dt, device=dev)
        self.kmin = torch.zeros((1, h, self.cap_blocks, d), dtype=dt, device=dev)
        self.kmax = torch.zeros_like(self.kmin)
        self.logical_pair_bytes = 2 * bs * d * self.pool.element_size()
        need_host = mode in ("zerocopy", "hybrid") or exact
        shape = (self.cap_blocks, h, 2, bs, d) if quant is None else (self.cap_blocks, h, packed_pair_bytes(bs, d))
        want = dt if quant is None else torch.uint8
        if host is None and need_host:
            host = pinned_empty(shape, want)
        elif host is not None and (tuple(host.shape) != shape or host.dtype != want):
            raise ValueError(f"host pool must be pinned {want} with shape {shape}, got {host.dtype} {tuple(host.shape)}")
        self.host = host
        self.pair_bytes = self.logical_pair_bytes if quant is None else packed_pair_bytes(bs, d)
        self.store = torch.zeros((self.cap_blocks, h, 2, bs, d), dtype=dt, device=dev) if mode == "resident" else None
        self._host_src = None
        if host is not None:
            self._host_src = kernels.pool_source(host) if quant is None else kernels.record_source(host, dt)
        self._store_src = kernels.pool_source(self.store) if self.store is not None else None
        # Hybrid: n_slots HBM slots per head holding the most recently selected blocks, seeded with the
        # most recent prompt blocks when the prompt closes.
        self.res = kernels.Residency.allocate(k_blocks, h, self.cap_blocks, bs, d, dt, dev, n_slots=n_slots) if mode == "hybrid" else None
        self._pool_src = kernels.pool_source(self.pool)

    # -- writes ---------------------------------------------------------------------------------

    def _store(self, src: kernels.Source, first: int, n: int, with_store: bool) -> None:
        """Store blocks [first, first+n) from `src` into the host pool / HBM store, with metadata."""
        if n <= 0:
            return
        if first + n > self.cap_blocks:
            raise RuntimeError(f"host pool full: {self.cap_blocks} blocks")
        common = dict(n_kv=self.h, head_dim=self.d, block_size=self.bs)
        # The metadata comes from the bytes a read will produce: the dequantised keys for an int8
        # host tier, unless the selected blocks are read from the exact HBM store.
        meta_from_host = self._host_src is not None and not (self.store is not None)
        if self._host_src is not None:
            kernels.store_blocks(src, dst=self._host_src, first_block=first, n_blocks=n,
                                 kmin=self.kmin if meta_from_host else None, kmax=self.kmax if meta_from_host else None, **common)
        if self.store is not None and with_store:
            kernels.store_blocks(src, dst=self._store_src, first_block=first, n_blocks=n, kmin=self.kmin, kmax=self.kmax, **common)

    def load_blocks(self, pairs: torch.Tensor, first: int) -> None:
        """Store `pairs` [n, h, 2, bs, d] (GPU, model dtype) as blocks first..first+n-1 (boundary / restore)."""
        x = pairs.contiguous()
        self._store(_renumbered(kernels.pool_source(x), first, x.element_size()), first, pairs.shape[0], with_store=True)
        self.n_sealed = max(self.n_sealed, first + pairs.shape[0])

    def set_current(self, keys: torch.Tensor, values: torch.Tensor, fill: int) -> None:
        """Sink and current block: keys/values [h, 2, bs, d] slices are written by the caller via `pool`."""
        self.fill = fill
        self.length = self.n_sealed * self.bs + fill

    def append(self, key: torch.Tensor, value: torch.Tensor, counters: TierCounters | None = None) -> None:
        """Write one decode token; seal the current block first if it is full (lazykv/tiered.py:306-314)."""
        if self.fill == self.bs:
            self._seal(counters)
        self.pool[1, :, 0, self.fill].copy_(key[0, :, 0])
        self.pool[1, :, 1, self.fill].copy_(value[0, :, 0])
        self.fill += 1
        self.length += 1

    def extend(self, keys: torch.Tensor, values: torch.Tensor, counters: TierCounters | None = None) -> None:
        """Write a multi-token forward's KV [1, h, T, d], leaving exactly the state T calls to
        `append` would (lazykv/tiered.py:316-332): sealing stays lazy, so a block the forward
        fills completely stays the current block until a later token arrives.

        Instead of a seal per block, at most two store launches: the current block, once it is full
        and more tokens follow, from its slot; then every further block the forward completes
        except the last, straight from `keys`/`values`. The last one goes to the current slot. The
        records and metadata are per-block functions of the same bytes, so they equal the seals'.
        """
        _lib.require_cuda(keys, values)
        t = keys.shape[2]
        if keys.shape != values.shape or keys.shape[0] != 1 or keys.shape[1] != self.h or keys.shape[3] != self.d:
            raise ValueError(f"extend takes KV [1, {self.h}, T, {self.d}], got {tuple(keys.shape)} / {tuple(values.shape)}")
        if t == 0:
            return
        if self.length + t > self.cap_blocks * self.bs:
            raise RuntimeError(f"host pool full: {self.length} + {t} tokens exceed {self.cap_blocks} blocks of {self.bs}")
        k = keys.contiguous()
        v = values.contiguous()
        top = min(self.bs - self.fill, t)  # tokens that complete the current block
        self._write_current(k, v, 0, top)
        rest = t - top
        if rest == 0:
            return
        self._seal(counters)
        spans = -(-rest // self.bs)  # blocks the remaining tokens cover; the last stays current
        direct = spans - 1
        if direct:
            first = self.n_sealed
            src = kernels.dense_source(k[:, :, top:], v[:, :, top:], self.bs)
            self._store(_renumbered(src, first, k.element_size()), first, direct, with_store=True)
            self.n_sealed += direct
            self.length += direct * self.bs
            if counters is not None:
                counters.seals += direct
                counters.seal_bytes += direct * self.h * self.pair_bytes
        self.fill = 0
        self._write_current(k, v, top + direct * self.bs, t)

    def _write_current(self, k: torch.Tensor, v: torch.Tensor, a: int, b: int) -> None:
        """Tokens [a, b) of a forward's KV [1, h, T, d] appended to the current block's slot."""
        n = b - a
        if n <= 0:
            return
        self.pool[1, :, 0, self.fill : self.fill + n].copy_(k[0, :, a:b])
        self.pool[1, :, 1, self.fill : self.fill + n].copy_(v[0, :, a:b])
        self.fill += n
        self.length += n

    def dense_kv(self, keys: torch.Tensor, values: torch.Tensor, scratch: DenseScratch) -> tuple[torch.Tensor, torch.Tensor, int]:
        """What a multi-token forward attends to (lazykv/tiered.py:334-351): this layer's whole KV --
        the sealed blocks, the current block's `fill` tokens -- followed by `keys`/`values`
        [1, h, T, d], as views [1, h, L + T, d] of `scratch`. Returns (keys, values, bytes read over
        the link).

        The sealed blocks are read by one store-kernel launch: in place from the host pool over the
        link (the model-dtype pairs copied, or int8 records dequantised as the decode reads them,
        which the reference refuses), or from the HBM store for the resident and exact tiers. Block 0
        comes from the sink slot, which is what the decode attends (exact even under an int8 tier).
        """
        _lib.require_cuda(keys, values)
        t = keys.shape[2]
        bs, n = self.bs, self.n_sealed
        total = n * bs + self.fill + t
        sk, sv = scratch.take(self.h, total, self.d, self.dtype, self.pool.device)
        moved = 0
        if n:
            src = self._store_src if self.store is not None else self._host_src
            dst = kernels.dense_source(sk, sv, bs)
            kernels.store_blocks(src, dst=dst, n_kv=self.h, head_dim=self.d, block_size=bs, first_block=0, n_blocks=n)
            if self.store is None:
                moved = n * self.h * self.pair_bytes
        # The sink over block 0, the current block and the new tokens: one launch.
        a = n * bs
        parts = []
        if n:
            parts += [(sk[0, :, :bs], self.pool[0, :, 0]), (sv[0, :, :bs], self.pool[0, :, 1])]
        if self.fill:
            parts += [(sk[0, :, a : a + self.fill], self.pool[1, :, 0, : self.fill]), (sv[0, :, a : a + self.fill], self.pool[1, :, 1, : self.fill])]
        kernels.copy_rows(parts + [(sk[0, :, a + self.fill : total], keys[0]), (sv[0, :, a + self.fill : total], values[0])])
        return sk[:, :, :total], sv[:, :, :total], moved

    def _seal(self, counters: TierCounters | None) -> None:
        """Store the full current block as block n_sealed (lazykv/tiered.py:353-375), on the device."""
        b = self.n_sealed
        if b >= self.cap_blocks:
            raise RuntimeError(f"host pool full: {self.cap_blocks} blocks")
        # Slot 1 of the pool, addressed as block b of a source whose block stride is zero.
        slot = self._pool_src
        src = kernels.Source(slot.k + self.h * 2 * self.bs * self.d * self.pool.element_size(), slot.v + self.h * 2 * self.bs * self.d * self.pool.element_size(),
                             0, slot.head_stride, slot.dtype, slot.deq_dtype, self.cap_blocks, slot.owners)
        self._store(src, b, 1, with_store=True)
        self.n_sealed += 1
        self.fill = 0
        if counters is not None:
            counters.seals += 1
            counters.seal_bytes += self.h * self.pair_bytes

    # -- decode ---------------------------------------------------------------------------------

    def candidates(self) -> tuple[int, int]:
        """(n_full, fill): blocks 1..n_full-1 are selectable, block n_full is current (:379-381)."""
        return self.n_sealed, self.fill

    def rank(self, query: torch.Tensor, out: torch.Tensor | None = None, ws: kernels.Workspace | None = None) -> torch.Tensor:
        """Top-K block ids [h, K] (int32, ascending, on the device) for a query [1, n_q, 1, d]."""
        n_full, _ = self.candidates()
        if n_full - 1 < self.k:
            raise ValueError(f"budget of {self.k} blocks covers all {n_full - 1} candidate blocks")
        idx = kernels.bound_topk(query, self.kmin, self.kmax, self.k, cand_offset=1, n_cand=n_full - 1, rank_mode=self.rank_mode, out_idx=out, ws=ws)
        assert idx is not None
        return idx

    def rank_host(self, query: torch.Tensor) -> np.ndarray:
        """The reference's `rank` (:383-387): ids [h, K] in descending bound order, on the host (syncs)."""
        n_full, _ = self.candidates()
        idx = kernels.bound_topk(query, self.kmin, self.kmax, self.k, cand_offset=1, n_cand=n_full - 1, rank_mode=self.rank_mode, sorted_=True)
        return idx.to(torch.int64).cpu().numpy()

    def fused_select(self) -> bool:
        """Whether a decode without given ids makes the whole step one call: lkv_select_decode for
        zero-copy or resident reads, lkv_select_hybrid_decode for hybrid ones, whose residency launch
        chooses the ids before the decode launch, so an exact remainder can exclude them."""
        n_full, _ = self.candidates()
        return (not self.exact or self.res is not None) and self.k <= n_full - 1

    def decode(self, query: torch.Tensor, scaling: float | None, idx: torch.Tensor | None = None, out: torch.Tensor | None = None, lse: torch.Tensor | None = None, ws: kernels.Workspace | None = None) -> tuple[torch.Tensor, torch.Tensor]:
        """Attention of one decode token over this layer's attended set. Returns out [n_q, d], lse [n_q].

        Without `idx`, the selection is made here: in the same call as the attention where
        `fused_select` allows (lkv_select_decode), else by `rank` first."""
        n_full, fill = self.candidates()
        scale = scaling if scaling is not None else self.d**-0.5
        if idx is None and self.fused_select():
            qq = query.reshape(-1, self.d)
            if not qq.is_contiguous():
                qq = qq.contiguous()
            out = out if out is not None else torch.empty(qq.shape, dtype=qq.dtype, device=qq.device)
            lse = lse if lse is not None else torch.empty((qq.shape[0],), dtype=torch.float32, device=qq.device)
            if self.res is not None:
                rem, rem_range = (self._host_src, (1, n_full)) if self.exact else (None, (0, 0))
                return kernels.select_hybrid_decode(qq, self.kmin, self.kmax, self.k, cand_offset=1, n_cand=n_full - 1, block_size=self.bs, scale=scale,
                                                    host=self._host_src, res=self.res, sink=self._pool_src, sink_block=0, cur=self._pool_src,
                                                    cur_block=1 if fill > 0 else -1, fill=fill, rem=rem, rem_range=rem_range,
                                                    rank_mode=self.rank_mode, out=out, lse=lse, ws=ws)
            sel = self._store_src if self.fetch == "resident" else self._host_src
            return kernels.select_decode(qq, self.kmin, self.kmax, self.k, cand_offset=1, n_cand=n_full - 1, block_size=self.bs, scale=scale, sel=sel,
                                         sink=self._pool_src, sink_block=0, cur=self._pool_src, cur_block=1 if fill > 0 else -1, fill=fill,
                                         rank_mode=self.rank_mode, out=out, lse=lse, ws=ws)
        if idx is None:
            idx = self.rank(query, ws=ws)
        sel = self._store_src if self.fetch == "resident" else self._host_src
        rem = None
        rem_range = (0, 0)
        if self.exact:
            rem, rem_range = self._host_src, (1, n_full)
        if self.res is not None:
            return kernels.hybrid_decode(
                query.reshape(-1, self.d), n_kv=self.h, block_size=self.bs, scale=scale, host=self._host_src, res=self.res, idx=idx,
                sink=self._pool_src, sink_block=0, cur=self._pool_src, cur_block=1 if fill > 0 else -1, fill=fill, rem=rem, rem_range=rem_range,
                out=out, lse=lse, ws=ws,
            )
        return kernels.sparse_decode(
            query.reshape(-1, self.d), n_kv=self.h, block_size=self.bs, scale=scale, sel=sel, idx=idx,
            sink=self._pool_src, sink_block=0, cur=self._pool_src, cur_block=1 if fill > 0 else -1, fill=fill,
            rem=rem, rem_range=rem_range, out=out, lse=lse, ws=ws,
        )

    def gpu_bytes(self) -> int:
        store = self.store.numel() * self.store.element_size() if self.store is not None else 0
        slots = self.res.slots.numel() * self.res.slots.element_size() if self.res is not None else 0
        return self.pool.numel() * self.pool.element_size() + store + slots

    def metadata_bytes(self) -> int:
        return 2 * self.kmin.numel() * self.kmin.element_size()

    def _not_resident_blocks(self) -> int:
        """Sealed blocks no GPU copy holds, summed over heads: all but the sink (pool slot 0) for a
        zero-copy tier, none for an HBM store, and those outside the slots for the hybrid tier
        (read from its table: a host sync, for reporting only)."""
        if self.store is not None:
            return 0
        held = int((self.res.slot_block >= 0).sum().item()) if self.res is not None else 0
        return max(0, self.h * max(0, self.n_sealed - 1) - held)

    def not_resident_bytes(self) -> int:
        """Host bytes of blocks VRAM does not hold, in the tier's storage format (lazykv/tiered.py:845-847)."""
        return self._not_resident_blocks() * self.pair_bytes

    def not_resident_logical_bytes(self) -> int:
        """The same blocks in the model dtype (lazykv/tiered.py:850-857)."""
        return self._not_resident_blocks() * self.logical_pair_bytes

    def host_bytes(self) -> int:
        return self.n_sealed * self.h * self.pair_bytes if self.host is not None else 0


class TieredCache(Cache):
    """Decode-time cache: dense layers share the prefilled FullGPUCache, selecting layers are
    tiered (lazykv/tiered.py:538-747).

    `full` is the exactly prefilled cache (a FullGPUCache, or a list of per-layer (keys, values)
    [1, h, L, d] on the GPU, which is copied into one). Its first `dense_layers` layers stay in it
    and keep growing during decode; every other layer becomes a TieredLayer, unless `tiers` brings
    them prebuilt (the layer-major prefill, which never holds them in `full`). `select` returns a
    `Decoded` (the finished attention of the step), or None to attend densely.

    The arguments are the reference's, in its order, and mean what they mean there, with these
    differences of effect:

    - `fetch`: "zerocopy" reads the selected pairs in place from the host pool. The reference's
      rung-6 fetches "runs" (its default) and "gather" keep `n_slots` HBM slots per head (K by
      default, more for spare slots) with least-recently-used victims, as the device-side hybrid
      ("hybrid"): its misses are read in place and written into their slots by the decode. As in
      the reference, an int8 tier takes "gather" rather than "runs" (and, as this library's
      departure, also "zerocopy", "resident" or "hybrid"). "resident" keeps every block in an HBM
      store.
    - `thrash_window` and `instrument` shape the reference's host-side counters and event timing
      of rung 6/7 copies. Residency is decided on the device here, without a host sync, so there
      is nothing for them to count or time; they are accepted and kept as attributes.
    - `stages` are rung 6's staging buffers for "gather". Nothing is staged here (a miss is read in
      place), so they are accepted and unused.
    - `prefetch`, `record_selection` and `replay_selection` (rung 7 and the Phase 6 ablation) are
      outside this path and refused, as the reference refuses them for the zero-copy fetch.
    - `exact` and `rank_dtype` are this library's own keywords: the exact split (ExactTieredCache)
      and the precision the bound is ranked in.
    """

    def __init__(
        self,
        full: FullGPUCache | list[tuple[torch.Tensor, torch.Tensor]],
        k_blocks: int,
        block_size: int,
        capacity_tokens: int,
        model: Any = None,
        prefetch: bool = False,
        dense_layers: int = QUEST_DENSE_LAYERS,
        host_pools: list[torch.Tensor] | None = None,
        thrash_window: int = 16,
        instrument: bool = False,
        n_slots: int | None = None,
        fetch: str = "runs",
        stages: Any = None,
        quant: str | None = None,
        record_selection: bool = False,
        replay_selection: Any = None,
        tiers: dict[int, TieredLayer] | None = None,
        *,
        exact: bool = False,
        rank_dtype: torch.dtype | None = torch.float32,
    ) -> None:
        if not isinstance(full, FullGPUCache):
            full = FullGPUCache.from_kv(list(full), capacity_tokens)
        super().__init__(layers=full.layers)
        mode = device_fetch(fetch)
        if quant is not None and fetch == "runs":
            # The reference's rule (lazykv/tiered.py:571-572): "runs" copies host bytes straight into
            # slots, which cannot hold an int8 record.
            raise ValueError(f"the int8 tier needs fetch='gather', got {fetch!r}")
        if prefetch and model is None:
            raise ValueError("prefetch needs the model, to speculate the next layer's query")
        if mode == "zerocopy" and (prefetch or record_selection or replay_selection is not None):
            raise ValueError("the zero-copy fetch has no residency to prefetch, record or replay")
        if prefetch or record_selection or replay_selection is not None:
            raise ValueError("residency prefetch / record / replay are rung 6-7 features outside this path")
        self.full = full
        self.k_blocks, self.block_size, self.dense_layers = k_blocks, block_size, dense_layers
        self.fetch, self.quant, self.exact_split = fetch, quant, exact
        self.prefetch, self.thrash_window, self.instrument, self.stages = False, thrash_window, instrument, stages
        self.counters = TierCounters()
        self.tiers = self._tier_layers(tiers, host_pools, capacity_tokens, n_slots, rank_dtype)
        self.counters.boundary_d2h_bytes = sum(t.boundary_d2h_bytes for t in self.tiers.values())
        first = next(iter(self.tiers.values()))
        self.n_slots = first.n_slots
        dev = first.pool.device
        # One index buffer and one workspace shared by every layer: layers run in order on one stream.
        self._idx = torch.empty((first.h, k_blocks), dtype=torch.int32, device=dev)
        self._ws = kernels.Workspace(dev)
        self._dense = DenseScratch()  # multi-token forwards: the layer's whole KV, one layer at a time
        if exact:
            self.policy_name = "tiered_exact"
        elif quant:
            self.policy_name = "tiered_int8"
        else:
            self.policy_name = {"zerocopy": "tiered_zerocopy", "runs": "tiered_sync", "gather": "tiered_sync"}.get(fetch, f"tiered_{fetch}")

    def _tier_layers(self, tiers: dict[int, TieredLayer] | None, host_pools: list[torch.Tensor] | None, capacity_tokens: int,
                     n_slots: int | None, rank_dtype: torch.dtype | None) -> dict[int, TieredLayer]:
        """The selecting layers' tiers: those given (one per layer from `dense_layers` on), or one
        built here from each layer's prefilled KV in `full`, with host pool `host_pools[j]` for the
        j-th selecting layer when pools are supplied."""
        selecting = range(self.dense_layers, len(self.full.layers))
        if tiers is not None:
            if sorted(tiers) != list(selecting):
                raise ValueError(f"prebuilt tiers must cover layers {selecting.start}..{selecting.stop - 1}, got {sorted(tiers)}")
            return tiers
        built: dict[int, TieredLayer] = {}
        for j, layer_idx in enumerate(selecting):
            dense = self.full.layers[layer_idx]
            length = dense.get_seq_length()
            pool = host_pools[j] if host_pools is not None else None
            built[layer_idx] = TieredLayer(dense.keys[:, :, :length], dense.values[:, :, :length], self.k_blocks, self.block_size, capacity_tokens,
                                           pool, n_slots, quant=self.quant, fetch=self.fetch, exact=self.exact_split, rank_dtype=rank_dtype)
        return built

    # -- transformers plumbing --------------------------------------------------------------------

    def update(self, key_states: torch.Tensor, value_states: torch.Tensor, layer_idx: int, *args: object, **kwargs: object) -> tuple[torch.Tensor, torch.Tensor]:
        tier = self.tiers.get(layer_idx)
        if tier is None:
            return self.full.layers[layer_idx].update(key_states, value_states)
        n_new = key_states.shape[-2]
        if n_new == 1:
            tier.append(key_states, value_states, self.counters)
            # Attention never reads this: select() supplies the attention of every decode step.
            return tier.pool[1:2, :, 0], tier.pool[1:2, :, 1]
        return self._ingest_turn(tier, key_states, value_states)

    def _ingest_turn(self, tier: TieredLayer, keys: torch.Tensor, values: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
        """A forward of several tokens (a user's turn, lazykv/tiered.py:649-663). Its queries attend
        the layer's whole KV densely, so the attention gets the sealed blocks (read once over the link
        into the dense scratch), the current block and the new tokens as one [1, h, L + T, d] view; the
        new tokens then enter the tier with the state token-by-token appends leave."""
        dense_k, dense_v, link_bytes = tier.dense_kv(keys, values, self._dense)
        tier.extend(keys, values, self.counters)
        counted = self.counters
        counted.ingest_forwards += 1
        counted.ingest_tokens += keys.shape[-2]
        counted.ingest_h2d_bytes += link_bytes
        return dense_k, dense_v

    def get_seq_length(self, layer_idx: int = 0) -> int:
        tier = self.tiers.get(layer_idx)
        return tier.length if tier is not None else self.full.layers[layer_idx].get_seq_length()

    def model_kwargs(self) -> dict[str, object]:
        return {"lazykv_selector": self}

    # -- decode path ----------------------------------------------------------------------------

    def select(self, layer_idx: int, query: torch.Tensor, key: torch.Tensor | None = None, value: torch.Tensor | None = None, scaling: float | None = None) -> Decoded | None:
        tier = self.tiers.get(layer_idx)
        if tier is None or query.shape[-2] != 1:
            return None
        if tier.fused_select():
            out, lse = tier.decode(query, scaling, ws=self._ws)
        else:
            idx = tier.rank(query, out=self._idx, ws=self._ws)
            out, lse = tier.decode(query, scaling, idx=idx, ws=self._ws)
        c = self.counters
        c.selections += 1
        c.selected_pairs += tier.h * tier.k
        if tier.fetch == "zerocopy":
            c.zerocopy_bytes += tier.h * tier.k * tier.pair_bytes
        if tier.exact:
            c.remainder_pairs += tier.h * (tier.n_sealed - 1 - tier.k)
        n_q = out.shape[0]
        return Decoded(out.view(1, n_q, 1, tier.d), lse.view(1, n_q))

    def close(self) -> None:
        pass

    def stats(self) -> CacheStats:
        """VRAM held for decode (dense layers' KV, slot pools, stores, metadata) and host bytes no
        GPU copy holds, so gpu / (gpu + host) is the residency fraction (lazykv/tiered.py:841-848)."""
        dense = sum(self.full.layers[i].resident_bytes() for i in range(len(self.full.layers)) if i not in self.tiers)
        gpu = dense + sum(t.gpu_bytes() + t.metadata_bytes() for t in self.tiers.values())
        host = sum(t.not_resident_bytes() for t in self.tiers.values())
        return CacheStats(seq_len=self.get_seq_length(self.dense_layers), gpu_resident_kv_bytes=gpu, host_kv_bytes=host, gpu_allocated_kv_bytes=gpu)

    def host_logical_bytes(self) -> int:
        """What the off-GPU KV would occupy in the model dtype, whatever precision the tier stores
        it in (lazykv/tiered.py:850-857): stats().host_kv_bytes over this is the int8 saving."""
        return sum(t.not_resident_logical_bytes() for t in self.tiers.values())

    def host_pinned_bytes(self) -> int:
        return sum(t.host.numel() * t.host.element_size() for t in self.tiers.values() if t.host is not None)

    def counters_dict(self) -> dict[str, Any]:
        from dataclasses import asdict

        return asdict(self.counters)


@dataclass
class ExactCounters:
    """What the exact split adds, with the reference's fields (lazykv/exact.py:55-66). The
    remainder is attended by the decode kernel on the device, so the CPU and merge times stay 0;
    `merges` counts exact steps, `cold_tokens` the remainder's tokens (the sealed blocks outside
    the sink and the selection), and `returned_bytes` is 0 (no partial returns to the host)."""

    merges: int = 0
    cpu_attention_s: float = 0.0
    host_merge_s: float = 0.0
    mirror_s: float = 0.0
    boundary_mirror_s: float = 0.0
    cpu_tokens: int = 0
    cold_tokens: int = 0
    returned_bytes: int = 0


class ExactTieredCache(TieredCache):
    """Rung 9 on the GPU: the selected blocks attended from HBM, every other sealed block from the
    host tier, merged exactly (lazykv/exact.py:155-264), all inside the decode's launches.

    With the reference's rung-6 fetches ("runs", its default, or "gather") the selected blocks come
    from the hybrid tier's HBM slots, as rung 9 builds on rung 6; with "resident" from an HBM store
    of every block. Unlike the reference, an int8 host tier is allowed: the cold partial (and, over
    slots, the selected blocks too) is computed from the dequantised records. `mirrors` and
    `threads` are the reference's float32 CPU mirrors and the thread count of its CPU pass; this
    path has no CPU pass, so they are accepted and unused (`threads` is kept as an attribute and
    torch's thread count is left alone)."""

    def __init__(self, full, *args: Any, mirrors: Any = None, threads: int | None = 8, **kwargs: Any) -> None:  # noqa: ANN001
        if kwargs.get("fetch") == "zerocopy":
            # lazykv/exact.py:169-172: the remainder excludes the selection, which the exact tier
            # reads from HBM.
            raise ValueError("rung 9 needs the selection on the host; it cannot use the zero-copy fetch")
        if kwargs.get("prefetch"):
            raise ValueError("rung 9 does not prefetch; the cold set is attended, not fetched")
        kwargs["exact"] = True
        super().__init__(full, *args, **kwargs)
        self.policy_name = "tiered_exact"
        self.exact = ExactCounters()
        self.threads = threads
        self.mirrors = mirrors

    def select(self, layer_idx: int, query: torch.Tensor, key: torch.Tensor | None = None, value: torch.Tensor | None = None, scaling: float | None = None) -> Decoded | None:
        got = super().select(layer_idx, query, key, value, scaling)
        tier = self.tiers.get(layer_idx)
        if got is not None and tier is not None:
            self.exact.merges += 1
            self.exact.cold_tokens += tier.h * (tier.n_sealed - 1 - tier.k) * tier.bs
        return got

    def mirror_bytes(self) -> int:
        return 0  # no float32 CPU mirror: the remainder is read from the host tier itself

    def exact_counters_dict(self) -> dict[str, Any]:
        """The exact split's counters, the thread count and the mirror bytes (lazykv/exact.py:300-304)."""
        from dataclasses import asdict

        d = asdict(self.exact)
        d["threads"] = self.threads
        d["mirror_bytes"] = self.mirror_bytes()
        return d
