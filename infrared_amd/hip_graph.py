"""hipGraph capture/replay of the decode step (replaces ``infrared/engine/cuda_graph.py``).

Same API as the reference module:

- ``default_buckets`` / ``pick_bucket`` (``infrared/engine/cuda_graph.py:58-81``);
- ``build_decode_static_inputs`` (``:105-155``): fixed-shape inputs for a batch
  bucket, pad-by-repeating row 0, key axis padded to ``t_max``. Built by one
  kernel (``ir_decode_inputs``) instead of a Python loop over ``B * ctx``
  tokens, and carrying the ``block_tables``/``context_lens`` the HIP decode kernel reads;
- ``HipGraphDecoder`` (in place of ``CudaGraphDecoder``, ``:170-287``): one
  captured graph per bucket sharing one memory pool; ``decode()`` builds the
  step's metadata in the static buffers and replays.

PyTorch-ROCm's ``torch.cuda.CUDAGraph`` is a hipGraph; the HIP kernels are
launched on torch's current stream, so they are captured as graph kernel
nodes. They neither synchronise nor allocate. The pool's decode buffers
(split-KV workspace, arrival counters, plan buffer) are grown during a
bucket's warm-up, outside capture; a larger bucket captured later may grow
them again, which replaces the pool's tensors, so every captured graph keeps
references to the buffers it was captured with and its replays stay on that
live memory. The kernel reads only ``context_lens[b]`` keys per row, so a
replay costs the real context, not ``t_max``.
"""

from __future__ import annotations

import contextlib
import gc
import threading
from collections.abc import Callable, Iterator, Sequence
from dataclasses import dataclass

import numpy as np
import torch

from infrared_amd import metadata
from infrared_amd._lib import check, dtype_code, lib, on_device, ptr, stream_ptr
from infrared_amd.paged_kv_cache import PagedContext, PagedKVPool, host_list, to_device


def default_buckets(max_num_seqs: int) -> tuple[int, ...]:
    """Powers of two below ``max_num_seqs``, then ``max_num_seqs`` itself."""
    if max_num_seqs < 1:
        raise ValueError("max_num_seqs must be >= 1")
    out: list[int] = []
    p = 1
    while p < max_num_seqs:
        out.append(p)
        p *= 2
    out.append(max_num_seqs)
    return tuple(out)


def pick_bucket(b: int, buckets: tuple[int, ...]) -> int:
    """Smallest bucket ``>= b``; raises ``ValueError`` past the largest."""
    for bucket in buckets:
        if bucket >= b:
            return bucket
    raise ValueError(f"batch size {b} exceeds largest bucket {buckets[-1]}")


@dataclass(slots=True)
class DecodeInputs:
    """Fixed-shape decode inputs for bucket ``B`` and key axis ``t_max``.

    ``ids`` ``[B, 1]``, ``positions`` ``[B, 1]``, ``write_slots`` ``[B]``,
    ``gather_slots`` ``[B, t_max]``, ``mask`` ``[B, 1, 1, t_max]`` (the
    reference fields), plus ``block_tables`` ``[B, ceil(t_max / bs)]`` int32 and
    ``context_lens`` ``[B]`` int32.
    """

    ids: torch.Tensor
    positions: torch.Tensor
    write_slots: torch.Tensor
    gather_slots: torch.Tensor
    mask: torch.Tensor
    block_tables: torch.Tensor
    context_lens: torch.Tensor


def build_decode_static_inputs(
    block_tables: Sequence[Sequence[int]],
    num_cached: Sequence[int],
    last_tokens: Sequence[int],
    bucket_b: int,
    t_max: int,
    block_size: int,
    device: torch.device | str,
    dtype: torch.dtype,
) -> DecodeInputs:
    """One decode step's inputs at fixed ``(bucket_b, t_max)``; rows ``[b:]`` repeat row 0.

    Row ``i``'s new token is at position ``num_cached[i]`` (written to
    ``slot(bt_i, num_cached[i])``) and attends ``[0, num_cached[i]]``.
    """
    device = torch.device(device)
    num_cached, last_tokens = _check_rows(num_cached, last_tokens, bucket_b, t_max)
    b = len(last_tokens)
    width = metadata.blocks_for(t_max, block_size)
    if device.type == "cuda" and dtype in _MASK_DTYPES and bucket_b < 65536:
        out = DecodeInputs(
            ids=torch.empty(bucket_b, 1, dtype=torch.long, device=device),
            positions=torch.empty(bucket_b, 1, dtype=torch.long, device=device),
            write_slots=torch.empty(bucket_b, dtype=torch.long, device=device),
            gather_slots=torch.empty(bucket_b, t_max, dtype=torch.long, device=device),
            mask=torch.empty(bucket_b, 1, 1, t_max, dtype=dtype, device=device),
            block_tables=torch.empty(bucket_b, width, dtype=torch.int32, device=device),
            context_lens=torch.empty(bucket_b, dtype=torch.int32, device=device),
        )
        _fill_inputs(out, block_tables, num_cached, last_tokens, block_size)
        return out
    rows = [i if i < b else 0 for i in range(bucket_b)]
    bt = metadata.block_tables_tensor(
        [list(block_tables[j])[:width] for j in rows], device, width
    )
    cl = torch.tensor([num_cached[j] + 1 for j in rows], dtype=torch.int32, device=device)
    nc = torch.tensor([num_cached[j] for j in rows], dtype=torch.long, device=device)
    ids = torch.tensor([[last_tokens[j]] for j in rows], dtype=torch.long, device=device)
    return DecodeInputs(
        ids=ids,
        positions=nc[:, None].clone(),
        write_slots=metadata.decode_write_slots(bt, nc, block_size),
        gather_slots=metadata.gather_slots_from_tables(bt, cl, block_size, t_max),
        mask=metadata.decode_mask(cl, t_max, dtype),
        block_tables=bt,
        context_lens=cl,
    )


_MASK_DTYPES = (torch.float32, torch.float16, torch.bfloat16)


def _check_rows(num_cached: Sequence[int], last_tokens: Sequence[int], bucket_b: int,
                t_max: int) -> tuple[list[int], list[int]]:
    """The cached lengths and last tokens of a step that fits ``(bucket_b,
    t_max)``, one of each per row; raises otherwise."""
    b = len(last_tokens)
    if not 0 < b <= bucket_b:
        raise ValueError(f"need 0 < b ({b}) <= bucket_b ({bucket_b})")
    cached = list(map(int, host_list(num_cached)[:b]))
    if len(cached) < b:
        raise IndexError(f"{len(cached)} cached lengths for {b} rows")
    for n in cached:
        if n < 0:
            raise ValueError(f"num_cached {n} is negative")
        if n + 1 > t_max:
            raise ValueError(f"context_len {n + 1} exceeds t_max {t_max}")
    return cached, list(map(int, host_list(last_tokens)))


def _fill_inputs(out: DecodeInputs, block_tables: Sequence[Sequence[int]], num_cached: list[int],
                 last_tokens: list[int], block_size: int) -> None:
    """Writes a step's inputs (lengths and tokens as ``_check_rows`` gives them)
    into ``out`` (device tensors, contiguous): one host array, one copy, one
    launch (``ir_decode_inputs``)."""
    b, (bucket_b, width) = len(last_tokens), out.block_tables.shape
    host = np.zeros(4 * b + b * width, dtype=np.int32)
    rows = host[: 4 * b].view(np.int64).reshape(b, 2)
    rows[:, 0] = num_cached
    rows[:, 1] = last_tokens
    metadata.fill_tables(host[4 * b :].reshape(b, width), [list(block_tables[j])[:width] for j in range(b)])
    dev = out.mask.device
    staging = to_device(host, dev)
    with on_device(dev):
        check(lib().ir_decode_inputs(
            ptr(staging), b, bucket_b, width, block_size, out.mask.shape[-1], dtype_code(out.mask.dtype), ptr(out.ids),
            ptr(out.positions), ptr(out.write_slots), ptr(out.gather_slots), ptr(out.mask), ptr(out.block_tables),
            ptr(out.context_lens), stream_ptr(dev),
        ), "ir_decode_inputs")
    # written through raw pointers: what is cached of these tensors (the pool's
    # reference-form check of gather_slots and mask) has to see that they changed
    torch.autograd.graph.increment_version([getattr(out, n) for n in DecodeInputs.__slots__])


_gc_lock = threading.Lock()
_gc_captures = 0  # captures under way
_gc_enabled = False  # whether the first of them found the collector on


@contextlib.contextmanager
def capturing(graph: torch.cuda.CUDAGraph, pool=None) -> Iterator[None]:
    """``torch.cuda.graph`` with Python's automatic garbage collection held off. A
    collection may find another graph in a reference cycle (a dropped decoder whose
    step function refers to it); a graph's destructor waits for the device, which
    is an error while a stream is capturing, and an error in a destructor ends the
    process."""
    global _gc_captures, _gc_enabled
    with _gc_lock:
        if _gc_captures == 0:
            _gc_enabled = gc.isenabled()
            gc.disable()
        _gc_captures += 1
    try:
        with torch.cuda.graph(graph) if pool is None else torch.cuda.graph(graph, pool=pool):
            yield
    finally:
        with _gc_lock:
            _gc_captures -= 1
            if _gc_captures == 0 and _gc_enabled:
                gc.enable()


@dataclass(slots=True)
class _Captured:
    graph: torch.cuda.CUDAGraph
    buf: DecodeInputs
    out: torch.Tensor
    # the pool buffers the graph's kernels address (kept alive for its replays)
    pool_buffers: tuple


class HipGraphDecoder:
    """Per-bucket hipGraph decode: capture once per bucket, then replay each step.

    ``model`` is anything with the reference model's call
    ``forward(ids, positions, mask, paged=PagedContext)`` returning
    ``[B, 1, vocab]``-like output (the last position is taken), or a plain
    callable ``fn(DecodeInputs, PagedContext) -> Tensor`` passed as
    ``step_fn``. Replays must not overlap (they share one memory pool).
    """

    def __init__(
        self,
        model,
        pool: PagedKVPool,
        *,
        max_num_seqs: int,
        t_max: int,
        block_size: int,
        use_triton: bool = True,
        warmup_steps: int = 3,
        step_fn: Callable[[DecodeInputs, PagedContext], torch.Tensor] | None = None,
    ) -> None:
        self.model = model
        self.pool = pool
        self.buckets = default_buckets(max_num_seqs)
        self.t_max = t_max
        self.block_size = block_size
        self.use_triton = use_triton
        self.warmup_steps = warmup_steps
        self.step_fn = step_fn
        self.device = pool.device
        self.dtype = pool.dtype
        self._graphs: dict[int, _Captured] = {}
        self._mempool = None

    def decode(
        self,
        block_tables: Sequence[Sequence[int]],
        num_cached: Sequence[int],
        last_tokens: Sequence[int],
    ) -> torch.Tensor:
        """Advance the running set one token by graph replay; returns the first ``b`` rows."""
        b = len(last_tokens)
        bucket = pick_bucket(b, self.buckets)
        if bucket in self._graphs and self.dtype in _MASK_DTYPES and bucket < 65536:
            cached, tokens = _check_rows(num_cached, last_tokens, bucket, self.t_max)
            _fill_inputs(self._graphs[bucket].buf, block_tables, cached, tokens, self.block_size)
        else:
            inp = build_decode_static_inputs(
                block_tables, num_cached, last_tokens, bucket, self.t_max, self.block_size,
                self.device, self.dtype,
            )
            if bucket in self._graphs:  # (a dtype or bucket the kernel does not take)
                self._copy_inputs(self._graphs[bucket].buf, inp)
            else:
                self._capture(bucket, inp)
        self._graphs[bucket].graph.replay()
        return self._graphs[bucket].out[:b]

    def _context(self, buf: DecodeInputs) -> PagedContext:
        return PagedContext(
            self.pool, buf.write_slots, buf.gather_slots, self.use_triton, buf.block_tables,
            buf.context_lens,
        )

    def _forward(self, buf: DecodeInputs) -> torch.Tensor:
        paged = self._context(buf)
        if self.step_fn is not None:
            return self.step_fn(buf, paged)
        logits = self.model.forward(buf.ids, buf.positions, buf.mask, paged=paged)
        return logits[:, -1]

    @staticmethod
    def _copy_inputs(dst: DecodeInputs, src: DecodeInputs) -> None:
        for name in DecodeInputs.__slots__:
            getattr(dst, name).copy_(getattr(src, name))

    def _capture(self, bucket: int, inp: DecodeInputs) -> None:
        buf = DecodeInputs(*(getattr(inp, n).clone() for n in DecodeInputs.__slots__))
        stream = torch.cuda.Stream(device=self.device)
        stream.wait_stream(torch.cuda.current_stream(self.device))
        with torch.cuda.stream(stream):
            for _ in range(self.warmup_steps):
                self._forward(buf)
        torch.cuda.current_stream(self.device).wait_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with capturing(graph, self._mempool):
            out = self._forward(buf)
        if self._mempool is None:
            self._mempool = graph.pool()
        held = tuple(getattr(self.pool, n, None) for n in ("_workspace", "_counters", "_plan_buf"))
        self._graphs[bucket] = _Captured(graph=graph, buf=buf, out=out, pool_buffers=held)
