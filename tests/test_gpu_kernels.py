"""GPU parity of the HIP kernels (called through the C ABI) against the CPU
oracle and torch library routines on the same seeded inputs.

Bars: bit-exact for the scatter, the gathers and block-table indexing;
max-abs error <= 1e-4 for fp32 and <= 2e-2 for bf16/fp16 against an fp32
reference.
"""

from __future__ import annotations

import pytest
import torch

from infrared_amd import kernels, metadata
from infrared_amd._lib import (
    DTYPE_BF16, ERR_BLOCK_RANGE, ERR_CONTEXT_RANGE, ERR_GATHER_RANGE, ERR_SLOT_RANGE, check, dtype_code, lib, ptr,
    stream_ptr,
)
from infrared_amd.workloads import DECODE_CONFIGS, DecodeConfig, make_decode_case
from oracle import naive as O

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2, torch.float16: 2e-2}


def _err():
    return torch.zeros(1, dtype=torch.int32, device=DEV)


# ------------------------------------------------------------------ scatter


@pytest.mark.parametrize("head_major", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h_kv,d", [(2, 64), (4, 128), (1, 8), (3, 4)])
def test_scatter_bit_exact_vs_index_put(dtype, h_kv, d, head_major):
    g = torch.Generator(device=DEV).manual_seed(d + h_kv)
    num_slots, n = 512, 97
    base = torch.randn(num_slots, h_kv, d, generator=g, device=DEV).to(dtype)
    if head_major:
        base = base.permute(1, 0, 2).contiguous().permute(1, 0, 2)
    kc, vc = base.clone(), (base * -1).clone()  # clone keeps the strides
    assert kc.stride() == base.stride()
    k = torch.randn(n, h_kv, d, generator=g, device=DEV).to(dtype)
    v = torch.randn(n, h_kv, d, generator=g, device=DEV).to(dtype)
    slots = torch.randperm(num_slots, device=DEV)[:n]
    err = _err()
    kernels.kv_scatter(kc, vc, k, v, slots, err)
    want_k, want_v = base.clone(), (base * -1).clone()
    want_k[slots] = k
    want_v[slots] = v
    torch.cuda.synchronize()
    assert torch.equal(kc, want_k) and torch.equal(vc, want_v)
    assert err.item() == 0
    # the CPU oracle agrees bit for bit
    ok, ov = base.cpu(), (base * -1).cpu()
    O.pool_write(ok, ov, k.cpu(), v.cpu(), slots.cpu())
    assert torch.equal(kc.cpu(), ok) and torch.equal(vc.cpu(), ov)


def test_scatter_strided_source_skip_and_flag():
    """k/v as views of a fused projection; negative slots skip; OOB slots are flagged, not written."""
    h_q, h_kv, d, n = 28, 4, 128, 64
    qkv = torch.randn(n, h_q + 2 * h_kv, d, device=DEV).bfloat16()
    k, v = qkv[:, h_q : h_q + h_kv], qkv[:, h_q + h_kv :]
    kc = torch.zeros(1024, h_kv, d, device=DEV, dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    slots = torch.arange(n, device=DEV) * 7
    slots[5] = -1
    slots[9] = 1024 + 3
    err = _err()
    kernels.kv_scatter(kc, vc, k, v, slots, err)
    torch.cuda.synchronize()
    assert err.item() == ERR_SLOT_RANGE
    keep = torch.ones(n, dtype=torch.bool, device=DEV)
    keep[5] = keep[9] = False
    want = torch.zeros_like(kc)
    want[slots[keep]] = k[keep]
    assert torch.equal(kc, want)
    want_v = torch.zeros_like(vc)
    want_v[slots[keep]] = v[keep]
    assert torch.equal(vc, want_v)


def test_scatter_duplicate_identical_rows_idempotent():
    """Pad-by-repeat rows write the same row to the same slot (infrared/engine/cuda_graph.py:22-25)."""
    kc = torch.zeros(64, 2, 64, device=DEV)
    vc = torch.zeros_like(kc)
    k = torch.randn(3, 2, 64, device=DEV)
    k = torch.cat([k, k[:1], k[:1]])
    v = k * 2
    slots = torch.tensor([10, 20, 30, 10, 10], device=DEV)
    kernels.kv_scatter(kc, vc, k, v, slots)
    torch.cuda.synchronize()
    assert torch.equal(kc[10], k[0]) and torch.equal(vc[20], v[1]) and torch.equal(kc[30], k[2])


# ------------------------------------------------------------------ gathers


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gather_slots_bit_exact(dtype):
    kc = torch.randn(300, 2, 64, device=DEV).to(dtype)
    vc = torch.randn(300, 2, 64, device=DEV).to(dtype)
    gs = torch.randint(0, 300, (3, 41), device=DEV)
    ok, ov = kernels.gather_slots(kc, vc, gs)
    wk, wv = O.pool_gather(kc.cpu(), vc.cpu(), gs.cpu())
    assert torch.equal(ok.cpu(), wk) and torch.equal(ov.cpu(), wv)
    err = _err()
    gs[1, 3] = 300
    ok, _ = kernels.gather_slots(kc, vc, gs, err)
    torch.cuda.synchronize()
    assert err.item() == ERR_GATHER_RANGE and ok[1, 3].eq(0).all()


@pytest.mark.parametrize("bs", [1, 4, 8, 16, 32])
def test_block_table_gather_bit_exact(bs):
    """Block-table indexing (slot = bt[p // bs] * bs + p % bs) against the oracle's loop."""
    g = torch.Generator().manual_seed(bs)
    b, h_kv, d = 5, 2, 64
    ctx = torch.randint(1, 200, (b,), generator=g)
    nblk = (ctx + bs - 1) // bs
    num_blocks = int(nblk.sum()) + 7
    perm = torch.randperm(num_blocks, generator=g)
    tables, off = [], 0
    for n in nblk.tolist():
        tables.append(perm[off : off + n].tolist())
        off += n
    kc = torch.randn(num_blocks * bs, h_kv, d, device=DEV).bfloat16()
    vc = torch.randn_like(kc)
    bt = metadata.block_tables_tensor(tables, DEV)
    cl = ctx.to(torch.int32).to(DEV)
    t_max = int(ctx.max()) + 5
    ok, ov = kernels.paged_gather(kc, vc, bt, cl, bs, t_max)
    gs = O.decode_gather_slots(tables, ctx.tolist(), bs, t_max)
    wk, wv = O.pool_gather(kc.cpu(), vc.cpu(), gs)
    valid = torch.arange(t_max)[None, :] < ctx[:, None]
    wk[~valid] = 0
    wv[~valid] = 0
    assert torch.equal(ok.cpu(), wk) and torch.equal(ov.cpu(), wv)


# ------------------------------------------------------------------ decode


def _check_decode(case, partition_tokens=0, seqs=None):
    cfg = case.config
    bt = case.block_tables[0]
    err = _err()
    out = kernels.paged_decode(
        case.q, case.k_cache, case.v_cache, bt, case.context_lens, cfg.block_size, cfg.scale,
        partition_tokens=partition_tokens, err_flags=err,
    )
    torch.cuda.synchronize()
    assert err.item() == 0
    ref = O.decode_reference(
        case.q.cpu(), case.k_cache.cpu(), case.v_cache.cpu(), bt.cpu(), case.context_lens.cpu(),
        cfg.block_size, cfg.scale, torch.float32, seqs=seqs,
    )
    got = out.float().cpu()
    rows = list(range(cfg.num_seqs)) if seqs is None else list(seqs)
    diff = (got[rows] - ref[rows]).abs().max().item()
    assert diff <= TOL[cfg.dtype], f"{cfg.name} P={partition_tokens}: max-abs {diff}"
    return out


@pytest.mark.parametrize("layout", ["head_major", "slot_major"])
def test_decode_qwen05b_fp32_parity(layout):
    """Qwen2.5-0.5B shape, fp32: 8 seqs, 14/2 heads, D=64, ctx U[1,512]; bar 1e-4."""
    _check_decode(make_decode_case("qwen0.5b-fp32", DEV, layout=layout))


@pytest.mark.parametrize("layout", ["head_major", "slot_major"])
@pytest.mark.parametrize("partition_tokens", [0, 256, 4096])
def test_decode_qwen7b_bf16_full_size_parity(partition_tokens, layout):
    """Qwen2.5-7B shape, bf16, full batch of 64 with ctx U[512,4096]; bar 2e-2 vs fp32,
    in both pool layouts."""
    _check_decode(make_decode_case("qwen7b-bf16", DEV, layout=layout), partition_tokens)


def test_decode_skewed_long_context_split_kv():
    """Lognormal contexts up to 32k through split-KV partitions + reduce."""
    case = make_decode_case("qwen7b-skewed", DEV)
    assert int(case.context_lens.max()) > 4096
    _check_decode(case, 512)
    _check_decode(case, 0)


_SWEEP = [
    # (dtype, h_q, h_kv, d, bs, partition)
    (torch.float32, 14, 2, 64, 16, 32),
    (torch.float32, 8, 8, 128, 16, 48),
    (torch.bfloat16, 28, 4, 128, 8, 64),
    (torch.bfloat16, 16, 2, 128, 32, 96),
    (torch.bfloat16, 40, 2, 64, 16, 16),
    (torch.bfloat16, 4, 4, 64, 1, 160),
    (torch.float16, 28, 4, 128, 16, 256),
    (torch.float16, 12, 2, 64, 4, 80),
]


@pytest.mark.parametrize("dtype,h_q,h_kv,d,bs,part", _SWEEP)
def test_decode_shape_sweep(dtype, h_q, h_kv, d, bs, part):
    """GQA groups 1..20 (two head groups at 20), both head dims, block sizes 1..32
    (per-lane and block-uniform addressing), partition sizes that split mid-block,
    and context lengths on both sides of tile and block boundaries."""
    cfg = DecodeConfig(f"sweep-{h_q}-{h_kv}-{d}-{bs}", 7, h_q, h_kv, d, bs, dtype, "uniform", 300, 300, seed=h_q + bs)
    case = make_decode_case(cfg, DEV)
    # every row owns blocks for 300 tokens; use shorter lengths within them
    case.context_lens.copy_(torch.tensor([1, 15, 16, 17, 31, 33, 300], dtype=torch.int32))
    _check_decode(case, part)


# Batches mixing empty, one-token and long rows (one row spanning many
# partitions), a single 32k-token row, and a batch wider than one workgroup.
_MIX_CFG = DecodeConfig("mixed-lengths", 8, 28, 4, 128, 16, torch.bfloat16, "uniform", 5000, 5000, seed=11)


@pytest.mark.parametrize("partition_tokens", [0, 64, 4096])
def test_decode_mixed_lengths_with_empty_rows(partition_tokens):
    case = make_decode_case(_MIX_CFG, DEV)
    case.context_lens.copy_(torch.tensor([0, 1, 5000, 0, 17, 4096, 0, 2048], dtype=torch.int32))
    out = _check_decode(case, partition_tokens)
    for r in (0, 3, 6):
        assert out[r].float().abs().max().item() == 0.0


@pytest.mark.parametrize("ctx", [1, 16, 32768])
def test_decode_single_sequence(ctx):
    """One sequence: a single key, one full tile, and 32k keys (8 default
    partitions per unit, merged by the reduce launch)."""
    cfg = DecodeConfig(f"one-seq-{ctx}", 1, 28, 4, 128, 16, torch.bfloat16, "uniform", ctx, ctx, seed=ctx)
    _check_decode(make_decode_case(cfg, DEV), 0)


def test_decode_large_batch():
    cfg = DecodeConfig("batch-600", 600, 8, 2, 64, 16, torch.float16, "uniform", 1, 64, seed=5)
    _check_decode(make_decode_case(cfg, DEV), 0)


def test_decode_all_rows_empty():
    case = make_decode_case(_MIX_CFG, DEV)
    case.context_lens.zero_()
    out = _check_decode(case, 0)
    assert out.float().abs().max().item() == 0.0


_VARIANT_CHILD = r"""
import sys, torch
sys.path.insert(0, {root!r})
from infrared_amd import kernels
from infrared_amd.workloads import DecodeConfig, make_decode_case
from oracle import naive as O
for ctx, part in ((5000, 256), (777, 64), (4096, 0)):
    cfg = DecodeConfig("variant", 8, 28, 4, 128, 16, torch.bfloat16, "uniform", 1, ctx, seed=ctx)
    case = make_decode_case(cfg, "cuda")
    bt = case.block_tables[0]
    out = kernels.paged_decode(case.q, case.k_cache, case.v_cache, bt, case.context_lens, 16, cfg.scale,
                               partition_tokens=part)
    ref = O.decode_reference(case.q.cpu(), case.k_cache.cpu(), case.v_cache.cpu(), bt.cpu(),
                             case.context_lens.cpu(), 16, cfg.scale, torch.float32)
    diff = (out.float().cpu() - ref).abs().max().item()
    print(ctx, part, diff, flush=True)
    assert diff <= 2e-2, diff
print("VARIANT OK")
"""


@pytest.mark.parametrize(
    "env",
    [{"IR_DECODE_MERGE": "kernel", "IR_DECODE_DEPTH": "2"}, {"IR_DECODE_DEPTH": "3", "IR_DECODE_WAVES": "8"}],
    ids=["reduce-launch-depth2", "depth3-waves8"],
)
def test_decode_launch_variants(env):
    """The tuning knobs' other launch shapes (a second merge launch, deeper load
    rings, 8 wavefronts) keep the oracle's results on split and unsplit
    sequences. The knobs are read once per process, so each runs in a child."""
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run(
        [sys.executable, "-c", _VARIANT_CHILD.format(root=root)], env={**os.environ, **env},
        capture_output=True, text=True, timeout=110, cwd=root,
    )
    assert res.returncode == 0 and "VARIANT OK" in res.stdout, res.stdout + res.stderr[-2000:]


def test_decode_shared_workspace_across_different_splits():
    """The partial rows start as garbage (every int32 = 2) and are shared by calls
    whose splits and batch sizes differ, as are the arrival counters; each call
    matches the oracle, repeats bit for bit and leaves the counters at zero."""
    case = make_decode_case(_MIX_CFG, DEV)
    cfg = case.config
    bt = case.block_tables[0]
    need = kernels.decode_workspace_bytes(8, 28, 4, 128, bt.shape[1], 16, 256)
    ws = torch.full((need // 4,), 2, dtype=torch.int32, device=DEV).view(torch.uint8)
    ctr = torch.zeros(kernels.decode_num_counters(8, 28, 4), dtype=torch.int32, device=DEV)
    lens = [
        torch.tensor([5000, 5000, 5000, 5000, 5000, 5000, 5000, 5000], dtype=torch.int32),
        torch.tensor([0, 1, 5000, 0, 17, 4096, 0, 2048], dtype=torch.int32),
        torch.tensor([33, 0, 0, 0, 0, 0, 0, 4999], dtype=torch.int32),
        torch.tensor([4000, 17, 5000], dtype=torch.int32),
    ]
    for cl in lens:
        cl = cl.to(DEV)
        b = cl.shape[0]
        outs = [
            kernels.paged_decode(case.q[:b], case.k_cache, case.v_cache, bt[:b], cl, 16, cfg.scale,
                                 partition_tokens=256, workspace=ws, counters=ctr)
            for _ in range(2)
        ]
        torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1])
        assert int(ctr.abs().sum()) == 0
        ref = O.decode_reference(case.q[:b].cpu(), case.k_cache.cpu(), case.v_cache.cpu(), bt[:b].cpu(), cl.cpu(), 16,
                                 cfg.scale)
        assert (outs[0].float().cpu() - ref).abs().max().item() <= TOL[cfg.dtype]


def test_decode_flags_bad_block_ids_and_contexts():
    """Out-of-pool block ids and over-long contexts are flagged and masked, never read."""
    case = make_decode_case("qwen7b-bf16", DEV, num_seqs=4)
    bt = case.block_tables[0].clone()
    bt[1, 3] = case.pool_blocks + 100
    err = _err()
    kernels.paged_decode(case.q, case.k_cache, case.v_cache, bt, case.context_lens, 16, 0.1, err_flags=err)
    torch.cuda.synchronize()
    assert err.item() & ERR_BLOCK_RANGE
    cl = case.context_lens.clone()
    cl[0] = bt.shape[1] * 16 + 50
    err.zero_()
    kernels.paged_decode(case.q, case.k_cache, case.v_cache, case.block_tables[0], cl, 16, 0.1, err_flags=err)
    torch.cuda.synchronize()
    assert err.item() & ERR_CONTEXT_RANGE


@pytest.mark.parametrize("block_size", [0, -16, 1 << 32])
def test_native_calls_refuse_a_zero_block_size(block_size):
    """A division in the native binding must not take the process down, nor by a size
    that is zero in 32 bits."""
    case = make_decode_case("qwen7b-bf16", DEV, num_seqs=2)
    bt, cl = case.block_tables[0], case.context_lens
    with pytest.raises(RuntimeError, match="block_size"):
        kernels.paged_decode(case.q, case.k_cache, case.v_cache, bt, cl, block_size, 0.1)
    cu = torch.tensor([0, 1, 2], dtype=torch.int32, device=DEV)
    with pytest.raises(RuntimeError, match="block_size"):
        kernels.paged_prefill(case.q, case.k_cache, case.v_cache, bt, cu, cl, 1, block_size, 0.1)


@pytest.mark.parametrize("missing", [(0,), (1,), (2,), (1, 2), (0, 1, 2)])
def test_prefill_refuses_an_incomplete_new_kv(missing):
    """new_kv = (k, v, slots) with any of them None is an error, not a read of nothing
    and not a step whose write is left out."""
    case = make_decode_case("qwen7b-bf16", DEV, num_seqs=2)
    cu = torch.tensor([0, 1, 2], dtype=torch.int32, device=DEV)
    rows = torch.zeros(2, 4, 128, dtype=torch.bfloat16, device=DEV)
    new_kv = [rows, rows, torch.zeros(2, dtype=torch.int64, device=DEV)]
    for i in missing:
        new_kv[i] = None
    with pytest.raises(RuntimeError, match="new_kv"):
        kernels.paged_prefill(case.q, case.k_cache, case.v_cache, case.block_tables[0], cu, case.context_lens, 1, 16,
                              0.1, new_kv=tuple(new_kv))


def test_decode_one_hot_probe_returns_exact_v_row():
    """A key whose score dwarfs the rest makes the output equal its V row, which pins
    the block-table address of that key exactly."""
    case = make_decode_case("qwen7b-bf16", DEV, num_seqs=3)
    bt = case.block_tables[0]
    for i in range(3):
        n = int(case.context_lens[i])
        p = n // 2 + 3
        s = int(bt[i, p // 16]) * 16 + p % 16
        for g in range(4):
            case.k_cache[s, g] = (case.q[i, 7 * g] * 64).to(case.k_cache.dtype)
            for h in range(7 * g, 7 * g + 7):
                case.q[i, h] = case.q[i, 7 * g]
    out = kernels.paged_decode(case.q, case.k_cache, case.v_cache, bt, case.context_lens, 16, 1.0)
    torch.cuda.synchronize()
    for i in range(3):
        n = int(case.context_lens[i])
        p = n // 2 + 3
        s = int(bt[i, p // 16]) * 16 + p % 16
        for h in range(28):
            assert torch.equal(out[i, h], case.v_cache[s, h // 7]), (i, h)


# ------------------------------------------------------------------ gather_slots + mask kernel


def _masked_check(q, kc, vc, gs, mask, scale, n_rep, tol):
    out = kernels.paged_attention_masked(q, kc, vc, gs, mask, scale)
    torch.cuda.synchronize()
    ref = O.paged_attention_naive(
        q.float().cpu(), kc.float().cpu(), vc.float().cpu(), gs.cpu(), mask.float().cpu(), scale, n_rep
    )
    diff = (out.float().cpu() - ref).abs().max().item()
    assert diff <= tol, diff
    return out


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_masked_decode_form_matches_naive(dtype):
    case = make_decode_case(
        DecodeConfig("m", 6, 28, 4, 128, 16, dtype, "uniform", 1, 700, seed=4), DEV
    )
    tables = [[int(x) for x in row] for row in case.block_tables[0].cpu()]
    ctx = case.context_lens.cpu().tolist()
    t_max = max(ctx) + 9
    gs = O.decode_gather_slots(tables, ctx, 16, t_max).to(DEV)
    mask = O.decode_mask(ctx, t_max, dtype).to(DEV)
    out = _masked_check(case.q[:, None], case.k_cache, case.v_cache, gs, mask, case.config.scale, 7, TOL[dtype])
    # and the block-table decode kernel agrees with it within the same bar
    dec = kernels.paged_decode(
        case.q, case.k_cache, case.v_cache, case.block_tables[0], case.context_lens, 16, case.config.scale
    )
    torch.cuda.synchronize()
    assert (dec.float() - out[:, 0].float()).abs().max().item() <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_masked_prefix_hit_prefill_matches_naive(dtype):
    """Prefill with a cached prefix: q rows [num_cached, length), causal mask with offset
    (infrared/model/inputs.py:33-54, infrared/engine/paged_engine.py:194-207)."""
    bs, h_kv, n_rep, d = 16, 2, 7, 64
    num_cached, length = 45, 83
    nb = (length + bs - 1) // bs
    table = torch.randperm(40)[:nb].tolist()
    kc = torch.randn(40 * bs, h_kv, d, device=DEV).to(dtype)
    vc = torch.randn_like(kc)
    gs = torch.tensor([[O.slot(table, p, bs) for p in range(length)]], device=DEV)
    mask = O.attention_mask([0], num_cached, length - num_cached, length, dtype).to(DEV)
    q = torch.randn(1, length - num_cached, h_kv * n_rep, d, device=DEV).to(dtype)
    _masked_check(q, kc, vc, gs, mask, d**-0.5, n_rep, TOL[dtype])


def test_masked_packed_varlen_matches_naive():
    """The packed mixed step: B=1, all chunks' queries and all histories in one frame
    with the varlen mask (infrared/engine/paged_engine.py:461-516)."""
    bs, h_kv, n_rep, d = 16, 4, 7, 128
    dtype = torch.bfloat16
    perm = torch.randperm(200).tolist()
    seqs = [(0, 5), (40, 1), (17, 1), (0, 33)]  # (num_cached, query tokens)
    tables, off = [], 0
    for start, q in seqs:
        nb = (start + q + bs - 1) // bs
        tables.append(perm[off : off + nb])
        off += nb
    q_seq, q_pos, k_seq, k_pos, gsl = [], [], [], [], []
    for i, (start, q) in enumerate(seqs):
        for p in range(start, start + q):
            q_seq.append(i)
            q_pos.append(p)
        for p in range(start + q):
            k_seq.append(i)
            k_pos.append(p)
            gsl.append(O.slot(tables[i], p, bs))
    mask = O.varlen_mask(
        torch.tensor(q_seq), torch.tensor(q_pos), torch.tensor(k_seq), torch.tensor(k_pos), dtype
    ).to(DEV)
    kc = torch.randn(200 * bs, h_kv, d, device=DEV).to(dtype)
    vc = torch.randn_like(kc)
    gs = torch.tensor([gsl], device=DEV)
    q = torch.randn(1, len(q_seq), h_kv * n_rep, d, device=DEV).to(dtype)
    _masked_check(q, kc, vc, gs, mask, d**-0.5, n_rep, TOL[dtype])


def test_masked_fully_masked_row_is_uniform_and_bad_slot_flagged():
    kc = torch.randn(64, 1, 64, device=DEV)
    vc = torch.randn_like(kc)
    gs = torch.arange(20, device=DEV)[None]
    mask = torch.zeros(1, 1, 2, 20, device=DEV)
    mask[0, 0, 1] = torch.finfo(torch.float32).min
    q = torch.randn(1, 2, 1, 64, device=DEV)
    out = _masked_check(q, kc, vc, gs, mask, 0.125, 1, 1e-4)
    assert torch.allclose(out[0, 1, 0].cpu(), vc[:20, 0].mean(0).cpu(), atol=1e-5)
    err = _err()
    gs[0, 4] = 64
    kernels.paged_attention_masked(q, kc, vc, gs, mask, 0.125, err_flags=err)
    torch.cuda.synchronize()
    assert err.item() == ERR_GATHER_RANGE


@pytest.mark.parametrize("b,sq,t,h_kv,n_rep,d,dtype,mask_dtype", [
    (1, 4, 1, 4, 7, 128, torch.bfloat16, torch.bfloat16),     # 28 columns: the narrow kernel, one key
    (3, 1, 1003, 2, 7, 64, torch.float32, torch.float32),     # split, ragged last 16 keys
    (2, 1, 2048, 4, 7, 128, torch.float16, torch.float32),    # split, whole tiles
    (1, 5, 63, 4, 7, 128, torch.bfloat16, torch.bfloat16),    # 35 columns, few keys: the narrow kernel
    (40, 5, 63, 4, 7, 128, torch.bfloat16, torch.bfloat16),   # 40 such sequences: the wide kernel, one ragged tile
    (40, 19, 64, 4, 7, 128, torch.float16, torch.float16),    # 133 columns: a second workgroup of 5
    (1, 292, 320, 4, 7, 64, torch.bfloat16, torch.bfloat16),  # 512 narrow workgroups, the most keys: the narrow kernel
    (1, 293, 320, 4, 7, 64, torch.bfloat16, torch.bfloat16),  # 516: the wide kernel
    (1, 40, 321, 4, 7, 64, torch.float16, torch.float16),     # one key more: the wide kernel
    (1, 40, 577, 2, 7, 64, torch.bfloat16, torch.bfloat16),   # split wide, ragged, head_dim 64
    (2, 37, 700, 4, 7, 128, torch.bfloat16, torch.float32),   # fp32 mask read per lane
    (1, 70, 321, 2, 4, 128, torch.bfloat16, torch.bfloat16),  # 4 heads a token: 16-bit mask read per lane
    (48, 130, 200, 1, 1, 64, torch.float16, torch.float16),   # one head a token
    (64, 27, 130, 1, 5, 128, torch.bfloat16, torch.bfloat16), # 5 heads: 27 tokens in a workgroup
    (1, 9, 4200, 1, 40, 64, torch.bfloat16, torch.bfloat16),  # 40 heads a token
    (2, 40, 1100, 2, 7, 128, torch.float16, torch.float16),   # two sequences
    (2, 250, 1100, 10, 7, 128, torch.float16, torch.float16), # two sequences, surveyed
])
@pytest.mark.parametrize("strided", [False, True])
def test_masked_kernels_at_their_edges(b, sq, t, h_kv, n_rep, d, dtype, mask_dtype, strided):
    """Random masks (zeros, finite biases, finfo.min, one row wholly masked) and a slot
    outside the pool, over both kernels and their splits; ``strided``: key stride 2 in the
    mask (the narrow kernel) and in the slots. The gated call gives the same bits."""
    g = torch.Generator().manual_seed(sq * t)
    slots_n = 1500
    kc = torch.randn(slots_n, h_kv, d, generator=g).to(dtype)
    vc = torch.randn(slots_n, h_kv, d, generator=g).to(dtype)
    gs = torch.randint(0, slots_n, (b, t), generator=g)
    low = max(torch.finfo(mask_dtype).min, torch.finfo(dtype).min)
    mask = torch.randn(b, 1, sq, t, generator=g).to(mask_dtype)
    mask[torch.rand(b, 1, sq, t, generator=g) < 0.6] = low
    mask[0, 0, 0, :] = low
    q = torch.randn(b, sq, h_kv * n_rep, d, generator=g).to(dtype)
    # the oracle without the key whose slot is bad (t = 1 keeps its only key)
    keep = torch.ones(t, dtype=torch.bool)
    bad = t // 2 if t > 1 else None
    if bad is not None:
        keep[bad] = False
    ref = O.paged_attention_naive(q.float(), kc.float(), vc.float(), gs[:, keep], mask[..., keep].float(), d**-0.5,
                                  n_rep)
    if bad is not None:
        gs[:, bad] = slots_n + 3
    gs, mask = gs.to(DEV), mask.to(DEV)
    if strided:
        gs = torch.stack([gs, gs], -1)[..., 0]
        mask = torch.stack([mask, mask], -1)[..., 0]
    args = (q.to(DEV), kc.to(DEV), vc.to(DEV), gs, mask, d**-0.5)
    err = _err()
    out = kernels.paged_attention_masked(*args, err_flags=err)
    assert (out.float().cpu() - ref).abs().max().item() <= TOL[dtype]
    assert err.item() == (ERR_GATHER_RANGE if bad is not None else 0)
    gate = torch.ones(1, dtype=torch.int32, device=DEV)
    gated = torch.full_like(out, 7.0)
    assert torch.equal(kernels.paged_attention_masked(*args, out=gated, run_if=gate), out)
    gate.zero_()
    gated.fill_(7.0)
    kernels.paged_attention_masked(*args, out=gated, run_if=gate)
    assert bool((gated == 7.0).all())


def _masked_without_workspace(q, kc, vc, gs, mask):
    """ir_paged_attention_masked: no survey, every tile walked, one part."""
    (b, sq, hq, d), (n, h_kv, _) = q.shape, kc.shape
    out = torch.empty_like(q)
    check(lib().ir_paged_attention_masked(
        ptr(q), *q.stride()[:3], ptr(kc), ptr(vc), *kc.stride()[:2], n, ptr(gs), *gs.stride(), ptr(mask),
        mask.stride(0), mask.stride(2), mask.stride(3), dtype_code(mask.dtype), ptr(out), *out.stride()[:3], b, sq,
        gs.shape[1], hq, h_kv, d, d**-0.5, dtype_code(q.dtype), None, None, stream_ptr(q.device)),
        "ir_paged_attention_masked")
    return out


def test_masked_runs_without_room_for_its_workspace():
    """An allocator that has no room for a call's partial rows (a pool that takes all the
    memory): the call runs in one part, as it does without a workspace."""
    g = torch.Generator(device=DEV).manual_seed(2)
    kc, vc = (torch.randn(4096, 4, 128, generator=g, device=DEV).bfloat16() for _ in range(2))
    q = torch.randn(1, 512, 28, 128, generator=g, device=DEV).bfloat16()
    gs = torch.randperm(4096, generator=g, device=DEV)[None]
    mask = torch.zeros(1, 1, 512, 4096, dtype=torch.bfloat16, device=DEV)
    need = lib().ir_paged_attention_masked_workspace_size(1, 512, 4096, 28, 4, 128, DTYPE_BF16, DTYPE_BF16, 1)
    assert need > 0
    want = _masked_without_workspace(q, kc, vc, gs, mask)
    out = torch.empty_like(q)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
    try:
        taken = []  # what the allocator still holds
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                taken.append(torch.empty(need, dtype=torch.uint8, device=DEV))
        kernels.paged_attention_masked(q, kc, vc, gs, mask, 128**-0.5, out=out)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(out, want)


@pytest.mark.parametrize("change", ["none", "row masked", "large scores", "nan in v", "inf in k", "bad slot", "faint bias"])
@pytest.mark.parametrize("n_rep,d,dtype,lens", [
    (7, 128, torch.bfloat16, [(2900, 1), (30, 40), (0, 129), (64, 64)]),
    (7, 64, torch.float16, [(0, 64), (4100, 3), (64, 150)]),
])
def test_masked_survey_leaves_out_only_what_adds_nothing(n_rep, d, dtype, lens, change):
    """A long packed frame with the block-diagonal varlen mask, and every reason not to
    leave a tile out: a row without a visible key, scores that reach past the mask,
    values that are not finite, a slot outside the pool, a row that sees only a large
    negative bias. Held against the same call without a workspace (no survey, every
    tile walked) and, where the values are finite, the oracle."""
    h_kv, slots_n = 9, 6000
    q_seq, q_pos, k_seq, k_pos = [], [], [], []
    for i, (start, n) in enumerate(lens):
        q_seq += [i] * n
        q_pos += range(start, start + n)
        k_seq += [i] * (start + n)
        k_pos += range(start + n)
    g = torch.Generator().manual_seed(d)
    sq, t = len(q_seq), len(k_seq)
    assert t >= 1024
    mask = O.varlen_mask(torch.tensor(q_seq), torch.tensor(q_pos), torch.tensor(k_seq), torch.tensor(k_pos), dtype)
    gs = torch.randperm(slots_n, generator=g)[:t][None]
    kc = torch.randn(slots_n, h_kv, d, generator=g).to(dtype)
    vc = torch.randn(slots_n, h_kv, d, generator=g).to(dtype)
    q = torch.randn(1, sq, h_kv * n_rep, d, generator=g).to(dtype)
    if change == "row masked":
        mask[0, 0, sq // 2] = torch.finfo(dtype).min
    elif change == "large scores":
        q *= 3000.0
        kc *= 40.0
        mask[mask < -6e4] = -61440.0  # (finfo(bf16).min would drown any score)
    elif change == "nan in v":
        vc[gs[0, 5]] = float("nan")
    elif change == "inf in k":
        kc[gs[0, 5], :, 3] = float("inf")
    elif change == "faint bias":
        # q.k * scale is 19.9e3, and -19.9e3 for the one key the row sees at -5e4: its
        # masked keys, at -65504 or so, come out ahead of it
        c, e = (32.0, 55.0) if d == 128 else (40.0, 62.0)
        q.fill_(c)
        kc.fill_(e)
        kc[gs[0, t // 2]] = -e
        mask[0, 0, sq // 2] = max(torch.finfo(dtype).min, -65536.0)
        mask[0, 0, sq // 2, t // 2] = -5e4
    ref = None
    naive = lambda m: O.paged_attention_naive(q.float(), kc.float(), vc.float(), gs, m, d**-0.5, n_rep)  # noqa: E731
    if change in ("none", "row masked", "faint bias"):
        ref = naive(mask.float())
    if change in ("large scores", "faint bias"):
        # leaving out every tile nothing is visible in would show
        blind = mask.float().masked_fill(mask <= -6e4, float("-inf"))
        assert (naive(blind) - naive(mask.float())).abs().max().item() > 10 * TOL[dtype]
    if change == "bad slot":
        gs[0, 7] = slots_n
    q, kc, vc, gs, mask = (x.to(DEV) for x in (q, kc, vc, gs, mask))
    err = _err()
    out = kernels.paged_attention_masked(q, kc, vc, gs, mask, d**-0.5, err_flags=err)
    assert err.item() == (ERR_GATHER_RANGE if change == "bad slot" else 0)
    dense = _masked_without_workspace(q, kc, vc, gs, mask)
    assert torch.equal(out.isnan(), dense.isnan())
    # Each call rounds every probability to dtype (half an eps) relative to its own parts'
    # running maxima, so the two differ by at most eps * sum(p |v|) / sum(p) <= eps * max |v|,
    # and by the rounding of the output, eps * |out|.
    eps = torch.finfo(dtype).eps
    vmax = vc[vc.isfinite()].abs().max().item()
    assert torch.allclose(out.float(), dense.float(), rtol=eps, atol=eps * vmax, equal_nan=True)
    if change == "nan in v":
        assert bool(out.isnan().any())
    if ref is not None:
        assert (out.float().cpu() - ref).abs().max().item() <= TOL[dtype]


def _survey_regions(blocks, h_kv, b, nt):
    """Byte offsets of walks and of the end of a surveyed call's workspace head, as the
    survey lays it out: tiles seen per column block, tokens seen per group of 8 tiles,
    then (parts, tiles) per (sequence, KV head, block), then a bound per key tile."""
    up = lambda x: (x + 255) // 256 * 256  # noqa: E731
    walks = up(b * blocks * (-(-nt // 64) * 64)) + up(b * blocks * -(-nt // 8) * 32)
    return walks, walks + up(b * h_kv * blocks * 8) + up(b * h_kv * nt * 4)


@pytest.mark.parametrize("room", ["full", "survey only", "two parts"])
def test_masked_survey_per_sequence_and_head(room):
    """Three frames in one call, each with its own block-diagonal mask; one KV head of the
    second has a NaN in V, so that head walks every tile there and the rest skip. The
    walks, read back from a workspace of the caller's, are those the masks ask for; the
    outputs are the unsurveyed call's and the oracle's; a gated call gives the same bits,
    and with a workspace that holds fewer parts, or none beside the survey, so do the walks."""
    b, sq, t, h_kv, n_rep, d, dtype = 3, 217, 2200, 4, 7, 128, torch.bfloat16
    frames = [[(900, 100), (1000, 100), (83, 17)], [(1900, 60), (83, 157)], [(100, 17), (1783, 100), (100, 100)]]
    g = torch.Generator().manual_seed(17)
    masks = []
    for lens in frames:
        assert (sum(n for _, n in lens), sum(s + n for s, n in lens)) == (sq, t)
        ids = [torch.tensor(x) for x in (
            [i for i, (s, n) in enumerate(lens) for _ in range(n)], [s + j for s, n in lens for j in range(n)],
            [i for i, (s, n) in enumerate(lens) for _ in range(s + n)], [p for s, n in lens for p in range(s + n)])]
        masks.append(O.varlen_mask(*ids, dtype))
    mask = torch.cat(masks)
    gs = torch.randperm(b * t, generator=g).view(b, t)
    kc, vc = (torch.randn(b * t, h_kv, d, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(b, sq, h_kv * n_rep, d, generator=g).to(dtype)
    ref = O.paged_attention_naive(q.float(), kc.float(), vc.float(), gs, mask.float(), d**-0.5, n_rep)
    nan_head = slice(2 * n_rep, 3 * n_rep)
    vc[gs[1, 5], 2] = float("nan")

    blocks, nt = -(-sq * n_rep // 128), -(-t // 64)
    seen = torch.zeros(b, sq, nt * 64, dtype=torch.bool)
    seen[..., :t] = mask[:, 0] > -6e4
    seen = seen.view(b, sq, nt, 64).any(-1)
    tiles = torch.stack([seen[:, i * 128 // n_rep : min(i * 128 + 127, sq * n_rep - 1) // n_rep + 1].any(1).sum(1)
                         for i in range(blocks)], 1)  # [b, blocks]
    assert int(tiles.min()) < nt // 2  # there is something to leave out
    tiles = tiles[:, None].expand(b, h_kv, blocks).clone()
    tiles[1, 2] = nt

    q, kc, vc, gs, mask = (x.to(DEV) for x in (q, kc, vc, gs, mask))
    walks_at, survey_end = _survey_regions(blocks, h_kv, b, nt)
    code = dtype_code(dtype)
    need = lib().ir_paged_attention_masked_workspace_size(b, sq, t, h_kv * n_rep, h_kv, d, code, code, 1)
    part = b * sq * h_kv * n_rep * (d + 2) * 4
    parts = (need - survey_end) // part
    assert need == survey_end + parts * part and parts > 2
    if room != "full":
        parts = 1 if room == "survey only" else 2
        need = survey_end + (0 if parts == 1 else parts * part)
    err = _err()

    def call(run_if=None, out=None):
        out = torch.empty_like(q) if out is None else out
        ws = torch.zeros(need, dtype=torch.uint8, device=DEV)
        check(lib().ir_paged_attention_masked_ws(
            ptr(q), *q.stride()[:3], ptr(kc), ptr(vc), *kc.stride()[:2], kc.shape[0], ptr(gs), *gs.stride(), ptr(mask),
            mask.stride(0), mask.stride(2), mask.stride(3), code, ptr(out), *out.stride()[:3], b, sq, t,
            h_kv * n_rep, h_kv, d, d**-0.5, code, ptr(err), ptr(run_if), ptr(ws), need, stream_ptr(q.device)),
            "ir_paged_attention_masked_ws")
        return out, ws[walks_at : walks_at + b * h_kv * blocks * 8].view(torch.int32).view(b, h_kv, blocks, 2).cpu()

    out, walks = call()
    want = torch.stack([torch.clamp((tiles + 5) // 6, max=parts), tiles], -1)
    want[1, 2, :, 0] *= -1  # parts < 0: a walk of all tiles
    assert torch.equal(walks, want.int())
    assert err.item() == 0
    dense = _masked_without_workspace(q, kc, vc, gs, mask)
    assert torch.equal(out.isnan(), dense.isnan())
    assert bool(out[1, :, nan_head].isnan().all()) and not out[[0, 2]].isnan().any()
    # (the bound of the test above: probabilities rounded against other running maxima)
    eps = torch.finfo(dtype).eps
    vmax = vc[vc.isfinite()].abs().max().item()
    assert torch.allclose(out.float(), dense.float(), rtol=eps, atol=eps * vmax, equal_nan=True)
    diff = (out.float().cpu() - ref).abs()
    diff[1, :, nan_head] = 0.0
    assert diff.max().item() <= TOL[dtype]
    if room == "full":
        got = kernels.paged_attention_masked(q, kc, vc, gs, mask, d**-0.5)
        assert torch.equal(got.nan_to_num(7.0), out.nan_to_num(7.0))
    gate = torch.ones(1, dtype=torch.int32, device=DEV)
    gated, gated_walks = call(gate)
    assert torch.equal(gated.nan_to_num(7.0), out.nan_to_num(7.0)) and torch.equal(gated_walks, walks)
    gate.zero_()
    untouched, _ = call(gate, torch.full_like(out, 3.0))
    assert bool((untouched == 3.0).all())


def test_config_table_is_consistent():
    for name, cfg in DECODE_CONFIGS.items():
        assert cfg.num_q_heads % cfg.num_kv_heads == 0, name
