"""Causal varlen prefill at head_dim 64 on the matrix-core kernels (the Qwen2.5-0.5B attention
shape the reference serves: 14 q / 2 kv heads, GQA 7, src/models/qwen2.rs:39 with
script/script.js:14), against the oracle's restatement of paged_attention (cpu.rs:57-112).

Two kernels serve it: the large one (varlen_prefill.hip) and the one for small batches
(prefill_thin.hip, with two or four slots an item). Every case that is small enough for either
runs on all three forms, whatever the dispatch rule says for its size (`kernel`).

Bounds as for head_dim 128: the fp32 accumulator output within max-abs 2e-3 and rel-L2 1e-3 of
the fp32 oracle, the bf16 output within the ulp bounds of tests/_util.py. Covered: GQA 7, a
cached prefix shared by every sequence, partial last query tiles (the large kernel's 4 x 64 and 8 x
32 item shapes and the one-head 256-row items of an odd group), page sizes 16, 32 and 48, kv_len <
q_len, the persistent schedule against one workgroup per item, V outside the fp16 range (the large
kernel's exact redo), the hi + lo P mode and the whole benchmark batch.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import PREFILL_ULP_BOUNDS, check_bf16_output, errors, to_np, with_kv_lens
from flour_amd import _lib, ops
from flour_amd.workloads import make_prefill, make_workload
from test_prefill_gpu import oracle_prefill, run, write

pytestmark = pytest.mark.gpu

D = 64


@pytest.fixture(params=[0, 2, 4], ids=["large", "two-slot", "four-slot"])
def kernel(request):
    """The kernel form that the test's calls run on."""
    assert _lib.lib().flour_hip_set_prefill_small(request.param) == 0
    yield request.param
    _lib.lib().flour_hip_set_prefill_small(1)


def check(c, seqs=None, tag=""):
    ref, rows = oracle_prefill(c, seqs)
    got32 = to_np(run(c, torch.float32))[rows]
    max_abs, rel = errors(got32, ref)
    print(f"{tag} fp32-out max_abs={max_abs:.3e} rel_l2={rel:.3e}", flush=True)
    assert max_abs <= 2e-3 and rel <= 1e-3
    if c.q.dtype == torch.bfloat16:
        rep = check_bf16_output(to_np(run(c, torch.bfloat16))[rows], got32, ref,
                                PREFILL_ULP_BOUNDS)
        print(f"{tag} bf16-out {rep}", flush=True)
    return got32


def go(c, persistent=1, out_dtype=torch.float32):
    H = c.q.shape[1]
    out = torch.full((c.q.shape[0], H, D), 7.0, dtype=out_dtype, device=c.q.device)
    _lib.lib().flour_hip_set_prefill_persistent(persistent)
    try:
        ops.varlen_prefill(c.q, c.k_pool, c.v_pool, c.cu_seqlens_q, c.kv_lens, c.block_tables,
                           c.max_seqlen_q, c.scale, block_size=c.block_size, out_dtype=out_dtype,
                           out=out)
        torch.cuda.synchronize()
    finally:
        _lib.lib().flour_hip_set_prefill_persistent(1)
    return out


@pytest.mark.parametrize("H,G,bs,lens,prefix", [
    (14, 2, 16, [300, 77, 1], 64),          # Qwen2.5-0.5B heads over a cached prefix
    (14, 2, 32, [129, 33, 64, 200], 32),    # 32-token pages
    (8, 2, 16, [1, 2, 31, 32, 33], 0),      # one-row and one-tile sequences
    (16, 16, 16, [257, 5], 48),             # n_rep 1
    (8, 1, 16, [1, 200], 160),              # n_rep 8
    (14, 2, 48, [150, 96], 96),             # 48-token pages
])
def test_prefill_d64_shapes(device, kernel, H, G, bs, lens, prefix):
    c = make_prefill(len(lens), H, G, D, bs, (1, 1), prefix=prefix, dtype=torch.bfloat16,
                     seed=H * 5 + G + bs, device=device, q_lens=lens)
    write(c)
    check(c, tag=f"D64 H={H} G={G} bs={bs} lens={lens} prefix={prefix}")


def test_prefill_d64_f16_pools(device, kernel):
    c = make_prefill(3, 14, 2, D, 16, (1, 1), prefix=32, dtype=torch.float16, seed=61,
                     device=device, q_lens=[200, 64, 9])
    write(c)
    check(c, tag="D64 f16")


def test_prefill_qwen25_05b_workload(device):
    """The head_dim-64 benchmark batch (8 prompts of U[256, 1024] rows, 14 / 2 heads): every
    row of every sequence against the oracle."""
    c = make_workload("prefill_bf16_qwen25_05b", device=device)
    write(c)
    lens = (c.cu_seqlens_q[1:] - c.cu_seqlens_q[:-1]).tolist()
    print(f"lens={lens}", flush=True)
    check(c, tag="qwen2.5-0.5b prefill (whole batch)")


@pytest.mark.parametrize("H,G", [(14, 2), (16, 4), (10, 2)])
def test_prefill_d64_persistent_and_partial_tiles(device, H, G):
    """Persistent schedule with the partial-last-tile item shapes (4 heads x 64 rows, 8 heads x
    32 rows, one-head 256-row items of odd groups 7 and 5) bit-identical to one workgroup per
    item, empty sequences and a sequence with kv_len < q_len (zero rows) included."""
    rng = np.random.default_rng(H * 7 + G)
    lens = []
    for i in range(30):
        full = int(rng.integers(0, 4)) * 128
        tail = [int(rng.integers(1, 33)), int(rng.integers(33, 65)), int(rng.integers(65, 129))][i % 3]
        lens.append(full + tail)
    lens[4] = 0
    c = make_prefill(len(lens), H, G, D, 16, (1, 1), prefix=64, dtype=torch.bfloat16,
                     seed=70 + H, device=device, q_lens=lens)
    write(c)
    c.kv_lens[9] = lens[9] - 1  # kv_len < q_len: the sequence attends nothing
    a, b = go(c, 1), go(c, 0)
    assert torch.equal(a, b)
    cu = to_np(c.cu_seqlens_q)
    assert bool((a[int(cu[9]):int(cu[10])] == 0.0).all())
    ref, rows = oracle_prefill(c, seqs=[0, 1, 2, 29])
    max_abs, rel = errors(to_np(a)[rows], ref)
    print(f"D64 persistent H={H} G={G}: max_abs={max_abs:.3e} rel_l2={rel:.3e}", flush=True)
    assert max_abs <= 2e-3 and rel <= 1e-3


def test_prefill_d64_v_outside_fp16_range(device, kernel):
    """V rows of +-1e5 and 1e-30 among N(0,1) rows: the large kernel recomputes the items that meet
    them in exact mode (bf16 V, P split in two), the small-batch kernel always keeps V in bf16 and P
    in two parts; judged against the output's own scale."""
    c = make_prefill(4, 14, 2, D, 16, (1, 1), prefix=32, dtype=torch.bfloat16, seed=81,
                     device=device, q_lens=[150, 40, 260, 7])
    c.v_new[10:14] *= 1e5
    c.v_new[100:103] *= 1e-30
    write(c)
    ref, rows = oracle_prefill(c)
    got = to_np(run(c, torch.float32))[rows]
    assert np.isfinite(got).all()
    scale = np.abs(ref).max(axis=-1, keepdims=True) + 1e-30
    err = np.abs(got - ref) / scale
    print(f"D64 V out of range: max rel-to-row-scale err={err.max():.3e}", flush=True)
    assert err.max() <= 2e-3


def test_prefill_d64_hilo_mode(device):
    c = make_prefill(3, 14, 2, D, 16, (1, 1), prefix=16, dtype=torch.bfloat16, seed=91,
                     device=device, q_lens=[333, 70, 1])
    write(c)
    assert _lib.lib().flour_hip_set_prefill_precise_p(1) == 0
    try:
        got = check(c, tag="D64 hi+lo P")
    finally:
        _lib.lib().flour_hip_set_prefill_precise_p(0)
    assert np.isfinite(got).all()


def test_prefill_d64_reference_layout(device, kernel):
    """q in the reference's head-major (1, heads, seq, D) layout and out written straight into
    (seq, heads, D): strided views on both sides."""
    c = make_prefill(1, 14, 2, D, 16, (1, 1), prefix=0, dtype=torch.bfloat16, seed=95,
                     device=device, q_lens=[190])
    write(c)
    q_hm = c.q.transpose(0, 1).contiguous()          # (heads, seq, D)
    q_view = q_hm.transpose(0, 1)                    # (seq, heads, D), strides (D, seq*D, 1)
    out = ops.varlen_prefill(q_view, c.k_pool, c.v_pool, c.cu_seqlens_q, c.kv_lens,
                             c.block_tables, c.max_seqlen_q, c.scale, out_dtype=torch.float32)
    torch.cuda.synchronize()
    ref, rows = oracle_prefill(c)
    max_abs, rel = errors(to_np(out)[rows], ref)
    assert max_abs <= 2e-3 and rel <= 1e-3


@pytest.mark.parametrize("H,G,bs,lens,prefix,short", [
    (14, 2, 16, [1000], 0, None),                     # one prompt, GQA 7
    (14, 2, 16, [511, 130, 64, 33, 1, 385, 500, 480], 0, 3),  # row and step edges
    (8, 8, 32, [129, 128, 1, 65], 32, None),          # one head an item, 32-token pages
    (6, 2, 48, [200, 31], 96, 1),                     # n_rep 3, 48-token pages
    (16, 1, 16, [40] * 64, 256, 7),                   # n_rep 16, 64 sequences
    (4, 2, 32, [1, 63, 64, 65, 129], 0, 2),           # n_rep 2: both heads, one or two row blocks
    (12, 2, 16, [300], 1008, None),                   # n_rep 6, a prefix that ends inside a step
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_small_batches(device, kernel, dtype, H, G, bs, lens, prefix, short):
    """Batches of the small-batch kernel's sizes on each form: against the oracle, with garbage in
    every row past the sequences' positions, bad block ids past the used pages, a sequence whose kv
    length is below its query count, and both schedules alike."""
    c = make_prefill(len(lens), H, G, D, bs, (1, 1), prefix=prefix, dtype=dtype, seed=H + bs,
                     device=device, q_lens=lens)  # (every pool row is filled)
    used = torch.zeros(c.k_pool.shape[1], dtype=torch.bool)
    for s, n in enumerate(c.kv_lens.tolist()):
        j = torch.arange(n)
        used[c.block_tables[s].cpu()[j // bs].long() * bs + j % bs] = True
        c.block_tables[s, (n + bs - 1) // bs:] = -7
    c.k_pool[:, ~used.to(device)] = float("nan")
    c.v_pool[:, ~used.to(device)] = float("inf")
    if short is not None:
        c.kv_lens[short] = lens[short] - 1
    got = go(c)
    ref, rows = oracle_prefill(c, None)
    max_abs, rel = errors(to_np(got)[rows], ref)
    print(f"small batch H={H} G={G} {dtype}: max_abs={max_abs:.3e} rel_l2={rel:.3e}", flush=True)
    assert max_abs <= 2e-3 and rel <= 1e-3
    if short is not None:
        a, b = c.cu_seqlens_q[short:short + 2].tolist()
        assert not got[a:b].any()
    assert torch.equal(got, go(c, persistent=0))
    assert torch.equal(go(c, out_dtype=dtype), got.to(dtype))


@pytest.mark.parametrize("bound", [1000, 1024, 40000, 65536])
def test_small_batch_with_a_loose_row_bound(device, kernel, bound):
    """max_seqlen_q is a bound: one far above the longest sequence changes nothing."""
    c = make_prefill(3, 14, 2, D, 16, (1, 1), prefix=32, dtype=torch.bfloat16, seed=97,
                     device=device, q_lens=[400, 64, 9])
    tight = go(c)
    c.max_seqlen_q = bound
    assert torch.equal(go(c), tight)


@pytest.mark.parametrize("H,G,lens,prefix,slots", [
    (14, 2, [31 * 32], 0, 2), (14, 2, [31 * 32], 4096, 2),  # 256 items with two slots each: one a CU
    (14, 2, [32 * 32], 4096, 4),                            # 264 and 132: four slots
    (14, 2, [63 * 32], 4096, 4), (14, 2, [64 * 32], 4096, 0),      # up to one a CU
    (14, 2, [32 * 32], 0, 2), (14, 2, [63 * 32], 0, 2),     # one prompt without a prefix: two slots
    (14, 2, [64 * 32], 0, 4), (14, 2, [95 * 32], 0, 4),     # there, four up to one and a half
    (14, 2, [96 * 32], 0, 0),
    (8, 8, [64 * 7] * 4, 0, 2), (8, 8, [64 * 8] * 4, 0, 4),      # one head an item
    (32, 8, [32 * 3] * 8, 0, 4), (32, 8, [32 * 3 + 4] * 8, 0, 0),
    (2, 2, [20] * 64, 256, 2), (2, 2, [20] * 65, 256, 0),   # up to 64 sequences
])
def test_small_batch_rule(device, H, G, lens, prefix, slots):
    """Which batches run on the small-batch kernel and with how many slots, on both sides of every
    line of the rule, told by the bits of the output."""
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    if cus != 256:
        pytest.skip("the sizes are those of 256 CUs")
    c = make_prefill(len(lens), H, G, D, 16, (1, 1), prefix=prefix, dtype=torch.bfloat16,
                     seed=len(lens), device=device, q_lens=lens)
    got = go(c)
    lib = _lib.lib()
    same = []
    try:
        for mode in (0, 2, 4):
            lib.flour_hip_set_prefill_small(mode)
            out = go(c)
            assert errors(to_np(out), to_np(got))[1] <= 1e-3
            if torch.equal(out, got):
                same.append(mode)
    finally:
        lib.flour_hip_set_prefill_small(1)
    assert same == [slots] if len(lens) <= 64 else slots in same


def test_prefixes_of_every_length(device, kernel):
    """Sequences behind cached prefixes of their own lengths, far apart and none, in one batch: every
    tile of each once, on every row, in both schedules."""
    lens = [33, 1, 300, 64, 0, 128, 40, 257, 16, 96]
    kv = [33, 4001, 300, 2064, 0, 128 + 31, 39, 257 + 640, 1016, 96 + 33]  # one below its rows
    c = with_kv_lens(make_prefill(len(lens), 14, 2, D, 16, (1, 1), dtype=torch.bfloat16, seed=99,
                                  device=device, q_lens=lens), kv)
    got = go(c)
    ref, rows = oracle_prefill(c)
    max_abs, rel = errors(to_np(got)[rows], ref)
    print(f"D64 ragged prefixes: max_abs={max_abs:.3e} rel_l2={rel:.3e}", flush=True)
    assert max_abs <= 2e-3 and rel <= 1e-3
    assert torch.equal(got, go(c, persistent=0))
