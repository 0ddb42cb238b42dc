"""fp32 causal varlen prefill on the fp32 matrix cores (head_dim 64 and 128) against the oracle's
restatement of paged_attention (src/backend/cpu.rs:57-112): max-abs <= 1e-5 on fp32 output,
16-bit outputs exactly the round-to-nearest-even of the fp32 result, zero rows where a
sequence's kv length is below its query count, and the same bounds at the fp32 benchmark
batch's full size."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from _util import errors, f32_to_bf16_bits, to_np, with_kv_lens
from flour_amd import _lib, ops
from flour_amd.workloads import make_prefill, make_workload

pytestmark = pytest.mark.gpu


def _run(c, out_dtype=torch.float32, out=None):
    res = ops.varlen_prefill(c.q, c.k_pool, c.v_pool, c.cu_seqlens_q, c.kv_lens, c.block_tables,
                             c.max_seqlen_q, c.scale, block_size=c.block_size,
                             out_dtype=out_dtype, out=out)
    torch.cuda.synchronize()
    return res


def _oracle(c):
    return O.paged_attention(to_np(c.q), to_np(c.k_pool), to_np(c.v_pool), to_np(c.block_tables),
                             to_np(c.cu_seqlens_q), to_np(c.kv_lens), c.block_size, c.scale,
                             bf16=True)


def _case(H, G, D, bs, lens, prefix, seed):
    c = make_prefill(len(lens), H, G, D, bs, (1, 1), prefix=prefix, dtype=torch.float32,
                     seed=seed, device="cuda:0", q_lens=lens)
    ops.kv_write(c.k_new, c.v_new, c.k_pool, c.v_pool, c.slot_mapping)
    return c


@pytest.mark.parametrize("H,G,D,bs,lens,prefix", [
    (8, 8, 64, 16, [1, 17, 40, 300], 32),    # partial tiles, a cached prefix
    (16, 4, 128, 16, [129, 5], 0),            # GQA 4 at head_dim 128
    (14, 2, 64, 16, [300, 77, 1], 64),        # Qwen2.5-0.5B heads (GQA 7)
    (8, 2, 64, 7, [50, 33, 64], 14),          # 7-token pages: table lookups per position
    (4, 4, 128, 32, [32, 31, 33, 96], 0),     # tile edges
    (2, 1, 64, 16, [700], 0),                 # 22 tiles, the longest walking 22 steps
])
def test_prefill_f32_matrix_cores_match_oracle(device, H, G, D, bs, lens, prefix):
    c = _case(H, G, D, bs, lens, prefix, seed=H + D + bs)
    ref = _oracle(c)
    got = to_np(_run(c))
    max_abs, rel = errors(got, ref)
    print(f"fp32 mfma prefill H={H} G={G} D={D} bs={bs}: max_abs={max_abs:.3e} rel={rel:.3e}",
          flush=True)
    assert max_abs <= 1e-5


@pytest.fixture
def tiles():
    """fp32 prefill on the tile kernel, whatever the dispatch rule says for the batch."""
    assert _lib.lib().flour_hip_set_prefill_f32_mfma(3) == 0
    yield
    _lib.lib().flour_hip_set_prefill_f32_mfma(1)


@pytest.mark.parametrize("H,G,D,bs,lens,prefix,short", [
    (128, 128, 64, 16, [129, 1, 127, 260], 0, None),         # n_rep 1: 128-row items, their edges
    (128, 64, 128, 32, [64, 65, 1, 63, 200, 130], 32, 3),    # n_rep 2: 64-row items, 32-token pages
    (128, 32, 128, 16, [32, 33, 31, 1, 97, 330], 16, None),  # n_rep 4: 32-row items
    (112, 16, 64, 48, [300, 230, 2], 48, 1),                 # n_rep 7: a wave without a head
    (96, 32, 128, 16, [680, 100], 0, None),                  # n_rep 3: one head an item
    (64, 16, 64, 16, [17] * 64, 128, 40),                    # 64 sequences
])
def test_prefill_f32_tiles_match_oracle(device, tiles, H, G, D, bs, lens, prefix, short):
    """The tile kernel (larger batches): against the oracle, with rows past
    each sequence's positions holding garbage, a sequence whose kv length is below its query count,
    a bad block id past the used pages and 16-bit outputs."""
    c = make_prefill(len(lens), H, G, D, bs, (1, 1), prefix=prefix, dtype=torch.float32,
                     seed=H + D + bs, device="cuda:0", q_lens=lens)  # (every pool row is filled)
    used = torch.zeros(c.k_pool.shape[1], dtype=torch.bool)
    for s, n in enumerate(c.kv_lens.tolist()):
        j = torch.arange(n)
        used[c.block_tables[s].cpu()[j // bs].long() * bs + j % bs] = True
        c.block_tables[s, (n + bs - 1) // bs:] = -7
    c.k_pool[:, ~used.to(device)] = float("nan")
    c.v_pool[:, ~used.to(device)] = float("inf")
    if short is not None:
        c.kv_lens[short] = lens[short] - 1
    got = _run(c)
    max_abs, _ = errors(to_np(got), _oracle(c))
    print(f"fp32 tiles H={H} G={G} D={D}: max_abs={max_abs:.3e}", flush=True)
    assert max_abs <= 1e-5
    if short is not None:
        a, b = c.cu_seqlens_q[short:short + 2].tolist()
        assert not got[a:b].any()
    for dt in (torch.bfloat16, torch.float16):
        assert torch.equal(_run(c, dt), got.to(dt))


@pytest.mark.parametrize("H,G,D", [(8, 8, 64), (32, 16, 128), (14, 2, 64), (64, 16, 128)])
def test_prefill_f32_tiles_prefixes_of_every_length(device, tiles, H, G, D):
    """Sequences behind cached prefixes of their own lengths, far apart and none, in one batch: every
    tile of each once, against the oracle on every row."""
    lens = [33, 1, 300, 64, 0, 128, 40, 257, 16, 96]
    kv = [33, 4001, 300, 2064, 0, 128 + 31, 39, 257 + 640, 1016, 96 + 33]  # one below its rows
    c = with_kv_lens(make_prefill(len(lens), H, G, D, 16, (1, 1), dtype=torch.float32, seed=D + H,
                                  device="cuda:0", q_lens=lens), kv)
    out = torch.full_like(c.q, 7.0)
    _run(c, out=out)
    max_abs, _ = errors(to_np(out), _oracle(c))
    print(f"fp32 ragged prefixes H={H} G={G} D={D}: max_abs={max_abs:.3e}", flush=True)
    assert max_abs <= 1e-5


@pytest.mark.parametrize("bound", [700, 20000, 1 << 20])
def test_prefill_f32_tiles_with_a_loose_row_bound(device, tiles, bound):
    """max_seqlen_q is a bound: one far above the longest sequence changes nothing."""
    c = make_prefill(4, 64, 16, 128, 16, (1, 1), prefix=0, dtype=torch.float32, seed=98,
                     device="cuda:0", q_lens=[680, 600, 1, 300])
    tight = _run(c)
    c.max_seqlen_q = bound
    assert torch.equal(_run(c), tight)


@pytest.mark.parametrize("H,G,D,lens,width,tiled", [
    # block table width in positions (0: the longest sequence's)
    (32, 8, 128, [640] * 4, 0, True), (32, 8, 128, [632] * 4, 0, False),   # 2.5 items per CU
    (32, 8, 128, [64] * 40, 0, True), (32, 8, 128, [62] * 60, 0, False),   # 64 rows each
    (28, 4, 128, [1024] * 4, 0, True), (28, 4, 128, [1016] * 4, 0, False),  # a spare slot: 4 per CU
    (28, 4, 128, [128] * 32, 0, True), (28, 4, 128, [126] * 50, 0, False),  # and 128 rows each
    (16, 16, 128, [1024] * 8, 0, True), (16, 16, 128, [1016] * 8, 0, False),  # 128-row items
    (16, 16, 128, [640] * 13, 0, True), (16, 16, 128, [632] * 15, 0, False),  # and 640 rows each
    (32, 8, 128, [640] * 4, 1200, True), (32, 8, 128, [640] * 4, 1216, False),  # room for a prefix:
])                                                                       # 0.75 x 2.5 x 640 positions
def test_prefill_f32_tile_rule(device, H, G, D, lens, width, tiled):
    """Which fp32 batches run on the tile kernel, on both sides of every line of the rule, told by
    the bits of the output."""
    if torch.cuda.get_device_properties(device).multi_processor_count != 256:
        pytest.skip("the sizes are those of 256 CUs")
    c = make_prefill(len(lens), H, G, D, 16, (1, 1), dtype=torch.float32, seed=len(lens),
                     device="cuda:0", q_lens=lens)
    if width:
        c.block_tables = torch.nn.functional.pad(c.block_tables,
                                                 (0, width // 16 - c.block_tables.shape[1]))
    got = _run(c)
    outs = []
    try:
        for mode in (2, 3):
            assert _lib.lib().flour_hip_set_prefill_f32_mfma(mode) == 0
            outs.append(_run(c))
    finally:
        _lib.lib().flour_hip_set_prefill_f32_mfma(1)
    assert errors(to_np(outs[0]), to_np(outs[1]))[0] <= 2e-5
    assert torch.equal(got, outs[tiled]) and not torch.equal(got, outs[not tiled])


def test_prefill_f32_matches_the_vector_kernel(device):
    """The matrix-core and vector fp32 paths agree to the fp32 bound on the same batch."""
    c = _case(8, 2, 128, 16, [200, 31, 64], 16, seed=3)
    mfma = to_np(_run(c))
    assert _lib.lib().flour_hip_set_prefill_f32_mfma(0) == 0
    try:
        simt = to_np(_run(c))
    finally:
        _lib.lib().flour_hip_set_prefill_f32_mfma(1)
    assert errors(mfma, simt)[0] <= 1e-5


def test_prefill_f32_16bit_outputs_round_the_fp32_result(device):
    c = _case(8, 8, 64, 16, [90, 33, 1], 0, seed=11)
    got32 = to_np(_run(c))
    assert np.array_equal(to_np(_run(c, torch.bfloat16)), f32_to_bf16_bits(got32))
    assert np.array_equal(to_np(_run(c, torch.float16)), got32.astype(np.float16).view(np.uint16))


def test_prefill_f32_kv_shorter_than_q_gives_zero_rows(device):
    for D in (64, 128):
        c = _case(8, 2, D, 16, [40, 50, 200], 0, seed=29)
        c.kv_lens[1] = 49
        out = torch.full((c.q.shape[0], 8, D), 7.0, dtype=torch.float32, device=device)
        _run(c, out=out)
        got = to_np(out)
        assert np.array_equal(got[40:90], np.zeros_like(got[40:90])), D
        assert errors(got, _oracle(c))[0] <= 1e-5, D


def test_prefill_f32_strided_q_and_out(device):
    """q in the reference's head-major (H, seq, D) layout as a transposed view; strided out."""
    c = _case(8, 4, 64, 16, [150], 0, seed=8)
    q_hm = c.q.transpose(0, 1).contiguous()
    out_hm = torch.empty((8, 150, 64), dtype=torch.float32, device=device)
    ops.varlen_prefill(q_hm.transpose(0, 1), c.k_pool, c.v_pool, c.cu_seqlens_q, c.kv_lens,
                       c.block_tables, c.max_seqlen_q, c.scale, out_dtype=torch.float32,
                       out=out_hm.transpose(0, 1))
    torch.cuda.synchronize()
    assert torch.equal(out_hm.transpose(0, 1), _run(c))


def test_prefill_f32_benchmark_batch_full_size(device):
    c = make_workload("prefill_f32_h8_d64", device)
    ops.kv_write(c.k_new, c.v_new, c.k_pool, c.v_pool, c.slot_mapping)
    got = to_np(_run(c))
    max_abs, rel = errors(got, _oracle(c))
    print(f"prefill_f32_h8_d64: max_abs={max_abs:.3e} rel={rel:.3e}", flush=True)
    assert max_abs <= 1e-5
