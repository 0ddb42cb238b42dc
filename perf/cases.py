"""The calls whose speed this repository answers for, from the smallest decode step to long
prompts. Head counts and lengths are those of the repository's own workloads (Llama-3-8B and
-70B, Qwen2-7B and Qwen2.5-0.5B attention shapes, the fp32 shapes that a config.json without a
dtype leads to); block tables are random permutations of a pool that holds a quarter more blocks
than the batch needs, as a pool in service has them.

Four kinds of call:

  decode   one new token per sequence over its paged context (ops.paged_decode, or the prepared
           form that a serving loop keeps)
  prefill  packed prompts, or suffixes over a shared cached prefix, whose K/V rows are in the pool
           (ops.varlen_prefill)
  write    RoPE on a packed batch's q and k and the scatter of its K/V rows (ops.rope_kv_write)
  step     a continuous-batching step over a KvBatch: its plan, then per layer rope_write_kv and
           attention, with sequences that decode and prompts in one packed batch
"""
import math
import random

import torch

from flour_amd import ops
from flour_amd.kv_cache import KvBatch

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BS = 16  # tokens per page, the reference's block size


def listed():
    return [
        # a small fp32 model (the default dtype) serving four short chats: all latency
        dict(name="decode_f32_b4_h8_d64", kind="decode", dtype="f32", seqs=4, heads=8, kv_heads=8,
             dim=64, lo=1, hi=256, prepared=True),
        # a Llama-3-8B-sized model in fp32, a small batch of chats
        dict(name="decode_f32_b16_h32_d128", kind="decode", dtype="f32", seqs=16, heads=32,
             kv_heads=8, dim=128, lo=256, hi=2048, prepared=True),
        # one user's chat: the reference's engine decodes one sequence at a time
        dict(name="decode_bf16_b1_llama3_8b", kind="decode", dtype="bf16", seqs=1, heads=32,
             kv_heads=8, dim=128, lo=2000, hi=2000, prepared=True),
        # the headline batch
        dict(name="decode_bf16_b64_llama3_8b", kind="decode", dtype="bf16", seqs=64, heads=32,
             kv_heads=8, dim=128, lo=512, hi=4096, prepared=False),
        # long documents
        dict(name="decode_bf16_long_llama3_70b", kind="decode", dtype="bf16", seqs=8, heads=64,
             kv_heads=8, dim=128, lo=16384, hi=32768, prepared=False),
        # a small model's batch: head_dim 64, seven query heads per kv head
        dict(name="decode_bf16_b64_qwen25_05b", kind="decode", dtype="bf16", seqs=64, heads=14,
             kv_heads=2, dim=64, lo=512, hi=4096, prepared=True),
        # one prompt of the reference's load test (up to 1,024 tokens to Qwen2.5-0.5B)
        dict(name="prefill_bf16_one_qwen25_05b", kind="prefill", dtype="bf16", seqs=1, heads=14,
             kv_heads=2, dim=64, lo=1000, hi=1000, prefix=0),
        # a batch of prompts of mixed lengths
        dict(name="prefill_bf16_varlen_llama3_8b", kind="prefill", dtype="bf16", seqs=8, heads=32,
             kv_heads=8, dim=128, lo=256, hi=2048, prefix=0),
        # user turns over one cached system prompt
        dict(name="prefill_bf16_prefix_qwen2_7b", kind="prefill", dtype="bf16", seqs=16, heads=28,
             kv_heads=4, dim=128, lo=128, hi=512, prefix=1024),
        # two long documents
        dict(name="prefill_bf16_long_llama3_8b", kind="prefill", dtype="bf16", seqs=2, heads=32,
             kv_heads=8, dim=128, lo=8192, hi=8192, prefix=0),
        # prompts to a Llama-3-8B-sized model in fp32
        dict(name="prefill_f32_h32_d128", kind="prefill", dtype="f32", seqs=8, heads=32,
             kv_heads=8, dim=128, lo=256, hi=1024, prefix=0),
        # a mixed continuous-batching step of two layers: chats that decode beside new prompts
        dict(name="step_bf16_mixed_llama3_8b", kind="step", dtype="bf16", seqs=16, prompts=3,
             heads=32, kv_heads=8, dim=128, lo=256, hi=2048, plo=64, phi=512, layers=2),
    ]


HEADS = [(8, 8, 64), (14, 2, 64), (32, 32, 64), (28, 4, 128), (32, 8, 128), (64, 8, 128),
         (16, 16, 128)]  # (query heads, kv heads, head_dim)


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        heads, kv_heads, dim = rng.choice(HEADS)
        c = dict(kind=rng.choice(["decode", "decode", "prefill", "prefill", "write", "step"]),
                 dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), heads=heads,
                 kv_heads=kv_heads, dim=dim)
        if c["kind"] == "decode":
            c["seqs"] = _log(rng, 1, 256)
            c["hi"] = _log(rng, 16, 32768)
            c["lo"] = max(1, int(c["hi"] * rng.choice([0.02, 0.125, 0.5, 1.0])))
            c["prepared"] = rng.random() < 0.5
            ok = 2e5 < work(c)["bytes"] < 8e8
        elif c["kind"] == "prefill":
            c["seqs"] = _log(rng, 1, 32)
            c["hi"] = _log(rng, 16, 8192)
            c["lo"] = max(1, int(c["hi"] * rng.choice([0.125, 0.5, 1.0])))
            c["prefix"] = rng.choice([0, 0, BS * _log(rng, 1, 128)])
            ok = 1e8 < work(c)["flops"] < (2e10 if c["dtype"] == "f32" else 5e11)
        elif c["kind"] == "write":
            c["seqs"] = _log(rng, 1, 16)
            c["hi"] = _log(rng, 16, 4096)
            c["lo"] = max(1, c["hi"] // 8)
            ok = 1e6 < work(c)["bytes"] < 5e8
        else:
            if c["dtype"] == "f32":
                continue
            c.update(seqs=_log(rng, 1, 48), prompts=rng.choice([0, 1, 2, 4]), lo=64,
                     hi=_log(rng, 128, 4096), plo=16, phi=_log(rng, 32, 1024), layers=2)
            w = work(c)
            ok = 1e6 < w["bytes"] < 4e8 and w["flops"] < 1e11
        if ok:
            return c


# ------------------------------------------------------------------ sizes and inputs
def _lens(case):
    """The lengths of a case's sequences (context, prompt or suffix lengths)."""
    rng = random.Random(1000003 * case["seqs"] + 1009 * case["hi"] + case["lo"])
    return [rng.randint(case["lo"], case["hi"]) for _ in range(case["seqs"])]


def _prompt_lens(case):
    rng = random.Random(7919 * case["prompts"] + 31 * case["phi"] + case["plo"])
    return [rng.randint(case["plo"], case["phi"]) for _ in range(case["prompts"])]


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _outlier_channels(k, seed):
    """Scales one in 500 of the (kv head, dim) channels of k (..., heads, dim), as the K
    projections of trained models have them; some never do."""
    rng = random.Random(seed)
    heads, dim = k.shape[-2], k.shape[-1]
    for _ in range(max(1, heads * dim // 500)):
        k[..., rng.randrange(heads), rng.randrange(dim)] *= 6.0
    return k


def _tables(lens, shared, seed):
    """Block tables of sequences of `lens` positions whose first `shared` blocks are the same
    physical blocks: (table as a CPU tensor, blocks in the pool)."""
    own = [(n + BS - 1) // BS - shared for n in lens]
    need = shared + sum(own)
    total = need + (need + 3) // 4
    perm = list(range(total))
    random.Random(seed).shuffle(perm)
    table = torch.zeros((len(lens), shared + max(own)), dtype=torch.int32)
    at = shared
    for s, n in enumerate(own):
        table[s, :shared] = torch.tensor(perm[:shared], dtype=torch.int32)
        table[s, shared:shared + n] = torch.tensor(perm[at:at + n], dtype=torch.int32)
        at += n
    return table, total


def _pools(case, blocks, seed):
    g, dt = _generator(seed + 1), DTYPES[case["dtype"]]
    shape = (blocks * BS, case["kv_heads"], case["dim"])
    k = _outlier_channels(_randn(g, shape, torch.float32), seed).to(dt)
    v = _randn(g, shape, dt)
    return k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous()


def _rope_tables(positions, dim, dtype):
    """cos and sin of pos / 10000^(2 i / dim), (positions, dim / 2)."""
    i = torch.arange(dim // 2, dtype=torch.float64)
    ang = torch.arange(positions, dtype=torch.float64)[:, None] * 10000.0 ** (-2 * i / dim)
    return ang.cos().to(dtype).cuda(), ang.sin().to(dtype).cuda()


def _inputs(case, seed):
    """The tensors of a decode, prefill or write call."""
    dt, lens = DTYPES[case["dtype"]], _lens(case)
    g = _generator(seed)
    if case["kind"] == "decode":
        table, blocks = _tables(lens, 0, seed)
        k, v = _pools(case, blocks, seed)
        return dict(q=_randn(g, (len(lens), case["heads"], case["dim"]), dt), k=k, v=v,
                    table=table.cuda(), kv=lens)
    if case["kind"] == "prefill":
        kv = [n + case["prefix"] for n in lens]
        table, blocks = _tables(kv, case["prefix"] // BS, seed)
        k, v = _pools(case, blocks, seed)
        return dict(q=_randn(g, (sum(lens), case["heads"], case["dim"]), dt), k=k, v=v,
                    table=table.cuda(), kv=kv)
    table, blocks = _tables(lens, 0, seed)
    rows = sum(lens)
    pos = torch.cat([torch.arange(n) for n in lens])
    seq = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens))
    slots = table[seq, pos // BS] * BS + pos % BS
    cos, sin = _rope_tables(max(lens), case["dim"], dt)
    return dict(q=_randn(g, (rows, case["heads"], case["dim"]), dt),
                k=_randn(g, (rows, case["kv_heads"], case["dim"]), dt),
                v=_randn(g, (rows, case["kv_heads"], case["dim"]), dt), slots=slots, pos=pos,
                num_slots=blocks * BS, cos=cos, sin=sin)


def _step_inputs(case, seed):
    """Per layer the contexts' K/V by sequence and the new rows' q, k, v, packed."""
    dt, lens, plens = DTYPES[case["dtype"]], _lens(case), _prompt_lens(case)
    g = _generator(seed)
    rows = len(lens) + sum(plens)
    H, G, D = case["heads"], case["kv_heads"], case["dim"]
    layers = [dict(ctx=[(_randn(g, (n, G, D), dt), _randn(g, (n, G, D), dt)) for n in lens],
                   q=_randn(g, (rows, H, D), dt), k=_randn(g, (rows, G, D), dt),
                   v=_randn(g, (rows, G, D), dt)) for _ in range(case["layers"])]
    cos, sin = _rope_tables(max([n + 1 for n in lens] + plens), D, dt)
    return layers, cos, sin, lens, plens


# ------------------------------------------------------------------ the calls
def prepare(case, seed):
    if case["kind"] == "step":
        return _prepare_step(case, seed)
    x = _inputs(case, seed)
    lens, scale = _lens(case), 1.0 / math.sqrt(case["dim"])
    st = dict(case=case, scale=scale, **x)
    if case["kind"] == "write":
        shape = (case["kv_heads"], x["num_slots"], case["dim"])
        st["k_pool"] = torch.zeros(shape, dtype=x["k"].dtype, device="cuda")
        st["v_pool"] = torch.zeros(shape, dtype=x["k"].dtype, device="cuda")
        st["slots"] = x["slots"].to(torch.int32).cuda()
        st["pos"] = x["pos"].to(torch.int32).cuda()
        st["q_out"] = torch.empty_like(x["q"])
        return st
    st["kv_lens"] = torch.tensor(x["kv"], dtype=torch.int32, device="cuda")
    st["workspace"] = ops.Workspace()
    if case["kind"] == "prefill":
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        st["cu"] = torch.tensor(cu, dtype=torch.int32, device="cuda")
    elif case["prepared"]:
        st["out"] = torch.empty_like(x["q"])
        st["step"] = ops.prepare_paged_decode(x["q"], x["k"], x["v"], x["table"], st["kv_lens"],
                                              scale, max(lens), st["out"], st["workspace"])
    return st


def _prepare_step(case, seed):
    layers, cos, sin, lens, plens = _step_inputs(case, seed)
    total = [n + 1 for n in lens] + plens
    blocks = sum((n + BS - 1) // BS for n in total) + 8
    batch = KvBatch(case["layers"], blocks, len(total), max(total),
                    max(max(lens), len(lens) + sum(plens)), case["heads"], case["kv_heads"],
                    case["dim"], dtype=DTYPES[case["dtype"]])
    ids = [batch.add_sequence() for _ in total]
    for i, n in enumerate(lens):  # the contexts as earlier steps left them
        batch.step([ids[i]], [n])
        for j, la in enumerate(layers):
            batch.write_kv(j, *la["ctx"][i])
    new = [1] * len(lens) + plens
    for i, n in zip(ids, new):
        batch.allocate_kv(i, n)
    for la in layers:
        del la["ctx"]
    torch.cuda.synchronize()
    pools = [t for j in range(case["layers"]) for t in batch.pool(j)]
    for t in pools:  # views of memory that the batch frees with itself: each keeps it alive
        t.owner = batch
    return dict(case=case, batch=batch, ids=ids, new=new, layers=layers, cos=cos, sin=sin,
                scale=1.0 / math.sqrt(case["dim"]), pools=pools)


def run(st):
    case = st["case"]
    if case["kind"] == "decode":
        if case["prepared"]:
            st["step"]()
            return st["out"]
        return ops.paged_decode(st["q"], st["k"], st["v"], st["table"], st["kv_lens"],
                                st["scale"], max(st["kv"]), workspace=st["workspace"])
    if case["kind"] == "prefill":
        return ops.varlen_prefill(st["q"], st["k"], st["v"], st["cu"], st["kv_lens"],
                                  st["table"], max(_lens(case)), st["scale"],
                                  workspace=st["workspace"])
    if case["kind"] == "write":
        ops.rope_kv_write(st["q"], st["k"], st["v"], st["k_pool"], st["v_pool"], st["slots"],
                          st["pos"], st["cos"], st["sin"], q_out=st["q_out"])
        return [st["q_out"], st["k_pool"], st["v_pool"]]
    st["batch"].plan(st["ids"], st["new"])
    outs = []
    for j, la in enumerate(st["layers"]):
        q = st["batch"].rope_write_kv(j, la["q"], la["k"], la["v"], st["cos"], st["sin"])
        outs += [q, st["batch"].attention(j, q, st["scale"])]
    return outs + st["pools"]


# ------------------------------------------------------------------ what a call cannot do without
def work(case):
    e = 4 if case["dtype"] == "f32" else 2
    H, G, D, lens = case["heads"], case["kv_heads"], case["dim"], _lens(case)
    if case["kind"] == "decode":
        n = sum(lens)
        return dict(bytes=2 * n * G * D * e + 2 * len(lens) * H * D * e + 4 * (n // BS),
                    flops=4 * n * H * D)
    if case["kind"] == "prefill":
        p, rows = case["prefix"], sum(lens)
        pairs = sum(n * p + n * (n + 1) // 2 for n in lens)
        return dict(bytes=2 * (rows + p) * G * D * e + 2 * rows * H * D * e,
                    flops=4 * pairs * H * D)
    if case["kind"] == "write":
        rows = sum(lens)
        return dict(bytes=2 * rows * (H + 2 * G) * D * e + max(lens) * D * e + 8 * rows,
                    flops=3 * rows * (H + G) * D)
    plens = _prompt_lens(case)
    rows = len(lens) + sum(plens)
    pairs = sum(n + 1 for n in lens) + sum(n * (n + 1) // 2 for n in plens)
    # per layer: q read and rotated, k and v read and written, contexts read, rows' output
    return dict(bytes=case["layers"] * e * D * (rows * (3 * H + 4 * G) + 2 * G * sum(lens)),
                flops=case["layers"] * (4 * pairs * H * D + 3 * rows * (H + G) * D))


def tolerance(case):
    # four times the distance from 64 bits: fp32 sums over at most some thousand positions (1.5e-7
    # to 3.3e-7), or the rounding of the output to 16 bits (1.7e-3, 2.9e-4), which a step does
    # for the rotated q and k too (3.1e-3)
    if case["dtype"] == "f32":
        return {"rel": 1.5e-6}
    return {"rel": {"bf16": 7e-3, "f16": 1.2e-3}[case["dtype"]] *
            (2 if case["kind"] == "step" else 1)}


# ------------------------------------------------------------------ 64-bit results
def _attend(q, k, v, scale):
    """Causal attention of the last rows of a sequence: q (rows, H, D), k / v (kv, G, D)."""
    rows, H, D = q.shape
    kv, G = k.shape[0], k.shape[1]
    hide = (torch.arange(kv, device="cuda")[None, :] >
            torch.arange(kv - rows, kv, device="cuda")[:, None])
    out = torch.empty((rows, H, D), dtype=torch.float64, device="cuda")
    for h in range(H):
        kh, vh = k[:, h // (H // G)].double(), v[:, h // (H // G)].double()
        s = torch.mm(q[:, h].double(), kh.t().contiguous()) * scale
        out[:, h] = torch.mm(torch.softmax(s.masked_fill_(hide, float("-inf")), dim=-1), vh)
    return out


def _rope(x, cos, sin):
    """Rotate-half RoPE of x (rows, heads, dim), cos / sin (rows, dim / 2)."""
    h = x.shape[-1] // 2
    x, c, s = x.double(), cos.double()[:, None, :], sin.double()[:, None, :]
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * c - b * s, a * s + b * c], dim=-1)


def exact(case, seed):
    scale = 1.0 / math.sqrt(case["dim"])
    if case["kind"] == "step":
        layers, cos, sin, lens, plens = _step_inputs(case, seed)
        pos = torch.tensor(lens + [i for n in plens for i in range(n)], device="cuda")
        outs = []
        for la in layers:
            q, k = (_rope(la[x], cos[pos], sin[pos]) for x in ("q", "k"))
            o, at = torch.empty_like(q), 0
            for i, n in enumerate([1] * len(lens) + plens):
                kk, vv = k[at:at + n], la["v"][at:at + n].double()
                if i < len(lens):
                    kk = torch.cat([la["ctx"][i][0].double(), kk])
                    vv = torch.cat([la["ctx"][i][1].double(), vv])
                o[at:at + n] = _attend(q[at:at + n], kk, vv, scale)
                at += n
            outs += [q, o]
        return outs + [None] * (2 * case["layers"])
    x = _inputs(case, seed)
    if case["kind"] == "write":
        cos, sin = x["cos"][x["pos"].cuda()], x["sin"][x["pos"].cuda()]
        pools = []
        for rows in (_rope(x["k"], cos, sin), x["v"].double()):
            p = torch.zeros((case["kv_heads"], x["num_slots"], case["dim"]), dtype=torch.float64,
                            device="cuda")
            p[:, x["slots"].long().cuda()] = rows.transpose(0, 1)
            pools.append(p)
        return [_rope(x["q"], cos, sin)] + pools
    out = torch.empty(x["q"].shape, dtype=torch.float64, device="cuda")
    new = _lens(case) if case["kind"] == "prefill" else [1] * len(x["kv"])
    at = 0
    for s, (n, kv) in enumerate(zip(new, x["kv"])):
        j = torch.arange(kv, device="cuda")
        slots = x["table"][s, j // BS].long() * BS + j % BS
        out[at:at + n] = _attend(x["q"][at:at + n], x["k"][:, slots].transpose(0, 1),
                                 x["v"][:, slots].transpose(0, 1), scale)
        at += n
    return out
