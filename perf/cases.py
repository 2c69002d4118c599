"""The work a user of this framework has it do, as timed cases.

A serving program calls the package per layer and per step: paged decode
attention (one query token per sequence), the same fused with the step's KV
append, paged prefill attention of one chunk, a transformer block's decode
step, and a whole model's decode step. The cases cover those calls from the
smallest model and batch the repository is tested with to its largest
benchmark shapes, in the three data types, with ragged lengths and odd sizes.

  listed()  the named cases;  draw(rng)  another case of the same ranges;
  prepare(case, seed)  what a program holds before the call, on the GPU;
  run(state)  one pass;  exact(case, seed)  the same outputs in 64 bits;
  work(case), tolerance(case)  what a pass cannot do without, and how far two
  correct implementations may differ.
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-gpt-inference_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from minivllm import hip_paged_decode as hpd  # noqa: E402
from minivllm.block import TransformerBlock  # noqa: E402
from minivllm.decode_batch_metadata import DecodeBatchMetadata  # noqa: E402
from minivllm.kv_block_pool import KVBlockPool  # noqa: E402
from minivllm.model import MiniGPT  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
EB = {"f32": 4, "bf16": 2, "f16": 2}


def _decode(name, kind, B, H, D, S, lo, hi, dtype, lens):
    return {"name": name, "kind": kind, "B": B, "H": H, "D": D, "S": S, "ctx_lo": lo, "ctx_hi": hi, "dtype": dtype,
            "lens": lens}


def listed():
    return [
        # One layer of the small fp32 model (8 heads of 32) that the runtime A/B benchmark serves, four
        # requests deep into their prompts: the shortest useful call, where launches and latency count.
        _decode("decode_small_model", "decode", 4, 8, 32, 16, 200, 256, "f32", 1),
        # A chat server at light load: 13 conversations of mixed length, the step's KV append included.
        _decode("append_decode_chat", "append", 13, 16, 128, 16, 100, 1000, "bf16", 2),
        # The benchmark's headline shape: 64 ragged sequences, 32 heads.
        _decode("decode_headline", "decode", 64, 32, 128, 16, 512, 4096, "bf16", 3),
        # One GPU's share of the same shape split 8 ways over heads, in f16.
        _decode("decode_head_share", "decode", 64, 4, 128, 16, 512, 4096, "f16", 4),
        # Long documents: 8 sequences of 32k to 128k tokens.
        _decode("decode_long", "decode", 8, 32, 128, 16, 32768, 131072, "bf16", 5),
        # A full batch: 256 sequences of 128 to 2048 tokens, append and attention in one call.
        _decode("append_decode_b256", "append", 256, 32, 128, 16, 128, 2048, "bf16", 6),
        # The first chunk of a typical prompt.
        {"name": "prefill_first", "kind": "prefill", "T": 512, "start": 0, "H": 16, "D": 128, "S": 16, "dtype": "bf16"},
        # A full-budget chunk in the middle of a long prompt.
        {"name": "prefill_middle", "kind": "prefill", "T": 2048, "start": 2048, "H": 16, "D": 128, "S": 16,
         "dtype": "bf16"},
        # The short last chunk of a long prompt, or a new turn after a cached conversation.
        {"name": "prefill_tail", "kind": "prefill", "T": 203, "start": 6000, "H": 16, "D": 128, "S": 16,
         "dtype": "bf16"},
        # A chunk of an fp32 model, ragged on both ends.
        {"name": "prefill_f32", "kind": "prefill", "T": 700, "start": 450, "H": 8, "D": 64, "S": 16, "dtype": "f32"},
        # One transformer block of the benchmark model (dim 2048) on a decode batch: norms, projections,
        # append, attention, MLP.
        {"name": "block_decode", "kind": "block", "B": 64, "H": 16, "D": 128, "S": 16, "ctx_lo": 128, "ctx_hi": 1024,
         "dtype": "bf16", "lens": 7},
        # A whole decode step of the benchmark model (12 layers, vocabulary 32000) at light load.
        {"name": "model_decode", "kind": "model", "B": 16, "H": 16, "D": 128, "S": 16, "ctx_lo": 256, "ctx_hi": 768,
         "dtype": "bf16", "lens": 8, "layers": 12, "vocab": 32000},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "append", "append", "prefill", "prefill", "prefill", "block", "model"])
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    S = rng.choice([16, 16, 32, 64])
    lens = rng.randrange(1 << 20)
    if kind in ("decode", "append"):
        while True:
            B, H, D = _log_int(rng, 1, 256), _log_int(rng, 2, 32), rng.choice([32, 64, 80, 96, 128, 128])
            hi = _log_int(rng, 32, 131072)
            lo = max(1, hi // rng.choice([1, 2, 8, 32]))
            if B * (lo + hi) // 2 * H * D * EB[dtype] * 2 < 8e9:
                break
        return {"kind": kind, "B": B, "H": H, "D": D, "S": S, "ctx_lo": lo, "ctx_hi": hi, "dtype": dtype,
                "lens": lens}
    if kind == "prefill":
        while True:
            T, H, D = _log_int(rng, 16, 4096), rng.choice([4, 8, 12, 16, 20, 32]), rng.choice([32, 64, 80, 128, 128])
            start = 0 if rng.random() < 0.3 else _log_int(rng, 16, 16384)
            if 4 * H * D * T * (start + T / 2) < (3e11 if dtype != "f32" else 6e10):
                break
        return {"kind": kind, "T": T, "start": start, "H": H, "D": D, "S": S, "dtype": dtype}
    dtype = rng.choice(["bf16", "bf16", "f16"])
    D = rng.choice([64, 128])
    H = rng.choice([8, 12, 16, 20]) if kind == "block" else rng.choice([8, 16])
    case = {"kind": kind, "B": _log_int(rng, 1, 200), "H": H, "D": D, "S": S, "ctx_lo": 64,
            "ctx_hi": _log_int(rng, 96, 2000), "dtype": dtype, "lens": lens}
    if kind == "model":
        case.update(layers=rng.randint(2, 12), vocab=rng.choice([8000, 32000, 50257]))
    return case


def _lens(case):
    """Context lengths: part of the case (they set its cost), spread over [ctx_lo, ctx_hi]."""
    r = random.Random(case["lens"])
    return [r.randint(case["ctx_lo"], case["ctx_hi"]) for _ in range(case["B"])]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _pool(layers, blocks, case, g):
    pool = KVBlockPool(layers, blocks, case["S"], case["H"], case["D"], device="cuda", dtype=DTYPES[case["dtype"]])
    pool.k.normal_(generator=g)
    pool.v.normal_(generator=g)
    return pool


def _normal(shape, case, g):
    return torch.empty(shape, device="cuda", dtype=DTYPES[case["dtype"]]).normal_(generator=g)


def _tables(case, seed, spare=8):
    """Block tables over a fragmented pool (a random permutation of its blocks), -1 past each row's blocks."""
    S, lens = case["S"], _lens(case)
    n = [-(-c // S) for c in lens]
    N, M = sum(n) + spare, max(n)
    perm = torch.randperm(N, generator=torch.Generator().manual_seed(seed))
    tables = torch.full((len(lens), M), -1, dtype=torch.int64)
    at = 0
    for b, k in enumerate(n):
        tables[b, :k] = perm[at:at + k]
        at += k
    ctx = torch.tensor(lens, dtype=torch.int64)
    last = ctx - 1
    slots = tables[torch.arange(len(lens)), last // S] * S + last % S
    return N, tables.cuda(), ctx.cuda(), slots.cuda()


def _module(case, seed):
    dt, dim = DTYPES[case["dtype"]], case["H"] * case["D"]
    with torch.random.fork_rng(devices=["cuda"]):
        torch.manual_seed(seed)
        with torch.device("cuda"):
            if case["kind"] == "block":
                m = TransformerBlock(dim, case["H"], 2048)
                m.attn.decode_attention_backend = "hip"
            else:
                m = MiniGPT(n_embd=dim, n_head=case["H"], vocab_size=case["vocab"], block_size=2048,
                            n_layer=case["layers"])
                m.set_decode_attention_backend("hip")
    return m.eval().to(dt)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "prefill":
        T, start, S = case["T"], case["start"], case["S"]
        n = -(-(start + T) // S)
        pool = _pool(1, n + 8, case, g)
        table = torch.randperm(n + 8, generator=torch.Generator().manual_seed(seed))[:n].cuda()
        return {"case": case, "q": _normal((T, case["H"], case["D"]), case, g), "pool": pool, "table": table}
    N, tables, ctx, slots = _tables(case, seed)
    st = {"case": case, "tables": tables, "ctx": ctx, "slots": slots}
    st["pool"] = _pool(case.get("layers", 1), N, case, g)
    row = (case["B"], case["H"], case["D"])
    if kind in ("decode", "append"):
        st["q"] = _normal(row, case, g)
        if kind == "append":
            st["k"], st["v"] = _normal(row, case, g), _normal(row, case, g)
        return st
    st["module"] = _module(case, seed)
    st["meta"] = DecodeBatchMetadata(positions=ctx - 1, context_lengths=ctx, block_tables=tables, slot_mapping=slots)
    if kind == "block":
        st["x"] = _normal((case["B"], 1, case["H"] * case["D"]), case, g)
    else:
        st["ids"] = torch.randint(0, case["vocab"], (case["B"], 1), device="cuda", generator=g)
    return st


def run(st):
    kind = st["case"]["kind"]
    with torch.inference_mode():
        if kind == "prefill":
            return hpd.paged_prefill_hip(st["q"], st["pool"], st["table"], st["case"]["start"], 0)
        if kind == "decode":
            return hpd.paged_attention_batch_hip(st["q"], st["pool"], st["tables"], st["ctx"], 0)
        if kind == "append":
            out = hpd.paged_attention_batch_append_hip(st["q"], st["pool"], st["tables"], st["ctx"], 0, st["k"],
                                                       st["v"], st["slots"])
        elif kind == "block":
            out = st["module"].forward_decode_batch(st["x"], metadata=st["meta"], kv_pool=st["pool"], layer_idx=0)
        else:
            out = st["module"].decode_batch(st["ids"], st["meta"], st["pool"])
        return {"out": out, "k": st["pool"].k, "v": st["pool"].v}


# ------------------------------------------------------------------ in 64 bits

def _attend(q, k, v):
    """softmax(q k^T / sqrt(D)) v of one query row per head: q [H, D], k and v [n, H, D]."""
    s = (k * q).sum(-1) / math.sqrt(q.shape[-1])
    return (torch.softmax(s, 0).unsqueeze(-1) * v).sum(0)


def _rows(pool, layer, table, n):
    """The first n tokens of a table row, [n, H, D] in 64 bits."""
    k, v = (t[layer].index_select(0, table).flatten(0, 1)[:n].double() for t in (pool.k, pool.v))
    return k, v


def _decode64(st, q, layer, k_new=None, v_new=None):
    S, out = st["case"]["S"], []
    for b, n in enumerate(_lens(st["case"])):
        k, v = _rows(st["pool"], layer, st["tables"][b, :-(-n // S)], n)
        if k_new is not None:
            k[n - 1], v[n - 1] = k_new[b], v_new[b]
        out.append(_attend(q[b], k, v))
    return torch.stack(out)


def _linear64(m, x):
    y = x @ m.weight.double().t().contiguous()
    return y if m.bias is None else y + m.bias.double()


def _norm64(m, x):
    y = (x - x.mean(-1, keepdim=True)) * torch.rsqrt(x.var(-1, unbiased=False, keepdim=True) + m.eps)
    return y * m.weight.double() + m.bias.double()


def _block64(st, m, x, layer):
    B, H, D = st["case"]["B"], st["case"]["H"], st["case"]["D"]
    q, k, v = (t.reshape(B, H, D) for t in _linear64(m.attn.qkv, _norm64(m.layer_norm_1, x)).chunk(3, -1))
    x = x + _linear64(m.attn.project, _decode64(st, q, layer, k, v).reshape(B, H * D))
    up = _linear64(m.ffn.network[0], _norm64(m.layer_norm_2, x))
    up = 0.5 * up * (1 + torch.erf(up / math.sqrt(2)))
    return x + _linear64(m.ffn.network[2], up)


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    with torch.inference_mode():
        if kind == "prefill":
            T, start = case["T"], case["start"]
            k, v = _rows(st["pool"], 0, st["table"], start + T)
            mask = torch.arange(start + T, device="cuda")[None] > start + torch.arange(T, device="cuda")[:, None]
            out = torch.empty(st["q"].shape, dtype=torch.float64, device="cuda")
            for h in range(case["H"]):
                s = st["q"][:, h].double() @ k[:, h].t().contiguous() / math.sqrt(case["D"])
                out[:, h] = torch.softmax(s.masked_fill_(mask, -math.inf), -1) @ v[:, h].contiguous()
            return out
        if kind == "decode":
            return _decode64(st, st["q"].double(), 0)
        if kind == "append":
            out = _decode64(st, st["q"].double(), 0, st["k"].double(), st["v"].double())
        elif kind == "block":
            out = _block64(st, st["module"], st["x"][:, 0].double(), 0)[:, None]
        else:
            m = st["module"]
            x = m.token_embedding_table.weight[st["ids"][:, 0]].double()
            x = x + m.position_embedding_table.weight[st["meta"].positions].double()
            for i, blk in enumerate(m.blocks):
                x = _block64(st, blk, x, i)
            out = _linear64(m.language_model_head, _norm64(m.layer_norm, x))[:, None]
        return {"out": out, "k": None, "v": None}


# ------------------------------------------------------------- work, tolerance

def work(case):
    kind, H, D, S, e = case["kind"], case["H"], case["D"], case["S"], EB[case["dtype"]]
    if kind == "prefill":
        T, start = case["T"], case["start"]
        blocks = -(-(start + T) // S)
        return {"bytes": 2 * (start + T) * H * D * e + 2 * T * H * D * e + 8 * blocks,
                "flops": 4 * H * D * (T * start + T * (T + 1) // 2)}
    B, lens = case["B"], _lens(case)
    tokens, blocks = sum(lens), sum(-(-c // S) for c in lens)
    index = 8 * (blocks + B)
    kv = 2 * tokens * H * D * e
    attn_flops = 4 * H * D * tokens
    if kind == "decode":
        return {"bytes": kv + 2 * B * H * D * e + index, "flops": attn_flops}
    if kind == "append":  # the new rows are read from k and v and written once; they need no second read
        return {"bytes": kv + 4 * B * H * D * e + index + 8 * B, "flops": attn_flops}
    dim, layers = H * D, case.get("layers", 1)
    weights = layers * (12 * dim * dim + 10 * dim)
    out = {"bytes": e * weights + layers * (kv + 2 * B * dim * e) + index + 16 * B,
           "flops": layers * (24 * B * dim * dim + attn_flops)}
    if kind == "block":
        out["bytes"] += 2 * B * dim * e
    else:
        out["bytes"] += e * (case["vocab"] * (dim + 1) + 2 * dim + 2 * B * dim + B * case["vocab"]) + 8 * B
        out["flops"] += 2 * B * dim * case["vocab"]
    return out


def tolerance(case):
    # About four times the error against exact() that the path shows (bf16 0.0017-0.0023 for attention, 0.0025
    # for a block, 0.0088 for the 12-layer model; f16 an eighth of those; f32 3e-7 to 6e-7).
    kind, dtype = case["kind"], case["dtype"]
    if kind == "model":
        return {"rel": {"bf16": 4e-2, "f16": 6e-3}[dtype]}
    if kind == "block":
        return {"rel": {"bf16": 1e-2, "f16": 1.5e-3}[dtype]}
    return {"rel": {"bf16": 1e-2, "f16": 1.2e-3, "f32": 2.4e-6}[dtype]}
