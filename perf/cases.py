"""Performance cases of the paged-KV attention path: the work one serving
step has it do, through the package's public entry points.

Kinds of case
  decode    AttentionStep.run over `layers` layers, every row decoding one
            token: append of the new K/V, then paged decode attention. The
            step (tables and plans) is made once per step by an engine and
            shared by its layers, so it is part of the state.
  prefill   AttentionStep.run over `layers` layers, every row a prompt chunk
            on tokens already in pages.
  step      a whole engine step of mixed rows through LlamaOp.pforward, the
            rotary embedding included: the host arguments of the step are
            packed inside the pass, as an engine does once per step.
  copy      LlamaOp.local_copy_blocks of whole blocks.
  exchange  LlamaOp.kv_exchange_pack and kv_exchange_scatter of a layer range.
  swap      torch.ops.swapping_ops.swap out to pinned host memory and back.

Row lengths belong to the case (its `lens` number); tensors and page tables
come from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from kunserve_amd import AttentionStep, KVPool, LlamaOp, rope_inv_freq

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
DEVICE = "cuda"


def listed() -> list:
    return [
        # One interactive user on a GQA model (32 query / 8 KV heads): the
        # smallest decode step there is, bound by latency and launches.
        dict(name="decode_one_row", kind="decode", layers=8, hq=32, hkv=8, dim=128, page=16,
             dtype="bf16", rows=1, kv_lo=777, kv_hi=777, mid=0, lens=1),
        # A chat batch on a 32-head model without GQA: 64 rows of lognormal
        # contexts around 700 tokens, the headline decode shape.
        dict(name="decode_chat", kind="decode", layers=4, hq=32, hkv=32, dim=128, page=16,
             dtype="fp16", rows=64, kv_lo=16, kv_hi=4096, mid=700, lens=2),
        # A full GQA batch at long contexts on the default 256-token pages.
        dict(name="decode_gqa_long", kind="decode", layers=2, hq=32, hkv=8, dim=128, page=256,
             dtype="bf16", rows=128, kv_lo=1024, kv_hi=8192, mid=0, lens=3),
        # A small GQA model (head size 64) at a medium batch.
        dict(name="decode_gqa_dim64", kind="decode", layers=4, hq=32, hkv=8, dim=64, page=16,
             dtype="fp16", rows=48, kv_lo=256, kv_hi=4096, mid=0, lens=4),
        # Three query heads per KV head, a few rows of ragged contexts.
        dict(name="decode_ratio3", kind="decode", layers=4, hq=24, hkv=8, dim=128, page=32,
             dtype="bf16", rows=20, kv_lo=100, kv_hi=3000, mid=0, lens=5),
        # A full batch of 512-token prompt chunks on prefixes already in
        # pages, no GQA: the headline prefill shape's first step.
        dict(name="prefill_chunks", kind="prefill", layers=1, hq=32, hkv=32, dim=128, page=16,
             dtype="fp16", rows=16, q_lo=512, q_hi=512, pre_lo=0, pre_hi=2048, lens=6),
        # One whole prompt of a GQA model in a single step, no prefix.
        dict(name="prefill_prompt_gqa", kind="prefill", layers=1, hq=32, hkv=8, dim=128, page=256,
             dtype="bf16", rows=1, q_lo=4000, q_hi=4000, pre_lo=0, pre_hi=0, lens=7),
        # The last chunks of several prompts: few tokens each, long prefixes.
        dict(name="prefill_tails", kind="prefill", layers=2, hq=32, hkv=8, dim=128, page=16,
             dtype="fp16", rows=12, q_lo=1, q_hi=128, pre_lo=512, pre_hi=4096, lens=8),
        # Chunks at the largest head size.
        dict(name="prefill_dim256", kind="prefill", layers=1, hq=16, hkv=8, dim=256, page=16,
             dtype="bf16", rows=4, q_lo=300, q_hi=512, pre_lo=0, pre_hi=2048, lens=9),
        # A whole mixed engine step: 48 decoding rows and two prompt chunks,
        # rotary embedding, append and attention of 8 layers.
        dict(name="engine_step_mixed", kind="step", layers=8, hq=32, hkv=8, dim=128, page=16,
             dtype="bf16", rows=48, kv_lo=64, kv_hi=2048, mid=0, chunks=2, q_lo=512, q_hi=512,
             pre_lo=0, pre_hi=1024, lens=10),
        # Blocks moved from the extend to the base region before parameters
        # are restored.
        dict(name="remap_copy", kind="copy", layers=32, hq=32, hkv=8, dim=128, page=16,
             dtype="fp16", blocks=777, lens=11),
        # A preempted group of requests swapped out to the host and back in.
        dict(name="swap_out_in", kind="swap", layers=16, hq=32, hkv=8, dim=128, page=16,
             dtype="fp16", blocks=96, lens=12),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "step",
                       "copy", "exchange", "swap"])
    ratio, hkv = rng.choice([(1, 32), (1, 16), (2, 8), (3, 8), (4, 8), (4, 8), (4, 4), (5, 8),
                             (6, 8), (7, 4), (8, 8), (8, 4)])
    case = dict(kind=kind, hq=ratio * hkv, hkv=hkv, dim=rng.choice([64, 128, 128, 128, 256]),
                page=rng.choice([16, 16, 32, 256]), dtype=rng.choice(["fp16", "bf16"]),
                lens=rng.randrange(1 << 20))
    if kind == "decode":
        hi = _log_int(rng, 40, 8192)
        lo = rng.choice([hi, max(16, hi // 8), 16])
        rows = _log_int(rng, 1, 128)
        # K and V of at most about 2 GiB a layer
        per = hkv * case["dim"] * 4 * (lo + hi) / 2
        rows = max(1, min(rows, int(2e9 / per)))
        case.update(layers=rng.choice([1, 2]), rows=rows, kv_lo=lo, kv_hi=hi, mid=0)
        case["layers"] = 2 if rows * per > 2e8 else 8 if rows * per < 2e7 else 4
    elif kind == "prefill":
        hi = _log_int(rng, 16, 4096)
        lo = rng.choice([hi, max(1, hi // 16)])
        pre = rng.choice([0, _log_int(rng, 64, 4096)])
        rows = _log_int(rng, 1, 32)
        # at most about 0.15 TFLOP and 16384 tokens
        per = 4.0 * case["hq"] * case["dim"] * hi * (pre + hi / 2)
        rows = max(1, min(rows, int(1.5e11 / per), 16384 // hi))
        case.update(layers=1, rows=rows, q_lo=lo, q_hi=hi, pre_lo=0, pre_hi=pre)
    elif kind == "step":
        hi = _log_int(rng, 64, 2048)
        case.update(dim=128, layers=4, rows=_log_int(rng, 1, 48), kv_lo=max(16, hi // 8),
                    kv_hi=hi, mid=0, chunks=rng.randrange(3), q_lo=rng.choice([32, 500]),
                    q_hi=512, pre_lo=0, pre_hi=rng.choice([0, 1024]))
    else:
        blocks = _log_int(rng, 4, 777 if kind == "copy" else 400 if kind == "exchange" else 96)
        case.update(hkv=8, hq=32, dim=128, page=16, blocks=blocks,
                    layers=32 if kind == "copy" else 16)
    return case


# ------------------------------------------------------------ row lengths


def _decode_lens(case) -> np.ndarray:
    rng = np.random.default_rng(case["lens"])
    if case["mid"]:
        kv = np.round(rng.lognormal(math.log(case["mid"]), 1.0, size=case["rows"]))
        return np.clip(kv, case["kv_lo"], case["kv_hi"]).astype(np.int64)
    return rng.integers(case["kv_lo"], case["kv_hi"] + 1, size=case["rows"])


def _chunk_lens(case, rows) -> tuple:
    rng = np.random.default_rng(case["lens"] + 1)
    q = rng.integers(case["q_lo"], case["q_hi"] + 1, size=rows)
    return q, rng.integers(case["pre_lo"], case["pre_hi"] + 1, size=rows)


def _rows(case) -> tuple:
    """(tokens, KV length after the step, decode flag) of each row."""
    kind = case["kind"]
    q, kv, dec = [], [], []
    if kind in ("decode", "step"):
        lens = _decode_lens(case)
        q += [1] * len(lens)
        kv += lens.tolist()
        dec += [1] * len(lens)
    if kind in ("prefill", "step"):
        ql, pre = _chunk_lens(case, case["rows"] if kind == "prefill" else case["chunks"])
        q += ql.tolist()
        kv += (ql + pre).tolist()
        dec += [0] * len(ql)
    return q, kv, dec


def _row_args(case, seed: int) -> dict:
    """Host arguments of the step, as an engine hands them over."""
    q, kv, dec = _rows(case)
    need = [-(-n // case["page"]) for n in kv]
    pages = sum(need) + sum(need) // 4 + 4
    perm = np.random.default_rng(seed).permutation(pages)
    tables, at = [], 0
    for n in need:
        tables.append(perm[at:at + n].tolist())
        at += n
    first = [n if d else n - t for t, n, d in zip(q, kv, dec)]
    return dict(q=q, kv=kv, dec=dec, first=first, pages=pages, tables=tables)


# ---------------------------------------------------------------- prepare


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype, scale=1.0) -> torch.Tensor:
    return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(0.0, scale, generator=g)


def _new_tokens(case, g, tokens: int) -> tuple:
    """q, k and v of the step's tokens for every layer. Scores have a
    standard deviation of 2, so rows attend unevenly."""
    dt, ln, d = DTYPES[case["dtype"]], case["layers"], case["dim"]
    return (_normal(g, (ln, tokens, case["hq"], d), dt, 2.0),
            _normal(g, (ln, tokens, case["hkv"], d), dt),
            _normal(g, (ln, tokens, case["hkv"], d), dt))


def _llama_op(case, pages: int) -> LlamaOp:
    return LlamaOp(pages, case["layers"], case["hq"], case["hkv"], case["page"], case["dim"],
                   14336, 128256, 256, 16384, 8192, 1, device=torch.device(DEVICE, 0),
                   dtype=DTYPES[case["dtype"]])


def prepare(case, seed: int) -> dict:
    kind, dt, g = case["kind"], DTYPES[case["dtype"]], _gen(seed)
    if kind in ("decode", "prefill"):
        a = _row_args(case, seed)
        pool = KVPool.allocate(a["pages"], case["layers"], case["hkv"], case["page"],
                               case["dim"], DEVICE, dt)
        pool.k.normal_(generator=g)
        pool.v.normal_(generator=g)
        q, k, v = _new_tokens(case, g, sum(a["q"]))
        step = AttentionStep(pool, case["hq"], a["q"], a["first"], [1 - d for d in a["dec"]],
                             a["tables"])
        return dict(kind=kind, args=a, pool=pool, q=q, k=k, v=v, step=step)
    if kind == "step":
        a = _row_args(case, seed)
        op = _llama_op(case, a["pages"])
        op.pool.k.normal_(generator=g)
        op.pool.v.normal_(generator=g)
        q, k, v = _new_tokens(case, g, sum(a["q"]))
        return dict(kind=kind, args=a, op=op, pool=op.pool, q=q, k=k, v=v,
                    q_now=torch.empty_like(q), ids=[[1] * n for n in a["q"]],
                    inv_freq=rope_inv_freq(case["dim"], 500000.0, torch.device(DEVICE, 0)))
    n = case["blocks"]
    rng = np.random.default_rng(seed)
    if kind == "swap":
        shape = (2 * n + 3, case["layers"], case["hkv"], case["page"], case["dim"])
        cache = [_normal(g, shape, dt) for _ in range(2)]
        host = [torch.zeros((n + 5,) + shape[1:], dtype=dt, pin_memory=True) for _ in range(2)]
        gpu, cpu = rng.permutation(2 * n + 3), rng.permutation(n + 5)
        return dict(kind=kind, cache=cache, host=host, src=gpu[:n].tolist(),
                    cpu=cpu[:n].tolist(), dst=gpu[n:2 * n].tolist())
    op = _llama_op(case, 2 * n + 3)
    op.pool.k.normal_(generator=g)
    op.pool.v.normal_(generator=g)
    perm = rng.permutation(2 * n + 3).tolist()
    return dict(kind=kind, op=op, pool=op.pool, src=perm[:n], dst=perm[n:2 * n],
                lo=case["layers"] // 4, hi=case["layers"] // 4 + case["layers"] // 2)


# -------------------------------------------------------------------- run


def run(s):
    kind = s["kind"]
    if kind in ("decode", "prefill"):
        outs = [s["step"].run(i, s["q"][i], s["k"][i], s["v"][i])
                for i in range(s["q"].shape[0])]
        return outs + [s["pool"].k, s["pool"].v]
    if kind == "step":
        # The rotation is in place: q arrives anew each step, as from the
        # QKV projection.
        s["q_now"].copy_(s["q"])
        a, op = s["args"], s["op"]
        step = op.pforward(len(a["q"]), sum(a["q"]), op.max_num_pages, 0, op.layers, s["ids"],
                           a["first"], [1 - d for d in a["dec"]], a["tables"])
        outs = [step.run(i, s["q_now"][i], s["k"][i], s["v"][i], rope=(s["inv_freq"], False))
                for i in range(op.layers)]
        return outs + [s["q_now"], s["pool"].k, s["pool"].v]
    if kind == "copy":
        s["op"].local_copy_blocks(s["op"].max_num_pages, s["src"], s["dst"])
        return [s["pool"].k, s["pool"].v]
    if kind == "exchange":
        packed = s["op"].kv_exchange_pack(s["src"], s["lo"], s["hi"])
        s["op"].kv_exchange_scatter(s["dst"], s["lo"], s["hi"], packed)
        return [packed, s["pool"].k, s["pool"].v]
    swap = torch.ops.swapping_ops.swap
    swap(s["src"], s["cpu"], False, *s["cache"], *s["host"])
    swap(s["cpu"], s["dst"], True, *s["cache"], *s["host"])
    return s["cache"] + s["host"]


# ------------------------------------------------------ work and tolerance


def work(case) -> dict:
    kind = case["kind"]
    if kind in ("copy", "exchange", "swap"):
        block = 2 * 2 * case["hkv"] * case["page"] * case["dim"]   # K and V, one layer
        layers = case["layers"] // 2 if kind == "exchange" else case["layers"]
        return {"bytes": block * layers * case["blocks"] * (2 if kind == "copy" else 4),
                "flops": 0}
    q, kv, _ = _rows(case)
    tokens, cached, pairs = sum(q), sum(kv), 0
    for t, n in zip(q, kv):
        pairs += t * (n - t) + t * (t + 1) // 2
    row = 2 * case["dim"]
    # K and V of every cached token read once (the new ones come from the
    # step's k and v), the new ones written, q read and out written.
    one = cached * case["hkv"] * row * 2 + tokens * case["hkv"] * row * 2 \
        + 2 * tokens * case["hq"] * row
    if kind == "step":   # q read and written by the rotation, k read
        one += 2 * tokens * case["hq"] * row
    return {"bytes": one * case["layers"],
            "flops": 4 * case["hq"] * case["dim"] * pairs * case["layers"]}


def tolerance(case):
    if case["kind"] in ("copy", "exchange", "swap"):
        return "exact"
    # Against 64 bits the path is off by 2.1e-4 to 2.7e-4 in fp16 and 1.7e-3 to
    # 2.3e-3 in bf16 (output rounding, and probabilities rounded for the matrix
    # units); with the rotary embedding's roundings of q and k by 3.5e-4 and
    # 3.9e-3.
    rel = 1e-3 if case["dtype"] == "fp16" else 8e-3
    return {"rel": 2 * rel if case["kind"] == "step" else rel}


# ------------------------------------------------------------------ exact


def _rotate(x, pos, inv_freq):
    """Rotary embedding of x [tokens, heads, dim] in float64, halves paired."""
    ang = pos.double()[:, None] * inv_freq.double()[None, :]
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def exact(case, seed: int):
    if case["kind"] in ("copy", "exchange", "swap"):
        return None
    s = prepare(case, seed)
    a, pool_k, pool_v = s["args"], s["pool"].k, s["pool"].v
    ps, d, hkv = case["page"], case["dim"], case["hkv"]
    ratio = case["hq"] // hkv
    rope = case["kind"] == "step"
    starts = np.concatenate([[0], np.cumsum(a["q"])]).tolist()
    pos = torch.cat([torch.arange(n - t, n, device=DEVICE) for t, n in zip(a["q"], a["kv"])])
    full_k = pool_k.double() if rope else None
    outs, rotated = [], []
    for layer in range(case["layers"]):
        q, k, v = s["q"][layer].double(), s["k"][layer].double(), s["v"][layer].double()
        if rope:
            q, k = _rotate(q, pos, s["inv_freq"]), _rotate(k, pos, s["inv_freq"])
            rotated.append(q)
        out = torch.empty_like(q)
        for b, (t, n) in enumerate(zip(a["q"], a["kv"])):
            lo, hi = starts[b], starts[b + 1]
            ids = torch.tensor(a["tables"][b], device=DEVICE)
            if rope:
                p = pos[lo:hi]
                full_k[ids[p // ps], layer, :, p % ps] = k[lo:hi]
            # cached rows [heads, tokens, dim], the step's own tokens last
            old = [x[ids, layer].double().transpose(0, 1).reshape(hkv, -1, d)[:, :n - t]
                   for x in (pool_k, pool_v)]
            kk = torch.cat([old[0], k[lo:hi].transpose(0, 1)], dim=1)
            vv = torch.cat([old[1], v[lo:hi].transpose(0, 1)], dim=1)
            seen = torch.arange(n, device=DEVICE)[None, :] <= pos[lo:hi][:, None]
            for h in range(hkv):
                kt, vh = kk[h].t().contiguous(), vv[h]
                qh = q[lo:hi, h * ratio:(h + 1) * ratio]
                for r0 in range(0, t, 1024):
                    qr = qh[r0:r0 + 1024]
                    sc = torch.matmul(qr.reshape(-1, d), kt).view(qr.shape[0], ratio, n)
                    sc = sc / math.sqrt(d)
                    sc.masked_fill_(~seen[r0:r0 + 1024, None, :], -math.inf)
                    p = torch.softmax(sc, dim=-1).view(-1, n)
                    out[lo + r0:lo + r0 + qr.shape[0], h * ratio:(h + 1) * ratio] = \
                        torch.matmul(p, vh).view(qr.shape[0], ratio, d)
        outs.append(out)
    if rope:
        return outs + [torch.stack(rotated), full_k, None]
    return outs + [None, None]
