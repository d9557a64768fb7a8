"""Workloads of the packed-KV path, as a serving program issues them.

Seven kinds of calls, each through the public entry points of ``nsn_amd``:

- ``decode``: one decode step of a batch over packed K/V plus a dense tail on
  the fast kernel -- a prepared launch (a serving loop's fixed-shape step) or
  a full ``decode_attention`` call;
- ``exact``: the batch-1 readout of ``kernels.launch`` on its default,
  exact-order kernel (the verification route);
- ``prefill``: one chunk of queries over the packed context, the tail and the
  chunk itself, with the chunk's append to the tail in the same launch;
- ``session``: a whole streaming-cache session: a chunked prompt, then decode
  steps, with the compression policy after each;
- ``encode`` / ``restore``: dense blocks to packed blocks and back;
- ``kscore``: decode scores over the per-sequence quantised K store.

Inputs are drawn on the GPU from the seed: token directions N(0, I) normalised
times lognormal norms with 2 % outlier tokens (20 times larger) for cached K/V
(``synthetic.kv_tokens``), N(0, 1) queries and new chunks.  Packed blocks are
built here in plain torch (``_encode``), so that every caller of a seed reads
the same bytes.  Ranges: 1..64 sequences, contexts up to 32K tokens, GQA groups
1..7, 3- and 5-bit codes (4-bit where the entry point takes it), fp16 and bf16.
"""
import math

import torch

from nsn_amd import codec, kernels, kscore
from nsn_amd.kernels import PackedKV
from nsn_amd.stream_cache import StreamingKVCache

BLOCK, DIM = 64, 128
SCALE = 1.0 / math.sqrt(DIM)
DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}

# the head layouts in the repository's tests and benchmark (query heads, kv heads)
HEADS = ((16, 16), (32, 8), (16, 4), (28, 4), (40, 8), (8, 8))


def listed():
    return [
        # one user, short context, MHA, one decode step: launches and latency
        dict(name="decode_single_1k", kind="decode", batch=1, hq=16, hkv=16, lmin=1023, lmax=1023, bits=3,
             tail="bf16", prepared=True),
        # the serving batch of the headline benchmark: 16 ragged sequences of 16K..32K tokens, GQA 32:8
        dict(name="decode_serving_32k", kind="decode", batch=16, hq=32, hkv=8, lmin=16384, lmax=32768, bits=3,
             tail="fp16", prepared=True),
        # many sequences at the 5-bit width
        dict(name="decode_5bit_8k", kind="decode", batch=64, hq=16, hkv=4, lmin=8192, lmax=8192, bits=5,
             tail="fp16", prepared=True),
        # a small ragged batch with an odd group, called without preparation (its shapes change)
        dict(name="decode_odd_group", kind="decode", batch=5, hq=28, hkv=4, lmin=900, lmax=6500, bits=3,
             tail="bf16", prepared=False),
        # the default (exact-order) readout of one sequence: 4096 packed tokens and a 37-token tail, GQA 32:8
        dict(name="exact_single_4k", kind="exact", batch=1, hq=32, hkv=8, lmin=4133, lmax=4133, bits=3,
             tail="bf16"),
        # a late chunk of a batch's 8K prompt, MHA
        dict(name="prefill_late_chunk", kind="prefill", batch=32, hq=16, hkv=16, n=512, cmin=7680, cmax=7680, bits=3,
             dtype="bf16", tail="fp16"),
        # one long document, a single sequence: few query tiles, a long context
        dict(name="prefill_single_32k", kind="prefill", batch=1, hq=32, hkv=8, n=512, cmin=32256, cmax=32256, bits=3,
             dtype="bf16", tail="bf16"),
        # short ragged chunks (a prompt's remainder, a follow-up question) over 5-bit contexts, fp16
        dict(name="prefill_ragged_5bit", kind="prefill", batch=6, hq=28, hkv=4, n=77, cmin=190, cmax=3100, bits=5,
             dtype="fp16", tail="fp16"),
        # a whole session: 1100 prompt tokens in chunks of 512, then 60 decode steps (one of them compresses)
        dict(name="session_prompt_decode", kind="session", batch=8, hq=16, hkv=16, prompt=1100, chunk=512, steps=60,
             bits=3, dtype="bf16"),
        # compressing the K side of the serving batch's prompts
        dict(name="encode_serving", kind="encode", batch=16, heads=8, blocks=400, bits=3, dtype="fp16"),
        # the dense copy a bridge or a native attention reads: packed blocks and the tail
        dict(name="restore_dense_8k", kind="restore", batch=8, heads=16, blocks=127, rest=71, bits=3, dtype="bf16"),
        # decode scores over the 5-bit per-sequence store, GQA 32:8 at 32K tokens
        dict(name="kscore_u8_32k", kind="kscore", batch=16, hq=32, hkv=8, dim=128, tokens=32768, store="u8", bits=5,
             recipe="nsn"),
    ]


# ------------------------------------------------------------------ drawing

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges, costing at most what the largest listed one does."""
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "exact", "session", "encode",
                       "restore", "kscore", "kscore"])
    if kind in ("decode", "exact"):
        hq, hkv = rng.choice(HEADS)
        if kind == "exact":
            batch, hi = 1, _log(rng, 100, 4200)
            lo = hi
        else:
            batch = _log(rng, 1, 64)
            hi = _log(rng, 100, max(200, min(32768, 16 * 8 * 32768 // (batch * hkv))))
            lo = hi if rng.random() < 0.3 else max(1, int(hi * rng.uniform(0.1, 1.0)))
        c = dict(kind=kind, batch=batch, hq=hq, hkv=hkv, lmin=lo, lmax=hi, bits=rng.choice([3, 3, 5]),
                 tail=rng.choice(["fp16", "bf16"]))
        if kind == "decode":
            c["prepared"] = rng.random() < 0.6
        return c
    if kind == "prefill":
        hq, hkv = rng.choice(HEADS)
        batch, n = _log(rng, 1, 32), _log(rng, 16, 512)
        cap = 32 * 16 * 512 * 8192 // (batch * hq * n)   # the late chunk's (query, key) pairs
        hi = _log(rng, 20, max(40, min(32256, cap)))
        lo = hi if rng.random() < 0.4 else int(hi * rng.uniform(0.05, 1.0))
        if rng.random() < 0.15:
            lo = hi = 0
        return dict(kind=kind, batch=batch, hq=hq, hkv=hkv, n=n, cmin=lo, cmax=hi, bits=rng.choice([3, 3, 5]),
                    dtype=rng.choice(["bf16", "bf16", "fp16"]), tail=rng.choice(["fp16", "bf16"]))
    if kind == "session":
        hq, hkv = rng.choice(HEADS)
        return dict(kind=kind, batch=_log(rng, 1, 8), hq=hq, hkv=hkv, prompt=_log(rng, 150, 1100),
                    chunk=rng.choice([128, 256, 512]), steps=rng.randint(10, 60), bits=rng.choice([3, 3, 5]),
                    dtype=rng.choice(["bf16", "fp16"]))
    if kind in ("encode", "restore"):
        batch, heads = _log(rng, 1, 32), rng.choice([4, 8, 16])
        blocks = _log(rng, 1, max(2, 16 * 8 * 400 // (batch * heads * 4)))
        c = dict(kind=kind, batch=batch, heads=heads, blocks=blocks, bits=rng.choice([3, 3, 4, 5]),
                 dtype=rng.choice(["fp16", "bf16"]))
        if kind == "restore":
            c["rest"] = rng.randint(0, 127)
        return c
    hq, hkv = rng.choice([(32, 8), (16, 4), (32, 4), (8, 8)])
    batch, dim = _log(rng, 1, 32), rng.choice([128, 128, 256])
    tokens = _log(rng, 500, min(65536, 16 * 8 * 32768 * 128 // (batch * hkv * dim)))
    store = rng.choice(["u8", "u8", "packed", "fp16"])
    return dict(kind=kind, batch=batch, hq=hq, hkv=hkv, dim=dim, tokens=tokens, store=store,
                bits=rng.choice([3, 4, 5]), recipe="fp16" if store == "fp16" else rng.choice(["nsn", "nsn", "kivi"]))


# ------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _lengths(case, seed):
    """Per-sequence lengths of a case, uniform in its range."""
    lo, hi = (case["cmin"], case["cmax"]) if case["kind"] == "prefill" else (case["lmin"], case["lmax"])
    g = torch.Generator().manual_seed(seed + 77)
    return [int(x) for x in torch.randint(lo, hi + 1, (case["batch"],), generator=g)]


def _tokens(g, shape, dtype):
    """K or V tokens [..., 128]: random directions, lognormal norms, 2 % outlier tokens."""
    u = torch.randn(shape, generator=g, device=DEV)
    u /= torch.linalg.vector_norm(u, dim=-1, keepdim=True)
    r = torch.empty(shape[:-1] + (1,), device=DEV).log_normal_(0.0, 1.0, generator=g)
    r *= torch.where(torch.rand(r.shape, generator=g, device=DEV) < 0.02, 20.0, 1.0)
    return u.mul_(r).to(dtype)


def _codes(x, bits, work=torch.float32):
    """Codes [..., 64, 128] and norm [..., 64], min, scale [..., 128] of blocks x [..., 64, 128]."""
    x = x.to(work)
    n = torch.linalg.vector_norm(x, dim=-1)
    d = x / n.clamp_min(1e-12)[..., None]
    lo, hi = d.amin(-2), d.amax(-2)
    s = (hi - lo) / float(2 ** bits - 1)
    q = torch.round((d - lo[..., None, :]) / torch.where(s == 0, torch.ones_like(s), s)[..., None, :])
    return q.clamp_(0, 2 ** bits - 1), n, lo, s


def _pack(q, bits):
    """LSB-first bitstream of codes [..., 64, 128]: u8 [..., 64*128*bits/8]."""
    w = q.to(torch.int64).reshape(q.shape[:-2] + (BLOCK * DIM // 8, 8))
    w = (w << (bits * torch.arange(8, device=q.device))).sum(-1, keepdim=True)
    w = (w >> (8 * torch.arange(bits, device=q.device))) & 255
    return w.to(torch.uint8).reshape(q.shape[:-2] + (BLOCK * DIM * bits // 8,))


def _unpack(codes, bits):
    w = codes.to(torch.int64).reshape(codes.shape[:-1] + (BLOCK * DIM // 8, bits))
    w = (w << (8 * torch.arange(bits, device=codes.device))).sum(-1, keepdim=True)
    w = (w >> (bits * torch.arange(8, device=codes.device))) & (2 ** bits - 1)
    return w.reshape(codes.shape[:-1] + (BLOCK, DIM))


def _encode(x, bits):
    """Packed fields of blocks x [..., 64, 128]: codes, fp16 norm / min / scale, fp32 decode factor."""
    q, n, lo, s = _codes(x, bits)
    n, lo, s = n.half(), lo.half(), s.half()
    d = lo.float()[..., None, :] + s.float()[..., None, :] * q
    f = n.float() / torch.linalg.vector_norm(d, dim=-1).clamp_min(1e-12)
    return _pack(q, bits), n, lo, s, f


def _decode64(codes, norm, mn, sc, bits):
    """The packed blocks' values [..., 64, 128] in 64 bits."""
    d = mn.double()[..., None, :] + sc.double()[..., None, :] * _unpack(codes, bits).double()
    return norm.double()[..., None] * d / torch.linalg.vector_norm(d, dim=-1, keepdim=True).clamp_min(1e-12)


def _side(g, case, lengths, blocks, tail_cap):
    """One side's packed cache and tails: blocks[b] packed blocks, the rest of lengths[b] in the tail."""
    B, H, bits = case["batch"], case["hkv"], case["bits"]
    cap = max(1, max(blocks))
    kv = PackedKV(codes=torch.zeros((B, H, cap, BLOCK * DIM * bits // 8), dtype=torch.uint8, device=DEV),
                  norm=torch.zeros((B, H, cap, BLOCK), dtype=torch.float16, device=DEV),
                  min=torch.zeros((B, H, cap, DIM), dtype=torch.float16, device=DEV),
                  scale=torch.zeros((B, H, cap, DIM), dtype=torch.float16, device=DEV),
                  factor=torch.zeros((B, H, cap, BLOCK), device=DEV),
                  blocks=torch.tensor(blocks, dtype=torch.int32, device=DEV),
                  tail=torch.zeros((B, H, tail_cap, DIM), dtype=DTYPES[case["tail"]], device=DEV), bits=bits)
    for b in range(B):
        nb, rest = blocks[b], lengths[b] - BLOCK * blocks[b]
        if nb:
            x = _tokens(g, (H, nb, BLOCK, DIM), torch.float16)
            for dst, src in zip((kv.codes, kv.norm, kv.min, kv.scale, kv.factor), _encode(x, bits)):
                dst[b, :, :nb] = src
        if rest:
            kv.tail[b, :, :rest] = _tokens(g, (H, rest, DIM), kv.tail.dtype)
    return kv


def _group(g, case, length):
    """The batch-1 group dict and tail of one side (the layout of ``kernels.launch``)."""
    H, nb = case["hkv"], length // BLOCK
    tail = _tokens(g, (1, H, length - BLOCK * nb, DIM), DTYPES[case["tail"]])
    if nb == 0:
        return None, tail
    codes, n, m, s, _ = _encode(_tokens(g, (1, H, nb, BLOCK, DIM), torch.float16), case["bits"])
    head = torch.zeros((1, H, nb, 12), dtype=torch.uint8, device=DEV)
    return {"codes": codes, "metas": (n[..., None], m[..., None, :], s[..., None, :]), "headers": head}, tail


def _kstore(g, case):
    """The K-score store (see ``kscore.make_store``) of per-channel codes over each sequence's tokens."""
    B, T, H, D = case["batch"], case["tokens"], case["hkv"], case["dim"]
    if case["store"] == "fp16":
        code = torch.randn((B, T, H * D), generator=g, device=DEV).half()
        return {"code": code, "is_fp16": True, "is_nsn": False, "T": T, "n_kv": H, "head_dim": D}
    nsn, top = case["recipe"] == "nsn", 2 ** case["bits"] - 1
    # codes of normal values between a channel's extremes, as the recipes give over many tokens
    unit = D ** -0.5 if nsn else 1.0
    span = unit * (7.0 + torch.rand((B, H * D), generator=g, device=DEV))
    code = torch.empty((B, T, H * D), dtype=torch.uint8, device=DEV)
    for b in range(B):
        z = torch.randn((T, H * D), generator=g, device=DEV) * (unit * top) / span[b] + 0.5 * top
        code[b] = z.round_().clamp_(0, top).to(torch.uint8)
    st = {"code": code, "is_fp16": False, "is_nsn": nsn, "min": (-0.5 * span).half(), "step": (span / top).half(),
          "T": T, "n_kv": H, "head_dim": D}
    if nsn:
        st["eff_norm"] = torch.empty((B, H, T), device=DEV).log_normal_(0.0, 1.0, generator=g).half()
    return kscore.pack_store(st, case["bits"]) if case["store"] == "packed" else st


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = {"case": case}
    if kind == "decode":
        L = _lengths(case, seed)
        blocks = [x // BLOCK for x in L]
        s["k"], s["v"] = (_side(g, case, L, blocks, BLOCK) for _ in range(2))
        s["q"] = torch.randn((case["batch"], case["hq"], DIM), generator=g, device=DEV).to(torch.bfloat16)
        s["len"] = torch.tensor(L, dtype=torch.int32, device=DEV)
        s["max"], s["status"] = max(L), torch.zeros(1, dtype=torch.int32, device=DEV)
        if case["prepared"]:
            s["launch"] = kernels.prepare_decode(s["q"], s["k"], s["v"], s["len"], max_seq_len=s["max"], kernel="fast",
                                                 status=s["status"])
    elif kind == "exact":
        L = _lengths(case, seed)[0]
        s["k"], s["v"] = (_group(g, case, L) for _ in range(2))
        s["q"] = torch.randn((1, case["hq"], 1, DIM), generator=g, device=DEV).to(torch.bfloat16)
        s["status"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    elif kind == "prefill":
        L, n, dt = _lengths(case, seed), case["n"], DTYPES[case["dtype"]]
        blocks = [max(0, (x - BLOCK) // BLOCK) for x in L]     # the streaming policy leaves 64..127 tail tokens
        s["k"], s["v"] = (_side(g, case, L, blocks, 2 * BLOCK + 512) for _ in range(2))
        s["q"] = torch.randn((case["batch"], case["hq"], n, DIM), generator=g, device=DEV).to(dt)
        s["kc"], s["vc"] = (torch.randn((case["batch"], case["hkv"], n, DIM), generator=g, device=DEV).to(dt)
                            for _ in range(2))
        s["len"], s["precise"] = torch.tensor(L, dtype=torch.int32, device=DEV), min(L) < BLOCK
        s["status"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    elif kind == "session":
        B, dt, total = case["batch"], DTYPES[case["dtype"]], case["prompt"] + case["steps"]
        s["cache"] = StreamingKVCache(1, B, case["hkv"], total, bits=case["bits"], dtype=dt, max_append=case["chunk"],
                                      device=torch.device(DEV, torch.cuda.current_device()))
        at = list(range(0, case["prompt"], case["chunk"])) + [case["prompt"]]
        spans = list(zip(at[:-1], at[1:])) + [(i, i + 1) for i in range(case["prompt"], total)]
        draw_ = lambda h: [torch.randn((B, h, j - i, DIM), generator=g, device=DEV).to(dt) for i, j in spans]  # noqa: E731
        s["q"], s["k"], s["v"] = draw_(case["hq"]), draw_(case["hkv"]), draw_(case["hkv"])
        s["chunks"] = len(at) - 1
        s["out"] = torch.empty((case["steps"], B, case["hq"], DIM), dtype=torch.bfloat16, device=DEV)
        s["status"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    elif kind == "encode":
        s["x"] = _tokens(g, (case["batch"], case["heads"], case["blocks"], BLOCK, DIM), DTYPES[case["dtype"]])
        s["status"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    elif kind == "restore":
        rows = case["batch"] * case["heads"]
        x = _tokens(g, (rows, case["blocks"], BLOCK, DIM), torch.float16)
        s["codes"], *metas, _ = _encode(x, case["bits"])
        s["metas"] = tuple(metas)
        s["tail"] = _tokens(g, (rows, case["rest"], DIM), DTYPES[case["dtype"]])
        s["status"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    else:
        s["store"] = _kstore(g, case)
        s["q"] = torch.randn((case["batch"], case["hq"], case["dim"]), generator=g, device=DEV).half()
    return s


# --------------------------------------------------------------------- runs

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        if case["prepared"]:
            return s["launch"]()
        return kernels.decode_attention(s["q"], s["k"], s["v"], s["len"], max_seq_len=s["max"], kernel="fast",
                                        check=False, status=s["status"])
    if kind == "exact":
        return kernels.launch(s["k"][0], s["k"][1], s["q"], s["v"][0], s["v"][1], status=s["status"])[:2]
    if kind == "prefill":
        out = kernels.prefill_attention(s["q"], s["k"], s["v"], s["len"], s["kc"], s["vc"], check=False,
                                        status=s["status"], append=True, precise_weights=s["precise"])
        return out, s["k"].tail, s["v"].tail
    if kind == "session":
        return _session(s)
    if kind == "encode":
        g = codec.encode_group(s["x"], 0, case["bits"], status=s["status"])
        return g["codes"], g["metas"], g["headers"]
    if kind == "restore":
        return codec.restore(s["codes"], s["metas"], case["bits"], DTYPES[case["dtype"]], tail=s["tail"],
                             status=s["status"])
    return kscore.decode_scores(s["q"], s["store"], case["hq"], case["hkv"], case["dim"])


def _session(s):
    c, outs = s["cache"], []
    c.reset(0)
    for i in range(s["chunks"]):
        outs.append(c.prefill(0, s["q"][i], s["k"][i], s["v"][i], append=True, check=False, status=s["status"]))
        c.post_prefill()
    for j in range(s["case"]["steps"]):
        i = s["chunks"] + j
        c.append(0, s["k"][i], s["v"][i])
        c.decode(0, s["q"][i][:, :, 0], kernel="fast", check=False, status=s["status"], out=s["out"][j])
        c.post_decode()
    nb = c.compressed[0] // BLOCK
    rest = c.length[0] - c.compressed[0]
    state = [[t[:, :, :nb] for t in (kv.codes, kv.norm, kv.min, kv.scale)] + [kv.tail[:, :, :rest]]
             for kv in (c.side(0, "K"), c.side(0, "V"))]
    return outs, s["out"], state


# --------------------------------------------------------------------- work

def _spans(case):
    """A session's (context, new tokens) per call."""
    P, c = case["prompt"], case["chunk"]
    return [(i, min(c, P - i)) for i in range(0, P, c)], [(P + j, 1) for j in range(case["steps"])]


def work(case):
    kind, bits = case["kind"], case.get("bits", 3)
    packed = 16 * bits + 2 + 8           # bytes per packed token and kv-head (codes, norm, min and scale shares)
    if kind in ("decode", "exact"):
        L = sum(_lengths(case, 0))
        tail = sum(x % BLOCK for x in _lengths(case, 0))
        kv = 2 * case["hkv"] * ((L - tail) * packed + tail * 2 * DIM)
        return {"bytes": kv + case["batch"] * case["hq"] * DIM * (2 + 2 + 4), "flops": 4 * DIM * case["hq"] * L}
    if kind == "prefill":
        n, hkv, hq, B = case["n"], case["hkv"], case["hq"], case["batch"]
        L = _lengths(case, 0)
        blocks = [max(0, (x - BLOCK) // BLOCK) for x in L]
        kv = 2 * hkv * sum(BLOCK * nb * packed + (x - BLOCK * nb) * 2 * DIM for x, nb in zip(L, blocks))
        pairs = sum(n * x + n * (n + 1) // 2 for x in L)
        return {"bytes": kv + B * n * DIM * (2 * 2 * hq + 2 * 2 * hkv + 2 * 2 * hkv), "flops": 4 * DIM * hq * pairs}
    if kind == "session":
        hq, hkv, B = case["hq"], case["hkv"], case["batch"]
        pre, dec = _spans(case)
        total = case["prompt"] + case["steps"]
        pairs = sum(n * x + n * (n + 1) // 2 for x, n in pre) + sum(x + 1 for x, _ in dec)
        new = B * total * DIM * (2 * 2 * hq + 2 * 2 * 2 * hkv)
        kv = B * 2 * hkv * packed * (sum(x for x, _ in pre + dec) + total)
        return {"bytes": new + kv, "flops": 4 * DIM * B * hq * pairs}
    if kind in ("encode", "restore"):
        tok = case["batch"] * case["heads"] * case["blocks"] * BLOCK
        rest = case["batch"] * case["heads"] * case.get("rest", 0)
        return {"bytes": tok * (packed + 2 * DIM) + rest * 4 * DIM, "flops": tok * DIM * 8}
    B, T, H, D = case["batch"], case["tokens"], case["hkv"], case["dim"]
    per = {"u8": D, "packed": D * case["bits"] // 8, "fp16": 2 * D}[case["store"]]
    per += 2 if case["recipe"] == "nsn" else 0
    return {"bytes": B * T * (H * per + 4 * case["hq"]), "flops": 2 * B * T * case["hq"] * D}


def tolerance(case):
    """Codes, metadata and restored values are exact by contract.  16-bit attention outputs move by the last
    place of their type when a sum's order moves; chunk outputs also by the 16-bit rounding of the weights."""
    kind = case["kind"]
    if kind in ("encode", "restore"):
        return "exact"
    if kind == "kscore":
        return {"rel": 1e-5, "max": 1e-3}
    if kind in ("decode", "exact"):
        return {"rel": 2e-3, "max": 3e-2}
    if kind == "session" or case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 1e-1}
    return {"rel": 2e-3, "max": 3e-2}


# -------------------------------------------------------------------- exact

def _softmax_av(q, k, v, last):
    """softmax(q k^T / sqrt(128)) v in 64 bits for one sequence: q [hq, n, 128], k, v [hkv, T, 128]; query i
    attends keys 0 .. last + i."""
    hq, n, _ = q.shape
    hkv, T, _ = k.shape
    s = torch.matmul(q.double().reshape(hkv, -1, DIM), k.transpose(1, 2).contiguous()) * SCALE
    s = s.reshape(hkv, hq // hkv, n, T)
    if n > 1:
        i = torch.arange(n, device=q.device)[:, None] + last
        s.masked_fill_(torch.arange(T, device=q.device)[None, :] > i, -math.inf)
    p = torch.softmax(s, -1).reshape(hkv, -1, T)
    return torch.matmul(p, v).reshape(hq, n, DIM)


def _context64(kv, b, nb, rest):
    """Sequence b's packed blocks and tail, [hkv, tokens, 128] in 64 bits."""
    x = _decode64(kv.codes[b, :, :nb], kv.norm[b, :, :nb], kv.min[b, :, :nb], kv.scale[b, :, :nb], kv.bits)
    return torch.cat((x.reshape(x.shape[0], -1, DIM), kv.tail[b, :, :rest].double()), 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "session":
        return _session64(case, seed)
    s = prepare(dict(case, prepared=False), seed)
    if kind == "decode":
        o = []
        for b, L in enumerate(_lengths(case, seed)):
            k, v = (_context64(s[x], b, L // BLOCK, L % BLOCK) for x in "kv")
            o.append(_softmax_av(s["q"][b][:, None], k, v, L)[:, 0])
        o = torch.stack(o)
        return o, o
    if kind == "exact":
        kv, bits = [], case["bits"]
        for g, tail in (s["k"], s["v"]):   # reconstructions are rounded to the tail's type, as the route states
            x = tail[0].double()
            if g is not None:
                n, m, sc = g["metas"]
                y = _decode64(g["codes"], n[..., 0], m[..., 0, :], sc[..., 0, :], bits).to(tail.dtype)
                x = torch.cat((y.reshape(x.shape[0], -1, DIM).double(), x), 1)
            kv.append(x)
        o = _softmax_av(s["q"][0], kv[0], kv[1], kv[0].shape[1])
        return o.reshape(1, 1, -1, DIM), o.reshape(1, -1, 1, DIM)
    if kind == "prefill":
        o = []
        for b, L in enumerate(_lengths(case, seed)):
            nb = max(0, (L - BLOCK) // BLOCK)
            k, v = (torch.cat((_context64(s[x], b, nb, L - BLOCK * nb), s[x + "c"][b].double()), 1) for x in "kv")
            o.append(_softmax_av(s["q"][b], k, v, L))
        return torch.stack(o), None, None
    if kind == "encode":
        n, lo, sc = [], [], []
        for x in s["x"]:
            _, a, b, c = _codes(x, case["bits"], torch.float64)
            n.append(a), lo.append(b), sc.append(c)
        n, lo, sc = torch.stack(n), torch.stack(lo), torch.stack(sc)
        return None, (n[..., None], lo[..., None, :], sc[..., None, :]), None
    if kind == "restore":
        x = _decode64(s["codes"], *s["metas"], case["bits"])
        return torch.cat((x.reshape(x.shape[0], -1, DIM), s["tail"].double()), 1)
    return _kscore64(case, s)


def _kscore64(case, s):
    B, T, H, D, G = case["batch"], case["tokens"], case["hkv"], case["dim"], case["hq"] // case["hkv"]
    st, out = s["store"], torch.empty((case["batch"], case["hq"], case["tokens"]), dtype=torch.float64, device=DEV)
    for b in range(B):
        if case["store"] == "fp16":
            k = st["code"][b].double()
        else:
            code = st["code"][b]
            if case["store"] == "packed":
                bits = case["bits"]
                w = code.to(torch.int64).reshape(T, -1, bits)
                w = (w << (8 * torch.arange(bits, device=DEV))).sum(-1, keepdim=True)
                code = ((w >> (bits * torch.arange(8, device=DEV))) & (2 ** bits - 1)).reshape(T, H * D)
            k = code.double() * st["step"][b].double() + st["min"][b].double()
        k = k.reshape(T, H, D).permute(1, 2, 0).contiguous()
        sc = torch.matmul(s["q"][b].double().reshape(H, G, D), k) / math.sqrt(D)
        if case["recipe"] == "nsn":
            sc *= st["eff_norm"][b].double()[:, None]
        out[b] = sc.reshape(case["hq"], T)
    return out


def _session64(case, seed):
    s = prepare(case, seed)
    bits, B = case["bits"], case["batch"]
    k, v = (torch.cat(s[x], 2) for x in "kv")           # the tail's type is the chunks' own

    def dense(x, packed):                               # packed tokens re-read from their blocks, the rest as stored
        y = x[:, :, :packed].reshape(B, case["hkv"], -1, BLOCK, DIM)
        c, n, m, sc, _ = _encode(y, bits)
        return torch.cat((_decode64(c, n, m, sc, bits).reshape(B, case["hkv"], packed, DIM), x[:, :, packed:].double()), 2)

    outs, steps, packed, kd, vd = [], [], 0, k.double(), v.double()
    pre, dec = _spans(case)
    for i, (ctx, n) in enumerate(pre + dec):
        o = torch.stack([_softmax_av(s["q"][i][b], kd[b, :, :ctx + n], vd[b, :, :ctx + n], ctx) for b in range(B)])
        (outs if i < len(pre) else steps).append(o)
        L = ctx + n
        if i < len(pre):
            target = max(packed, max(0, (L - BLOCK) // BLOCK * BLOCK))
        else:
            target = packed + BLOCK if L - packed >= 2 * BLOCK else packed
        if target != packed:
            packed, kd, vd = target, dense(k, target), dense(v, target)
    return outs, torch.stack([o[:, :, 0] for o in steps]) if steps else None, None
