"""GPU parity of the chunked-prefill attention (nsn_prefill_attention) through the C-ABI.

Expected values: the context K/V restored by the oracle (C restatement of
nsn_encode + nsn_decode: fp32 reconstructions for fp16 data, rounded to bf16
for bf16 data as the reference's restore returns them), the tail and the
chunk K/V as stored, then the oracle's float64 chunked-prefill attention
(oracle.prefill_attention64, pinned row by row against the decode oracle).
Tolerance (north star): |out - ref| <= 2e-3 + 1e-2 * |ref| elementwise, plus
the output's own rounding (bf16: 2^-8, fp16: 2^-11 relative) and nothing
else.  K/V and queries are N(0,1) activations, as in the chunked-prefill
configuration, except where a test scales them.
"""
import numpy as np
import pytest
import torch

from nsn_amd import cache, kernels
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
ATOL, RTOL = 2e-3, 1e-2
SCALE = 0.08838834764831845


def normal_tokens(rng, prefix, ntok):
    """fp16 [*prefix, ntok, 128] N(0,1) activations (the C4 configuration's K/V)."""
    return rng.standard_normal(tuple(prefix) + (ntok, 128)).astype(np.float16)


def restore_ctx(x16, length, bits, dtype, packed_dtype=None):
    """[H, T, 128] fp16 source -> fp32 [H, length, 128]: packed blocks restored
    (fp32, rounded to ``packed_dtype`` when bf16), tail tokens as stored in `dtype`."""
    H = x16.shape[0]
    C = (length // 64) * 64
    parts = []
    if C:
        blocks = x16[:, :C].astype(np.float32).reshape(H, C // 64, 64, 128)
        q, n, m, s, err = O.nsn_encode(blocks, bits)
        assert err == 0
        y = O.nsn_decode_f32(q, n, m, s).reshape(H, C, 128)
        if packed_dtype == torch.bfloat16:
            y = O.from_bf16_bits(O.cast_bits(y, "bfloat16"))
        parts.append(y)
    if length > C:
        parts.append(torch.from_numpy(x16[:, C:length]).to(dtype).float().numpy())
    return np.concatenate(parts, axis=1) if parts else np.zeros((H, 0, 128), np.float32)


def run_case(seed, B, Hq, Hkv, ctx_lengths, n, bits, dtype, tail_dtype=None, chunk_scale=None, weighted=0.0,
             precise=None):
    """chunk_scale: optional [n] multipliers of the chunk's V rows (values past
    fp16's range).  weighted: a term added to the bound, times the attention
    over |V| (only the out-of-fp16-range case uses it; see there)."""
    rng = np.random.default_rng(seed)
    tail_dtype = tail_dtype or dtype
    T = max(max(ctx_lengths), 1)
    kx = normal_tokens(rng, (B, Hkv), T)
    vx = normal_tokens(rng, (B, Hkv), T)
    kch = torch.from_numpy(normal_tokens(rng, (B, Hkv), n)).to(dtype)
    vch = torch.from_numpy(normal_tokens(rng, (B, Hkv), n)).to(dtype)
    if chunk_scale is not None:
        vch = (vch.float() * torch.from_numpy(chunk_scale.astype(np.float32))[None, None, :, None]).to(dtype)
    q = torch.from_numpy(rng.standard_normal((B, Hq, n, 128)).astype(np.float32)).to(dtype)
    if max(ctx_lengths) > 0:
        kk, seq = cache.pack_sequences(torch.from_numpy(kx).to(DEV), ctx_lengths, bits=bits, tail_dtype=tail_dtype)
        vv, _ = cache.pack_sequences(torch.from_numpy(vx).to(DEV), ctx_lengths, bits=bits, tail_dtype=tail_dtype)
    else:
        kk = vv = None
        seq = torch.zeros(B, dtype=torch.int32, device=DEV)
    out = kernels.prefill_attention(q.to(DEV), kk, vv, seq, kch.to(DEV), vch.to(DEV), precise_weights=precise)
    got = out.float().cpu().numpy()
    for b in range(B):
        L = ctx_lengths[b]
        kc = restore_ctx(kx[b], L, bits, tail_dtype, dtype)
        vc = restore_ctx(vx[b], L, bits, tail_dtype, dtype)
        ref = O.prefill_attention64(q[b].float().numpy(), kc, vc, kch[b].float().numpy(), vch[b].float().numpy())
        ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11      # the output's own rounding
        err = np.abs(got[b] - ref)
        bound = ATOL + (RTOL + ulp) * np.abs(ref)
        if weighted:
            bound = bound + weighted * O.prefill_attention64(q[b].float().numpy(), kc, np.abs(vc),
                                                             kch[b].float().numpy(), np.abs(vch[b].float().numpy()))
        ratio = float((err / bound).max())
        print(f"prefill case seed {seed} sequence {b}: max err {float(err.max()):.2e}, max err/bound {ratio:.3f}",
              flush=True)
        assert ratio <= 1.0, (b, float(err.max()), ratio)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_packed_context_tail_and_chunk(dtype):
    # sequence 0: 4 blocks + 44 tail tokens; sequence 1: 1 block + 13 tail; one query tile of 150
    run_case(21, 2, 4, 2, [300, 77], 150, 3, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_second_query_tile_ragged(dtype):
    """A workgroup covers 256 chunk queries: 520 queries take three tiles, the
    last with 8 rows, so the query offset, the end clamp and the causal mask
    of queries >= 256 against chunk blocks are all compared with the oracle."""
    run_case(25, 2, 4, 2, [300, 77], 520, 3, dtype)


def test_prefill_c4_chunk_of_512():
    # the C4 chunk size (two full query tiles) over a packed context + tail, GQA 2:1
    run_case(26, 2, 4, 2, [1000, 130], 512, 3, torch.float16)


@pytest.mark.parametrize("precise", [None, False])
def test_prefill_no_context_is_causal_attention(precise):
    """No context: by default (None) the bf16 weights carry their lo parts; the
    single-rounded form (False) is held to the same bound."""
    run_case(22, 1, 2, 2, [0], 200, 3, torch.bfloat16, precise=precise)


def test_prefill_block_aligned_context_gqa8():
    # context of whole blocks only (no tail); 8 q-heads per kv-head
    run_case(23, 1, 8, 1, [256], 64, 3, torch.bfloat16)


def test_prefill_5bit():
    run_case(24, 2, 2, 2, [192, 100], 70, 5, torch.float16)


@pytest.mark.parametrize("tail_dtype,precise", [(torch.bfloat16, None), (torch.float16, None),
                                                (torch.float16, True)])
def test_prefill_5bit_bf16_products(tail_dtype, precise):
    """5-bit packed context under bf16 queries and chunk (the bf16 MFMA form of
    the 5-bit kernel): over a bf16 or an fp16 tail, single-rounded or hi + lo
    weights, across two query tiles with a ragged second one."""
    run_case(29, 2, 4, 2, [300, 77], 300, 5, torch.bfloat16, tail_dtype=tail_dtype, precise=precise)


@pytest.mark.parametrize("precise", [None, True])
def test_prefill_bf16_products_with_an_fp16_tail(precise):
    """C4's mix: bf16 queries and chunk on the bf16 MFMA over an fp16 tail,
    with single-rounded weights (the default over a context) and with the
    weights as bf16 hi + lo (precise_weights=True)."""
    run_case(27, 2, 4, 2, [300, 77], 150, 3, torch.bfloat16, tail_dtype=torch.float16, precise=precise)


def test_prefill_bf16_values_beyond_fp16_range():
    """bf16 chunk values of order 1e6 compute on the bf16 products (fp16 would
    overflow).  This is a range test, not a precision test: with values of
    order 1e6 of both signs the output cancels to far below them, and no fp32
    computation meets an absolute 2e-3 there (fp32 softmax weights alone carry
    2^-24 of the attention-weighted |v|, ~0.06).  The bound therefore adds
    2^-8 of the attention-weighted |v| (the bf16 weights' rounding); every
    N(0,1) case above is held to the north-star bound alone."""
    scale = np.ones(200)
    scale[3::11] = 1e6
    run_case(28, 1, 2, 2, [130], 200, 3, torch.bfloat16, chunk_scale=scale, weighted=2.0 ** -8)


@pytest.mark.parametrize("bits,dtype", [(3, torch.bfloat16), (5, torch.float16)])
@pytest.mark.parametrize("lengths,n", [([1, 2, 63], 1), ([64, 65, 127], 31), ([128, 129, 191], 33), ([192, 193, 255], 65),
                                       ([256, 320, 390], 257)])
def test_prefill_edges_of_the_block_pipeline(lengths, n, bits, dtype):
    """0 to 6 packed blocks (the packed-only loop runs from 3 on), with and
    without a tail block, by chunks around a wave's 32 queries, one block and
    one workgroup: every prologue, hand-over and last half block."""
    run_case(40, 3, 2, 1, lengths, n, bits, dtype, precise=min(lengths) < 64)


@pytest.mark.parametrize("Hq,Hkv,n", [(7, 1, 1), (7, 1, 37), (6, 2, 85), (6, 2, 86), (10, 2, 256), (3, 1, 300)])
def test_prefill_tiles_across_heads(Hq, Hkv, n):
    """A tile's 256 rows run over the ends of a group's heads: several whole
    heads a tile, 3 x 85 rows (one short of it) and 3 x 86 (two over), a head
    a tile, and heads that begin and end inside one; causal inside the chunk."""
    run_case(42, 2, Hq, Hkv, [200, 70], n, 3, torch.float16)


@pytest.mark.parametrize("B,Hq,Hkv,n", [(1, 6, 2, 85), (2, 32, 8, 300), (2, 64, 2, 256), (2, 65, 5, 256), (3, 28, 4, 600)])
def test_prefill_tiles_of_single_heads(B, Hq, Hkv, n):
    """A call whose q-heads' tiles fit the 256 CUs has one head a tile (128 and
    256 of them; 260 and 252 around the limit), an append by one head of each
    group; the oracle's output and the tails as without the append's launch."""
    rng = np.random.default_rng(46)
    L = [200] * B
    x = [torch.from_numpy(normal_tokens(rng, (B, Hkv), 200)).to(DEV) for _ in range(2)]
    q, kc, vc = (torch.from_numpy(normal_tokens(rng, (B, h), n)).to(DEV) for h in (Hq, Hkv, Hkv))
    sides = []
    for t in x:
        kv, seq = cache.pack_sequences(t, L, tail_dtype=torch.float16)
        room = torch.zeros((B, Hkv, 64 + n, 128), dtype=torch.float16, device=DEV)
        room[:, :, :kv.tail.shape[2]] = kv.tail
        kv.tail = room
        sides.append(kv)
    out = kernels.prefill_attention(q, sides[0], sides[1], seq, kc, vc, append=True).float().cpu().numpy()
    for kv, new in zip(sides, (kc, vc)):
        assert torch.equal(kv.tail[:, :, 8:8 + n], new) and not bool(kv.tail[:, :, 8 + n:].any())
    for b in range(B):
        ctx = [restore_ctx(t[b].cpu().numpy(), 200, 3, torch.float16) for t in x]
        ref = O.prefill_attention64(*(a.float().cpu().numpy() if torch.is_tensor(a) else a
                                      for a in (q[b], *ctx, kc[b], vc[b])))
        assert np.all(np.abs(out[b] - ref) <= ATOL + (RTOL + 2.0 ** -11) * np.abs(ref))


@pytest.mark.parametrize("dtype,bits", [(torch.bfloat16, 3), (torch.float16, 5)])
@pytest.mark.parametrize("splits,Hq,n", [(2, 4, 70), (3, 2, 1), (5, 4, 300), (16, 2, 33)])
def test_prefill_context_splits(monkeypatch, splits, Hq, n, dtype, bits):
    """The tiles' blocks shared by several workgroups and merged: contexts too
    short to split (one of 300 tokens writes its output itself), 17 blocks (two
    splits) and 40 (up to five), chunk blocks masked for the first rows of a
    split, rows past the last, and more splits asked than the blocks allow."""
    monkeypatch.setattr(kernels._lib.lib(), "nsn_prefill_splits", lambda *a: splits)
    run_case(43, 3, Hq, 2, [300, 1050, 2500], n, bits, dtype)


@pytest.mark.parametrize("blocks,tail,n,splits", [(11, 640, 128, 1), (13, 640, 64, 2), (14, 640, 128, 2), (0, 1536, 64, 2)])
def test_prefill_splits_of_unknown_lengths(monkeypatch, blocks, tail, n, splits):
    """Lengths that stay on the device: as many splits as the packed capacity,
    two blocks of tail and the chunk fill; a long tail's empty room does not
    count, and a context without packed blocks counts all of it."""
    lib, used = kernels._lib.lib(), []
    real = lib.nsn_prefill_attention_split

    def launch(a, s, ws, stream):
        used.append(s)
        return real(a, s, ws, stream)
    monkeypatch.setattr(lib, "nsn_prefill_attention_split", launch)
    rng = np.random.default_rng(47)
    sides = []
    for _ in range(2):
        kv, seq = cache.pack_sequences(torch.from_numpy(normal_tokens(rng, (1, 8), max(64 * blocks, 64))).to(DEV),
                                       [max(64 * blocks, 64)], tail_dtype=torch.float16)
        kv.tail = torch.zeros((1, 8, tail, 128), dtype=torch.float16, device=DEV)
        if not blocks:
            kv = kernels.PackedKV(None, None, None, None, None, None, kv.tail, 3)
        sides.append(kv)
    q, kc, vc = (torch.from_numpy(normal_tokens(rng, (1, h), n)).to(DEV) for h in (32, 8, 8))
    kernels.prefill_attention(q, sides[0], sides[1], seq, kc, vc, check=False)
    assert used == [splits]


def test_prefill_context_splits_append(monkeypatch):
    """The splits of the last tile append the chunk between them: tails and
    status as without splits, output within one rounding of it."""
    rng = np.random.default_rng(44)
    x = [torch.from_numpy(normal_tokens(rng, (2, 2), 2000)).to(DEV) for _ in range(2)]
    q, kc, vc = (torch.from_numpy(normal_tokens(rng, (2, h), 90)).to(DEV) for h in (4, 2, 2))
    got = []
    for splits in (1, 4):
        monkeypatch.setattr(kernels._lib.lib(), "nsn_prefill_splits", lambda *a: splits)
        sides = []
        for t in x:
            kv, seq = cache.pack_sequences(t, [2000, 700])
            room = torch.zeros((2, 2, 192, 128), dtype=torch.float16, device=DEV)
            room[:, :, :kv.tail.shape[2]] = kv.tail
            kv.tail = room
            sides.append(kv)
        out = kernels.prefill_attention(q, sides[0], sides[1], seq, kc, vc, append=True)
        got.append((out, sides[0].tail, sides[1].tail))
    for a, b in zip(got[0][1:], got[1][1:]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    d = (got[0][0].float() - got[1][0].float()).abs()
    # fp16 outputs of the same sums in another order, with fp16 weights whose scale moves with the split's maximum
    assert bool((d <= 2.0 ** -10 * got[0][0].float().abs() + 2.0 ** -10).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("where,B,Hq,n,L,splits", [
    ("k_factors", 1, 2, 90, 1920, 4),   # every block of the second of four splits: NaN scores only
    ("k_chunk", 1, 1, 512, 512, 2),     # a NaN key in each chunk block; the later tile's second split is the chunk
    # a NaN value in a split where the earlier queries of a head see no token
    # (32 sequences: the unsplit call's tiles run over head ends as well)
    ("v_chunk", 32, 3, 600, 384, 2),
    ("v_factors", 1, 2, 90, 1920, 4),
])
def test_prefill_context_splits_keep_nonfinite_values(monkeypatch, where, B, Hq, n, L, splits, dtype):
    """Nonfinite K/V in one split only: the NaN outputs and the status are those
    of the unsplit call, the other rows within one rounding of the output and
    one of the weights (whose scale moves with the split's maximum)."""
    from nsn_amd import _dev, _lib
    rng = np.random.default_rng(45)
    (kk, seq), (vv, _) = (cache.pack_sequences(torch.from_numpy(normal_tokens(rng, (B, 1), L)).to(DEV), [L] * B,
                                               tail_dtype=dtype) for _ in range(2))
    q, kc, vc = (torch.from_numpy(normal_tokens(rng, (B, h), n)).to(DEV, dtype) for h in (Hq, 1, 1))
    if where == "k_factors":
        kk.factor.view(B, 1, -1, 64)[:, :, 8:16] = float("nan")
    elif where == "v_factors":
        vv.factor.view(B, 1, -1, 64)[:, :, 8:16] = float("nan")
    elif where == "k_chunk":
        kc[:, :, ::64] = float("nan")
    else:
        vc[:, :, -1] = float("nan")
    got = []
    for s in (1, splits):
        monkeypatch.setattr(kernels._lib.lib(), "nsn_prefill_splits", lambda *a, s=s: s)
        st = _dev.new_status(DEV)
        out = kernels.prefill_attention(q, kk, vv, seq, kc, vc, check=False, status=st, precise_weights=False)
        got.append((out.float(), _dev.read_status(st)))
    (one, s1), (many, s2) = got
    print(f"nonfinite {where}: {int(one.isnan().sum())} NaN of {one.numel()} unsplit, {int(many.isnan().sum())} split",
          flush=True)
    assert s1 == s2 == _lib.ST_NONFINITE_OUTPUT
    assert bool(one.isnan().any()) and torch.equal(one.isnan(), many.isnan())
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    d = (one - many).abs().nan_to_num(0.0)
    # N(0,1) values: a row's weights, rounded twice, move it by at most 2u of the attended |v| (< 4)
    assert bool((d <= 2 * u * one.abs().nan_to_num(0.0) + 8 * u).all())


def test_prefill_repeats_bit_for_bit():
    """Every read of a product's result waits for it: the same call twice gives
    the same bits (a maximum read too early moves only the last place)."""
    rng = np.random.default_rng(41)
    L, n = [700, 330], 300
    x = [torch.from_numpy(normal_tokens(rng, (2, 2), 700)).to(DEV) for _ in range(2)]
    (kk, seq), (vv, _) = (cache.pack_sequences(t, L, tail_dtype=torch.float16) for t in x)
    q, kc, vc = (torch.from_numpy(rng.standard_normal((2, h, n, 128)).astype(np.float32)).to(DEV, torch.bfloat16)
                 for h in (4, 2, 2))
    first = kernels.prefill_attention(q, kk, vv, seq, kc, vc)
    for _ in range(4):
        assert torch.equal(first.view(torch.int16), kernels.prefill_attention(q, kk, vv, seq, kc, vc).view(torch.int16))
