"""The entry points of include/qdc_hip_workspace.h: the recurrence through a
workspace, at the edges of its chunks, slices and wavefront splits, against the
token-by-token oracle; and its argument checks, which need no GPU."""
import os
import re

import numpy as np
import pytest
import torch

from conftest import ROOT, normwise
from qdc_amd import _lib

F32, BF16, X2 = _lib.QDC_F32, _lib.QDC_BF16, _lib.QDC_BF16X2
FAKE = 0x10000  # a non-null, 16-byte aligned address never dereferenced by validation
BIG = 1 << 60


def test_exports_match_header():
    text = open(os.path.join(ROOT, "include", "qdc_hip_workspace.h")).read()
    names = set(re.findall(r"^\s*\w+\s+(qdc_\w+)\s*\(", text, re.M))
    assert names == set(_lib.WORKSPACE_SIGNATURES)
    for name in names:
        assert hasattr(_lib.lib(), name), name


def test_delta_scan_ws_validation():
    lib = _lib.lib()
    size = lib.qdc_delta_scan_workspace
    need = size(2, 33, 4, 128, 48)
    assert need == 2 * 4 * 3 * 544 * 4
    assert size(2, 33, 4, 96, 48) == 0 and size(2, 33, 4, 256, 48) == 0  # key_dim
    assert size(2, 33, 4, 128, 40) == 0                                  # value_dim % 16
    assert size(0, 33, 4, 128, 48) == 0 and size(2, 0, 4, 128, 48) == 0
    assert size(1, 1 << 30, 4, 128, 48) == 0                             # too many chunks

    def f(out=FAKE, dt=F32, q=FAKE, k=FAKE, v=FAKE, beta=FAKE, decay=FAKE, batch=2, seq=33,
          heads=4, kh=2, kd=128, vd=48, ld_qk=256, ld_v=192, ws=FAKE + (1 << 30), nbytes=need):
        return lib.qdc_delta_scan_ws(out, dt, q, k, v, beta, decay, batch, seq, heads, kh, kd, vd,
                                     ld_qk, ld_v, ws, nbytes, None)

    assert f(dt=7) == -3
    assert f(heads=3) == -2 and f(kd=96) == -2 and f(vd=40) == -2
    assert f(ld_qk=255) == -2 and f(ld_v=191) == -2 and f(ld_qk=258) == -2
    assert f(nbytes=need - 1) == -2
    assert f(q=FAKE + 4) == -2 and f(ws=FAKE + (1 << 30) + 8) == -2
    for name in ("out", "q", "k", "v", "beta", "decay", "ws"):
        assert f(**{name: None}) == -1, name
    for name in ("out", "q", "k", "v", "beta", "decay"):  # workspace over another argument
        assert f(**{name: FAKE + (1 << 30) + 16}) == -5, name
    assert f(seq=0, out=None) == 0 and f(batch=0, out=None) == 0


# key_dim x value_dim; heads and batch on both sides of 512 slices of 16 columns
# (whole slices / key parts), value_dim leaving 1..4 slices in the last workgroup
SCAN = [(1, 1, 1, 1, 128, 16), (1, 15, 1, 2, 128, 48), (2, 16, 2, 2, 64, 32), (1, 17, 2, 4, 32, 80),
        (1, 33, 1, 1, 32, 16), (2, 49, 1, 2, 128, 128), (9, 33, 4, 64, 128, 16),
        (6, 17, 16, 32, 128, 48), (5, 31, 8, 32, 64, 64), (3, 48, 8, 64, 32, 80),
        (4, 1, 16, 64, 128, 48), (4, 32, 64, 64, 128, 32)]


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,KH,H,kd,vd", SCAN)
def test_delta_scan_ws_edges(B, S, KH, H, kd, vd):
    """fp32 sums of at most 3 kd products a token, errors of about 1e-7 as in the
    other forms: the repository's fp32 bar of 1e-5 per sequence, and every element
    within 1e-5 of the largest output of its sequence."""
    from oracle import forward
    from qdc_amd import ops
    rng = np.random.default_rng(S * 1000 + kd + vd)
    q = rng.standard_normal((B, S, KH, kd), dtype=np.float32)
    k = rng.standard_normal((B, S, KH, kd), dtype=np.float32)
    q /= np.linalg.norm(q, axis=-1, keepdims=True) * np.float32(np.sqrt(kd))
    k /= np.linalg.norm(k, axis=-1, keepdims=True)
    v = rng.standard_normal((B, S, H, vd), dtype=np.float32)
    beta = rng.random((B, S, H), dtype=np.float32)
    decay = -rng.random((B, S, H), dtype=np.float32) * np.float32(0.5)
    # the column blocks of rows with other data around them
    rows = torch.full((B, S, 2 * KH * kd + H * vd + 8), float("nan"), device="cuda")
    views = []
    at = 4
    for x in (q, k, v):
        w = x.shape[2] * x.shape[3]
        rows[..., at:at + w] = torch.from_numpy(x.reshape(B, S, w)).cuda()
        views.append(rows[..., at:at + w].unflatten(-1, x.shape[2:]))
        at += w
    gates = [torch.from_numpy(x).cuda() for x in (beta, decay)]
    lib = _lib.lib()
    need = lib.qdc_delta_scan_workspace(B, S, H, kd, vd)
    assert need > 0
    out = {}
    for dtype, code in ((torch.float32, F32), (torch.bfloat16, BF16)):
        work = torch.full((need // 4,), float("nan"), device="cuda")  # all of it is written first
        out[dtype] = torch.empty((B, S, H, vd), dtype=dtype, device="cuda")
        ld = rows.shape[-1]
        _lib.check(lib.qdc_delta_scan_ws(out[dtype].data_ptr(), code,
                                         *(t.data_ptr() for t in views + gates), B, S, H, KH, kd,
                                         vd, ld, ld, work.data_ptr(), need,
                                         torch.cuda.current_stream().cuda_stream), "scan")
    assert torch.equal(out[torch.bfloat16], out[torch.float32].bfloat16())
    got = out[torch.float32].cpu().numpy()
    if S > 48:  # the operator takes this form
        assert torch.equal(ops.delta_scan(*views, *gates), out[torch.float32])
    for b in range(B):
        exp = forward.delta_recurrence(q[b], k[b], v[b], beta[b], decay[b])
        assert normwise(got[b], exp) <= 1e-5
        assert np.abs(got[b] - exp).max() <= 1e-5 * np.abs(exp).max()


# whole slices (more than 512) over ten chunks and more with a ragged last one: the LDS
# tiles and running row pointers of that form are used over and over
LONG_SCAN = [(5, 187, 16, 16, 128, 128), (5, 193, 8, 16, 64, 128), (9, 171, 16, 16, 32, 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,KH,H,kd,vd", LONG_SCAN)
def test_delta_scan_ws_long(B, S, KH, H, kd, vd):
    """As above; decays spread over 0.001 .. 0.5 a token, so that what a chunk leaves
    in the state is seen in all that follow."""
    from oracle import forward
    from qdc_amd import ops
    assert B * H * vd // 16 > 512
    rng = np.random.default_rng(S + kd)
    q = rng.standard_normal((B, S, KH, kd), dtype=np.float32)
    k = rng.standard_normal((B, S, KH, kd), dtype=np.float32)
    q /= np.linalg.norm(q, axis=-1, keepdims=True) * np.float32(np.sqrt(kd))
    k /= np.linalg.norm(k, axis=-1, keepdims=True)
    v = rng.standard_normal((B, S, H, vd), dtype=np.float32)
    beta = rng.random((B, S, H), dtype=np.float32)
    decay = -np.exp(rng.uniform(np.log(1e-3), np.log(0.5), (B, S, H))).astype(np.float32)
    got = ops.delta_scan(*(torch.from_numpy(x).cuda() for x in (q, k, v, beta, decay)))
    got = got.cpu().numpy()
    for b in range(B):
        exp = forward.delta_recurrence(q[b], k[b], v[b], beta[b], decay[b])
        assert normwise(got[b], exp) <= 1e-5
        assert np.abs(got[b] - exp).max() <= 1e-5 * np.abs(exp).max()


def test_attention_fused_validation():
    lib = _lib.lib()

    def f(out=FAKE, odt=BF16, q=BIG, k=BIG, v=BIG, gate=BIG, mask=None, batch=2, seq=33, heads=4,
          kv=2, hd=64, q_tok=256, q_head=64, k_tok=128, k_head=64, v_tok=128, v_head=64,
          g_tok=256, g_head=64, o_tok=256, dt=BF16):
        return lib.qdc_attention_fused(out, odt, q, k, v, gate, mask, batch, seq, heads, kv, hd,
                                       q_tok, q_head, k_tok, k_head, v_tok, v_head, g_tok, g_head,
                                       o_tok, 0.125, dt, None)

    assert f(odt=7) == -3 and f(dt=X2) == -3
    assert f(heads=3) == -2 and f(hd=96) == -2 and f(kv=0) == -2 and f(batch=-1) == -2
    assert f(q_tok=260) == -2 and f(k_head=68) == -2 and f(v_tok=130) == -2  # 16-byte rows
    assert f(v_head=32) == -2 and f(g_tok=260) == -2 and f(g_head=68) == -2
    assert f(o_tok=248) == -2 and f(o_tok=260) == -2
    assert f(q=BIG + 8) == -2 and f(out=FAKE + 4) == -2 and f(mask=BIG + 2) == -2
    for name in ("out", "q", "k", "v", "gate"):
        assert f(**{name: None}) == -1, name
    for name in ("q", "k", "v", "gate", "mask"):
        assert f(**{name: FAKE + 16}) == -5, name
    assert f(seq=0, out=None) == 0 and f(batch=0, out=None) == 0


# lengths around the tiles of 32 queries and keys; 1..6 query heads per KV head, so
# that a workgroup's four units cross query blocks; every head size
ATTENTION = [(1, 1, 2, 1, 64, "none"), (2, 31, 6, 6, 64, "holes"), (1, 32, 3, 1, 128, "prefix"),
             (3, 33, 5, 1, 128, "holes"), (2, 65, 8, 2, 256, "prefix"), (1, 97, 6, 1, 256, "none"),
             (1, 160, 4, 2, 64, "none"), (2, 64, 2, 2, 256, "first"), (1, 200, 4, 1, 128, "first")]


@pytest.mark.gpu
@pytest.mark.parametrize("out", ["f32", "bf16", "split"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,H,KV,hd,kind", ATTENTION)
def test_attention_fused_edges(B, S, H, KV, hd, kind, dtype, out):
    """Against 64 bits on the same inputs.  Per element the bf16 form may differ by
    the rounding of the weights, 2^-8 of the weighted mean of |v| (each weight is
    rounded by at most 2^-9 and so is what it replaces), the fp32 form by fp32 sums
    (1e-5 of it); then by the rounding of the output (bf16 2^-9, two terms 2^-17)."""
    from qdc_amd import ops
    rng = np.random.default_rng(S * 10 + H + hd)
    T = B * S
    # q | k | v | gate as the packed projection holds them, scores of a few units
    proj = torch.from_numpy(rng.standard_normal((T, (2 * H + 2 * KV) * hd), dtype=np.float32))
    proj[:, :H * hd] *= 2.0
    proj = proj.to(dtype).cuda()
    q, k, v, gate = (x.unflatten(1, (-1, hd)) for x in
                     proj.split([H * hd, KV * hd, KV * hd, H * hd], 1))
    mask = None
    if kind != "none":
        m = np.ones((B, S), np.int32)
        if kind == "prefix":       # the first queries see no key: an even spread over all
            m[:, :S // 2] = 0
        elif kind == "first":      # nothing kept but the last key
            m[:, :-1] = 0
        else:
            m[rng.random((B, S)) < 0.4] = 0
        mask = torch.from_numpy(m)
    scale = hd ** -0.5
    got = ops.attention_fused(q, k, v, gate, None if mask is None else mask.cuda(), scale, B,
                              out_dtype={"f32": torch.float32, "bf16": torch.bfloat16,
                                         "split": ops.BF16X2}[out])
    got = (ops.join_split(got) if out == "split" else got).double().cpu().view(B, S, H, hd)
    assert torch.isfinite(got).all()
    q, k, v, gate = (x.cpu().double().view(B, S, -1, hd).transpose(1, 2) for x in (q, k, v, gate))
    k, v = (x.repeat_interleave(H // KV, 1) for x in (k, v))
    see = torch.ones(S, S, dtype=torch.bool).tril()[None, None]
    if mask is not None:
        see = see & mask.bool()[:, None, None, :]
    low = -torch.finfo(torch.float32).max
    p = torch.softmax((q @ k.transpose(2, 3) * scale).masked_fill(~see, low), -1)
    exact = (torch.sigmoid(gate) * (p @ v)).transpose(1, 2)
    spread = (torch.sigmoid(gate) * (p @ v.abs())).transpose(1, 2)
    bound = spread * (1e-5 if dtype == torch.float32 else 2.0 ** -8 + 1e-5)
    bound = bound + exact.abs() * {"f32": 0.0, "bf16": 2.0 ** -8, "split": 2.0 ** -16}[out] + 1e-30
    assert ((got - exact).abs() <= bound).all(), ((got - exact).abs() / bound).max()


def test_attention_fused_scale_validation():
    """The running maximum is taken before the scale: a scale that is not positive and
    finite (with its log2(e) factor) is refused before anything else is looked at."""
    lib = _lib.lib()
    for scale in (0.0, -0.125, float("nan"), float("inf"), -float("inf"), 3e38):
        status = lib.qdc_attention_fused(None, BF16, BIG, BIG, BIG, BIG, None, 2, 33, 4, 2, 64, 256,
                                         64, 128, 64, 128, 64, 256, 64, 256, scale, BF16, None)
        assert status == -4, scale


def test_attention_fused_limits():
    """The forward takes the kernel exactly where its grid fits: beyond, the form with a
    score matrix, which took these sizes before."""
    from qdc_amd import ops
    lib = _lib.lib()
    # (batch, seq, heads, kv_heads); a group of 128 heads over one KV head of 16384 tokens
    # is 65536 units of 32 queries, one more than the grid holds in fp32
    sizes = [(1, 16384, 128, 1), (1, 16352, 128, 1), (1, 65535, 128, 1), (1, 65536, 128, 1),
             (1 << 22, 2, 2, 2), ((1 << 22) - 1, 2, 2, 2), (8, 2048, 8, 2), (1, 1 << 25, 8, 2)]
    for dtype, code in ((torch.float32, F32), (torch.bfloat16, BF16)):
        for hd in (64, 96, 128, 256):
            for B, S, H, KV in sizes:
                status = lib.qdc_attention_fused(None, code, BIG, BIG, BIG, BIG, None, B, S, H, KV, hd,
                                                 H * hd, hd, KV * hd, hd, KV * hd, hd, H * hd, hd,
                                                 H * hd, 0.125, code, None)
                assert status in (-1, -2)   # -1: sizes taken, the null pointer refused
                assert ops.attention_fused_takes(dtype, hd, B, S, H, KV) == (status == -1), (hd, B, S)
    assert not ops.attention_fused_takes(torch.float32, 64, *sizes[0])
    assert ops.attention_fused_takes(torch.bfloat16, 64, *sizes[0])
    assert not ops.attention_fused_takes(torch.float16, 64, 1, 1, 1, 1)


def attention_exact(q, k, v, gate, mask, scale, B):
    """What ``ops.attention_fused`` gives, in 64 bits on the same inputs, and the gated
    weighted mean of |v|, ``[B, S, H, hd]``; also the scaled scores ``[B, H, S, S]`` with
    -inf at the keys a query does not see."""
    H, KV = q.shape[1], k.shape[1]
    q, k, v, gate = (x.cpu().double().view(B, -1, x.shape[1], x.shape[2]).transpose(1, 2)
                     for x in (q, k, v, gate))
    k, v = (x.repeat_interleave(H // KV, 1) for x in (k, v))
    S = q.shape[2]
    see = torch.ones(S, S, dtype=torch.bool).tril()[None, None]
    if mask is not None:
        see = see & mask.cpu().bool()[:, None, None, :]
    scores = q @ k.transpose(2, 3) * scale
    low = -torch.finfo(torch.float32).max
    p = torch.softmax(scores.masked_fill(~see, low), -1)
    out = [(torch.sigmoid(gate) * (p @ x)).transpose(1, 2) for x in (v, v.abs())]
    return out[0], out[1], scores.masked_fill(~see, -torch.inf)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.6, 0.75, 1.0, 8.0])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,H,KV,hd,kind", [(2, 200, 4, 2, 64, "prefix"), (1, 161, 4, 1, 256, "none"),
                                              (1, 200, 3, 1, 128, "first")])
def test_attention_fused_scales(B, S, H, KV, hd, kind, dtype, scale):
    """Queries scaled beforehand, up to scale 1 and beyond; masked prefixes longer than a
    step of 64 keys, after which queries see their first key, and queries that see
    none.  Bounds as in the test of the edges (fp32 output)."""
    from qdc_amd import ops
    rng = np.random.default_rng(S + H)
    T = B * S
    q, k, v, gate = (torch.from_numpy(rng.standard_normal((T, n, hd), dtype=np.float32))
                     for n in (H, KV, KV, H))
    q, k, v, gate = (x.to(dtype).cuda() for x in (q * (2.0 * hd ** -0.5 / scale), k, v, gate))
    mask = None
    if kind != "none":
        m = np.ones((B, S), np.int32)
        m[:, :(100 if kind == "prefix" else S - 1)] = 0
        mask = torch.from_numpy(m).cuda()
    got = ops.attention_fused(q, k, v, gate, mask, scale, B, out_dtype=torch.float32)
    got = got.double().cpu().view(B, S, H, hd)
    exact, spread, _ = attention_exact(q, k, v, gate, mask, scale, B)
    bound = spread * (1e-5 if dtype == torch.float32 else 2.0 ** -8 + 1e-5) + 1e-30
    assert torch.isfinite(got).all()
    assert ((got - exact).abs() <= bound).all(), ((got - exact).abs() / bound).max()


def rescalings(scores, dtype):
    """Walks the kernel's order over scaled scores ``[B, H, S, S]`` (-inf: not seen): 32
    queries a wavefront, keys in steps of 64 (bf16) or tiles of 32 dealt to four
    wavefronts (fp32); where a lane's maximum passes what its exponents are taken from by
    2^8, all queries of the wavefront move to their own.  Returns how often that happens to
    sums that are not empty, and how often to some of a wavefront's queries only."""
    x = np.asarray(scores) * np.log2(np.e)
    S = x.shape[-1]
    tile, walks = (64, 1) if dtype == torch.bfloat16 else (32, 4)
    half = np.arange(S) % 8 // 4  # which half-wavefront holds a key
    full = partly = 0
    for rows in x.reshape(-1, S, S):
        for q0 in range(0, S, 32):
            block = rows[q0:q0 + 32, :q0 + 32]
            for w in range(walks):
                base = np.full(block.shape[0], -np.inf)
                for k0 in range(w * tile, block.shape[1], walks * tile):
                    part = block[:, k0:k0 + tile]
                    h = half[k0:k0 + part.shape[1]]
                    tops = np.stack([part[:, h == n].max(1, initial=-np.inf) for n in (0, 1)], 1)
                    seen = tops > -np.inf
                    if (seen & (tops > base[:, None] + 8)).any():
                        moved = tops.max(1) > base
                        held = np.isfinite(base)
                        full += (moved & held).any()
                        partly += (moved & held).any() and (~moved & held).any()
                        base = np.maximum(base, tops.max(1))
    return full, partly


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,H,KV,hd,holes", [(1, 420, 4, 2, 64, False), (2, 450, 3, 1, 128, True),
                                               (1, 500, 4, 1, 256, True)])
def test_attention_fused_rescales(B, S, H, KV, hd, holes, dtype):
    """Scores that rise by 6 to 12 every 96 keys for half of the queries and stay level
    for the others, so that sums already begun are rescaled, in some lanes only, again and
    again.  Scores reach 60: a product's error of up to (hd / 2) roundings of its terms'
    sum moves a weight by that much, twice (its own and the maximum's); otherwise the
    bounds of the edges."""
    from qdc_amd import ops
    rng = np.random.default_rng(S + hd)
    T, scale = B * S, hd ** -0.5
    q, k, v, gate = (rng.standard_normal((T, n, hd), dtype=np.float32) for n in (H, KV, KV, H))
    q[..., 0] = hd ** 0.25 * rng.uniform(0.5, 1.0, (T, H)) * (rng.random((T, H)) < 0.5)
    k[..., 0] = hd ** 0.25 * (12.0 * (np.arange(T) % S // 96))[:, None]
    q, k, v, gate = (torch.from_numpy(x).to(dtype).cuda() for x in (q, k, v, gate))
    mask = None
    if holes:
        mask = torch.from_numpy((rng.random((B, S)) < 0.7).astype(np.int32)).cuda()
    exact, spread, scores = attention_exact(q, k, v, gate, mask, scale, B)
    full, partly = rescalings(scores, dtype)
    assert full > 20 and partly > 20
    size = [x.double().cpu().abs() for x in (q, k)]
    terms = max((size[0][:, h] @ size[1][:, h // (H // KV)].t()).max().item() for h in range(H)) * scale
    bound = spread * (1e-5 + 2 * hd / 2 * 2.0 ** -24 * terms
                      + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)) + 1e-30
    got = ops.attention_fused(q, k, v, gate, mask, scale, B, out_dtype=torch.float32)
    got = got.double().cpu().view(B, S, H, hd)
    assert torch.isfinite(got).all()
    assert ((got - exact).abs() <= bound).all(), ((got - exact).abs() / bound).max()


@pytest.mark.gpu
@pytest.mark.parametrize("out", ["f32", "bf16", "split"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hd", [64, 128, 256])
def test_attention_fused_gate(hd, dtype, out):
    """Sequences of one token and queries of zeros weigh their key by exactly 1: what is
    left is the output gate, and that is the gate merge's, bit for bit, over the whole
    range."""
    from qdc_amd import ops
    T, H = 300, 2
    g = torch.Generator(device="cuda").manual_seed(hd)
    v = torch.randn((T, H, hd), generator=g, device="cuda").to(dtype)
    gate = torch.empty((T, H, hd), device="cuda").uniform_(-100, 100, generator=g)
    gate[1::2] *= 0.1
    gate[0, 0, :6] = torch.tensor([float("inf"), -float("inf"), float("nan"), 0.0, 89.0, -89.0])
    gate = gate.to(dtype)
    odt = {"f32": torch.float32, "bf16": torch.bfloat16, "split": ops.BF16X2}[out]
    got = ops.attention_fused(torch.zeros_like(v), v, v, gate, None, hd ** -0.5, T, out_dtype=odt)
    want = ops.attention_gate(v.float().view(T, H, 1, hd), gate, out_dtype=odt).view_as(got)
    assert torch.equal(torch.nan_to_num(got, nan=1e30), torch.nan_to_num(want, nan=1e30))


def test_linear_parts_validation():
    lib = _lib.lib()

    def f(out=FAKE, a=BIG, w=BIG, rows=5, inner=128, cols=256, ld_a=128, ld_w=128, parts=2,
          dt=BF16):
        return lib.qdc_linear_parts(out, a, w, rows, inner, cols, ld_a, ld_w, parts, dt, None)

    assert f(dt=F32) == -3
    assert f(inner=96) == -2 and f(cols=192) == -2 and f(ld_a=120) == -2 and f(ld_w=132) == -2
    assert f(parts=0) == -2 and f(parts=3) == -2 and f(inner=32, ld_a=64, dt=BF16) == -2
    assert f(dt=X2) == -2                          # a split row holds 2 inner values
    assert f(a=BIG + 8) == -2 and f(out=FAKE + 4) == -2 and f(rows=1 << 23, ld_a=512) == -2
    assert f(out=None) == -1 and f(a=None) == -1 and f(w=None) == -1
    assert f(a=FAKE + 16) == -5 and f(w=FAKE + 16) == -5
    assert f(rows=0, out=None) == 0

    def g(res=FAKE, normed=FAKE + (1 << 20), x=BIG, sums=BIG, parts=2, norm=BIG, mask=None, rows=5,
          width=256, odt=BF16):
        return lib.qdc_residual_rms_parts(res, normed, x, sums, parts, norm, mask, rows, width,
                                          1e-6, odt, None)

    assert g(odt=7) == -3
    assert g(width=320) == -2 and g(parts=0) == -2 and g(rows=-1) == -2 and g(x=BIG + 4) == -2
    for name in ("res", "normed", "x", "sums", "norm"):
        assert g(**{name: None}) == -1, name
    for name in ("normed", "sums", "norm", "mask"):
        assert g(**{name: FAKE + 16}) == -5, name
    assert g(x=FAKE + 16) == -5 and g(x=FAKE + (1 << 20)) == -5   # x itself is fine for res only
    assert g(rows=0, res=None) == 0


def test_linear_parts_rule():
    """Parts only where a tile's walk is long and the tiles are few; every choice is one
    the entry point takes (at least 4 steps of 64 values a part)."""
    from qdc_amd import ops
    assert ops.linear_parts_for(63, 3584, 1024, True) == 0
    assert ops.linear_parts_for(1200, 2048, 1024, False) == 0
    assert ops.linear_parts_for(16384, 3584, 1024, True) == 0
    assert ops.linear_parts_for(1200, 3584, 1000, True) == 0
    assert ops.linear_parts_for(1200, 3584, 1024, True) == 4
    for rows in (64, 129, 700, 1601):
        for inner in (32, 64, 96, 480, 2048, 3072, 3584):
            for split in (False, True):
                parts = ops.linear_parts_for(rows, inner, 1024, split)
                slots = inner * (2 if split else 1)
                assert parts == 0 or (slots % 64 == 0 and (parts == 1 or slots // 64 >= 4 * parts))


@pytest.mark.parametrize("split", [False, "mlp", "all"])
@pytest.mark.parametrize("hidden,inner,vw", [(1024, 3584, 2048), (1024, 3072, 3072), (768, 3584, 2048),
                                             (256, 768, 1536)])
def test_rows_kept_where_the_rule_cuts(hidden, inner, vw, split):
    """A model holds a projection into the residual stream in the checkpoint's layout,
    beside the transposed one, only where some row count reads it, and as its own
    copy."""
    from qdc_amd import backbone, config, ops, weights
    cfg = config.BackboneConfig(hidden=hidden, head_dim=64, heads=vw // 64, kv_heads=1, key_heads=1,
                                value_heads=vw // 64, key_dim=64, value_dim=64, eps=1e-6,
                                rope_theta=1e7, rotary_dim=16, intermediate=inner, vocab=8,
                                layer_types=("linear_attention", "full_attention"))
    w = {n: torch.zeros(s, dtype=torch.bfloat16) for n, s in weights.all_shapes(cfg).items()}
    model = backbone.QwenBackbone.from_weights(w, cfg, "cpu", torch.bfloat16, split_gemm_inputs=split)
    for i, layer in enumerate(model.layers):
        for key, name, width, two in (
                ("down", "mlp.down_proj", inner, bool(split)),
                ("out", ("linear_attn.out_proj", "self_attn.o_proj")[i], vw, split == "all")):
            ever = any(ops.linear_parts_for(rows, width, hidden, two) for rows in range(1, 4000))
            assert (key + "_rows" in layer) == ever
            if ever:
                rows = layer[key + "_rows"]
                src = w[f"layers.{i}.{name}.weight"]
                assert rows.shape == (hidden, width) and rows.data_ptr() != src.data_ptr()


# rows around a tile of 128 and its wavefronts' 64; parts that do not divide the steps
LINEAR = [(1, 64, 256, 1), (33, 128, 256, 2), (63, 320, 512, 3), (64, 1024, 1024, 8),
          (65, 448, 2048, 7), (127, 192, 1024, 2), (128, 64, 512, 1), (129, 576, 256, 4),
          (300, 704, 1024, 5)]


@pytest.mark.gpu
@pytest.mark.parametrize("out", ["f32", "bf16", "split"])
@pytest.mark.parametrize("split_a", [False, True])
@pytest.mark.parametrize("rows,inner,width,parts", LINEAR)
def test_linear_residual_rms_edges(rows, inner, width, parts, split_a, out):
    """Against 64 bits on the same bf16 values: products are exact in fp32, so the
    residual stream is within fp32 sums of it (1e-5), the norm within that and its
    own rounding (bf16 2^-8 per element)."""
    from qdc_amd import ops
    g = torch.Generator(device="cuda").manual_seed(rows + inner)

    def randn(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    x, w = randn(rows, width), (randn(width, inner) * 0.1).bfloat16()
    a = randn(rows, inner)
    if split_a:
        hi = a.bfloat16()
        lo = (a - hi.float()).bfloat16()
        a = torch.stack([hi.view(rows, -1, 4), lo.view(rows, -1, 4)], 2).reshape(rows, 2 * inner)
        exact_a = ops.join_split(a).double()
    else:
        a = a.bfloat16()
        exact_a = a.double()
    wide = torch.full((rows, a.shape[1] + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[:, :a.shape[1]] = a
    norm = randn(width) * 0.1
    norm = norm if out == "f32" else norm.bfloat16()
    mask = (torch.rand(rows, generator=g, device="cuda") > 0.3).int()
    res, normed = ops.linear_residual_rms(x, wide[:, :a.shape[1]], w, norm, 1e-6, parts,
                                          token_mask=mask,
                                          out_dtype=ops.BF16X2 if out == "split" else None)
    exact = x.double() + exact_a @ w.double().t()
    assert ((res.double() - exact).abs() <= 1e-5 * exact.abs().max()).all()
    want = exact * torch.rsqrt(exact.square().mean(-1, keepdim=True) + 1e-6)
    want = want * (1.0 + norm.double()) * mask[:, None]
    got = (ops.join_split(normed) if out == "split" else normed).double()
    rel = 2.0 ** -8 if out == "bf16" else 2.0 ** -16
    assert ((got - want).abs() <= rel * want.abs() + 2e-5).all()
    plain = ops.linear_residual_rms(x, a, w, norm, 1e-6, parts,
                                    out_dtype=ops.BF16X2 if out == "split" else None)
    assert torch.equal(plain[0], res)
    assert torch.equal(plain[1][mask.bool()], normed[mask.bool()])
    assert not normed[~mask.bool()].any()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_forward_takes_unaligned_weights(dtype):
    """Weights that are views into one buffer, not on 16 bytes, as a checkpoint reader
    may hand them over: a forward at a size of the cut product (bf16) and of the small
    fp32 products gives what aligned weights give, up to the order of sums (one bf16
    rounding, 2^-8, may go the other way)."""
    from qdc_amd import backbone, config, ops, weights
    inner = 3072 if dtype == torch.bfloat16 else 512
    cfg = config.BackboneConfig(hidden=256, head_dim=64, heads=4, kv_heads=1, key_heads=2, value_heads=2,
                                key_dim=64, value_dim=64, eps=1e-6, rope_theta=1e7, rotary_dim=16,
                                intermediate=inner, vocab=64,
                                layer_types=("linear_attention", "full_attention"))
    if dtype == torch.bfloat16:
        assert ops.linear_parts_for(70, inner, 256, False)
    aligned = weights.random_device_weights(cfg, seed=5, dtype=dtype, std=0.05)
    flat = torch.empty(sum(t.numel() + 8 for t in aligned.values()) + 8, dtype=dtype, device="cuda")
    shifted, at = {}, 1
    for name, t in aligned.items():
        shifted[name] = flat[at:at + t.numel()].view(t.shape).copy_(t)
        at += (t.numel() + 7) // 8 * 8
    assert all(t.data_ptr() % 16 for t in shifted.values())
    ids = torch.arange(70, dtype=torch.int32, device="cuda").remainder(64).view(1, 70)
    states = [backbone.batch_backbone_states(backbone.QwenBackbone.from_weights(w, cfg, "cuda", dtype),
                                             ids, None) for w in (aligned, shifted)]
    bar = 1e-5 if dtype == torch.float32 else 2.0 ** -8
    assert normwise(states[1].cpu().numpy(), states[0].cpu().numpy()) <= bar


def test_linear_f32_validation():
    lib = _lib.lib()
    FAR = FAKE + (1 << 30)

    def f(out=FAKE, res=FAR, a=BIG, b=BIG, norm=BIG, mask=None, w=BIG, rows=5, inner=256, cols=128,
          head=128, ld_a=256, ld_b=256, ld_w=256, ld_out=128, inp=1, swiglu=0):
        return lib.qdc_linear_f32(out, res, a, b, norm, mask, w, rows, inner, cols, head, ld_a, ld_b,
                                  ld_w, ld_out, 1e-6, inp, swiglu, None)

    assert f(inp=3) == -4 and f(inp=-1) == -4
    assert f(inner=192) == -2 and f(cols=96) == -2 and f(ld_a=252) == -2 and f(ld_b=254) == -2
    assert f(ld_w=124) == -2 and f(ld_out=124) == -2 and f(swiglu=1, ld_w=252) == -2
    assert f(inp=2, head=96) == -2 and f(inp=2, swiglu=1) == -2 and f(inp=2, head=512) == -2
    assert f(a=BIG + 4) == -2 and f(res=FAR + 8) == -2 and f(mask=BIG + 1) == -2
    for name in ("out", "res", "a", "b", "norm", "w"):
        assert f(**{name: None}) == -1, name
    for name in ("res", "a", "b", "norm", "mask", "w"):
        assert f(**{name: FAKE + 16}) == -5, name
    for name in ("a", "b", "norm", "mask", "w"):
        assert f(**{name: FAR + 16}) == -5, name
    assert f(rows=0, out=None) == 0


def test_linear_f32_ignores_unused_pointers():
    """Pointers an input does not use are ignored, wherever they point: the calls get as
    far as the overlap of out and a (-5)."""
    lib = _lib.lib()
    odd = BIG + 1
    for inp, res, b, norm, mask in ((0, odd, odd, odd, odd), (2, odd, BIG, BIG, odd)):
        assert lib.qdc_linear_f32(FAKE, res, FAKE + 16, b, norm, mask, BIG, 5, 256, 128, 128, 256, 256,
                                  256, 128, 1e-6, inp, 0, None) == -5, inp
    assert lib.qdc_linear_f32(FAKE, FAKE + (1 << 30), FAKE + 16, BIG, BIG, odd, BIG, 5, 256, 128, 128,
                              256, 256, 256, 128, 1e-6, 1, 0, None) == -2


LINEAR_F32 = [(1, 128, 64), (15, 256, 128), (16, 512, 64), (17, 256, 1792), (64, 512, 256),
              (129, 128, 192), (411, 256, 512)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["rows", "rows_glu", "norm", "norm_masked", "norm_glu", "gated"])
@pytest.mark.parametrize("rows,inner,cols", LINEAR_F32)
def test_linear_f32_edges(rows, inner, cols, kind):
    """Against 64 bits: fp32 sums of at most 512 products and the row operators' own
    rounding, the repository's fp32 bar of 1e-5 per call and per largest element."""
    from qdc_amd import ops
    g = torch.Generator(device="cuda").manual_seed(rows + inner + cols)

    def randn(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    def strided(t):  # rows inside wider rows
        wide = torch.full((t.shape[0], t.shape[1] + 12), float("nan"), device="cuda")
        wide[:, 4:4 + t.shape[1]] = t
        return wide[:, 4:4 + t.shape[1]]

    glu = kind.endswith("glu")
    a, b, w = randn(rows, inner), randn(rows, inner), randn(inner, (2 if glu else 1) * cols) * 0.1
    x, residual = a.double(), None
    if kind.startswith("norm"):
        weight, mask = randn(inner) * 0.1, None
        if kind == "norm_masked":
            mask = (torch.rand(rows, generator=g, device="cuda") > 0.4).int()
        residual, got = ops.linear_f32(strided(a), w, add=strided(b), weight=weight, eps=1e-6,
                                       token_mask=mask, swiglu=glu)
        assert torch.equal(residual, a + b)
        x = (a + b).double()
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * (1.0 + weight.double())
        x = x if mask is None else x * mask[:, None]
    elif kind == "gated":
        weight = randn(128 if inner > 128 else 64) + 1.0
        got = ops.linear_f32(strided(a), w, z=strided(b), weight=weight, eps=1e-6)
        heads = x.view(rows, -1, weight.numel())
        heads = heads * torch.rsqrt(heads.square().mean(-1, keepdim=True) + 1e-6) * weight.double()
        x = heads.reshape(rows, inner) * torch.nn.functional.silu(b.double())
    else:
        got = ops.linear_f32(strided(a), w, swiglu=glu)
    want = x @ w.double()
    if glu:
        want = torch.nn.functional.silu(want[:, :cols]) * want[:, cols:]
    err = (got.double() - want)
    assert err.norm() <= 1e-5 * want.norm()
    assert err.abs().max() <= 1e-5 * want.abs().max()
