"""GPU parity at the sizes where launch plans change: remainders of tiles,
splits and waves, and the smallest and largest of each plan's range, against
the CPU oracle (tests/util.py's tolerances) or a float64 product of the same
operands."""
from __future__ import annotations

import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from rxq4 import capi
from tests import kquant_blocks as kb
from tests import util

pytestmark = pytest.mark.gpu


def dev(a: np.ndarray) -> torch.Tensor:
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).cuda()


def host16(t: torch.Tensor) -> np.ndarray:
    return t.cpu().view(torch.int16).numpy().view(np.uint16)


# ------------------------------------------------- long rows, idle last waves
# Rows of more than 64 slots whose waves hold more than 16 KB: the rows of the
# ranges give 1022, 1021 and 1022 waves, so the last workgroup of four has
# waves without rows.  (Parity: what those waves load is discarded; that it lies
# in range 0 is tests/test_gemv_units.py's, on the CPU.)
@pytest.mark.parametrize("rows,K", [((2503, 2604), 13824), ((5101,), 13824), ((1, 5099, 3), 13824)])
def test_long_rows_with_idle_waves(rows, K):
    x = util.x_f16(7001, K)
    Ws = [util.weights(7002 + i, M, K) for i, M in enumerate(rows)]
    ys = [torch.empty(M, dtype=torch.float16, device="cuda") for M in rows]
    capi.gemv_multi_f16([(y, dev(W), M) for y, W, M in zip(ys, Ws, rows)], dev(x), K)
    for y, W, M in zip(ys, Ws, rows):
        pick = np.unique(np.r_[0, M // 2, max(0, M - 40):M])
        ref = orc.gemv_f64(np.ascontiguousarray(W[pick]), K, orc.bits_f16(x).astype(np.float32))
        assert util.rounded_ok(host16(y)[pick], ref).all(), (rows, M)


# ------------------------------------------------------------ prefill attention
def attention64(q, k, v, H, KV, D, N, start, scale, ks=None, vs=None):
    """float64 attention of the same operands on the GPU: [N, H * D]."""
    kk, vv = k.double(), v.double()
    if ks is not None:
        kk, vv = kk * ks.double()[:, :, None], vv * vs.double()[:, :, None]
    out = torch.empty((N, H, D), dtype=torch.float64, device="cuda")
    qq = q.double().view(N, H, D)
    hidden = torch.arange(start + N, device="cuda")[None, :] > start + torch.arange(N, device="cuda")[:, None]
    for h in range(H):
        s = (qq[:, h].contiguous() @ kk[:, h // (H // KV)].t().contiguous()) * scale
        s.masked_fill_(hidden, float("-inf"))
        out[:, h] = torch.softmax(s, 1) @ vv[:, h // (H // KV)].contiguous()
    return out.view(N, H * D)


# (heads, KV heads, head_dim, tokens, cached positions, int8): split over KV
# chunks (long contexts; chunks past early blocks' ends) and unsplit, query
# row blocks of 128 exactly full, one row over and one short, groups that are
# no power of two, several blocks per KV head, every padded head size and
# sizes inside the padding, the first and last position of a 64-position tile.
PREFILL = [
    (32, 8, 128, 2, 4000, False), (32, 8, 128, 45, 8000, False), (32, 8, 128, 45, 4096, "scales"),
    (16, 4, 128, 32, 2015, False), (16, 4, 128, 33, 1983, False), (4, 4, 128, 127, 1000, False),
    (4, 4, 128, 129, 960, False), (35, 7, 128, 61, 1500, False), (14, 2, 64, 50, 3001, False),
    (32, 8, 128, 1100, 0, False), (8, 2, 64, 900, 63, "plain"), (64, 8, 64, 700, 1, False),
    (4, 2, 80, 200, 777, False), (6, 2, 96, 70, 64, False), (4, 1, 96, 19, 5000, "scales"),
    (4, 2, 72, 65, 128, False), (4, 4, 40, 33, 300, False), (2, 2, 8, 17, 100, False),
    (8, 4, 256, 40, 900, False), (3, 1, 256, 90, 65, "scales"), (5, 1, 136, 31, 2000, False),
    (8, 1, 16, 3, 70, "plain"),
    # the VALU kernel's side of its line and the other: 2, 4 and 7 heads a group
    # (four workgroups' worth of heads past 128 dims), one round of workgroups and
    # more, int8
    (32, 8, 80, 16, 40, False), (32, 8, 80, 3, 200, False), (5, 1, 256, 68, 0, False), (5, 1, 256, 68, 200, False),
    (4, 4, 96, 68, 0, "scales"), (4, 4, 96, 200, 0, False), (4, 4, 80, 128, 0, False), (16, 8, 80, 57, 31, "scales"), (14, 2, 160, 9, 60, "scales"), (4, 2, 72, 129, 0, False),
]


@pytest.mark.parametrize("H,KV,D,N,start,i8", PREFILL)
def test_prefill_attention_ranges(H, KV, D, N, start, i8):
    print(f"prefill H={H} KV={KV} D={D} N={N} start={start} int8={i8}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(7100 + N + D)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    S = start + N
    q = rnd(N, H * D).half()
    ks = vs = None
    if i8:
        k, v = (rnd(S, KV, D).mul(40).round().clamp(-127, 127).to(torch.int8) for _ in range(2))
        if i8 == "scales":
            ks, vs = (rnd(S, KV).abs() * 0.01 + 0.005 for _ in range(2))
    else:
        k, v = rnd(S, KV, D).half(), rnd(S, KV, D).half()
    one = D ** -0.5 * (0.03 if i8 == "plain" else 1.0)
    for scale in (one, -one, 0.0):  # a negative scale turns the order round, 0 gives means
        out = torch.full((N, H * D), float("nan"), dtype=torch.float16, device="cuda")
        capi.attention_prefill_f16(out, q, k, v, H, KV, D, N, start, scale, bool(i8), ks, vs)
        ref = attention64(q, k, v, H, KV, D, N, start, scale, ks, vs).cpu().numpy()
        for a in range(0, N, 16):  # the bar of tests/test_gpu_attn.py, per few rows
            assert util.rel_err(out[a:a + 16].float().cpu().numpy(), ref[a:a + 16]) <= util.TOL, (scale, a)
        assert util.rounded_ok(host16(out).reshape(ref.shape), ref).all(), scale


def aligned_inputs(H, KV, D, N, S, height, g, i8):
    """q, K, V (fp16, or int8 K and V with K scales) whose scores at scale 1 / D
    are close to height[pos] * a for query rows of a = 0.5 .. 2: every query row
    and K row is a multiple of one +-1 vector of its KV head, with some noise.
    V is positive, so that no output is a small difference."""
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    u = torch.sign(rnd(KV, D))
    a = torch.exp2(torch.rand(N, H, 1, generator=g, device="cuda") * 2 - 1)
    q = (a * u.repeat_interleave(H // KV, 0) + 0.02 * rnd(N, H, D)).half().view(N, H * D)
    if not i8:
        return q, (height.view(-1, 1, 1) * u + 0.02 * rnd(S, KV, D)).half(), (rnd(S, KV, D).abs() + 0.5).half(), None
    k = (u * 60 + rnd(S, KV, D)).round().clamp(-127, 127).to(torch.int8)
    v = (rnd(S, KV, D).abs() * 20 + 10).round().clamp(0, 127).to(torch.int8)
    return q, k, v, (height.view(-1, 1) / 60).expand(S, KV).contiguous()


# Where the query rows split over the KV chunks and where they do not, both wave
# groups, every padded head size.
DIMS = [(16, 4, 128, 45, 4000), (32, 8, 128, 1100, 0), (4, 2, 80, 70, 500), (8, 2, 64, 40, 3000), (6, 2, 96, 130, 900),
        (4, 1, 256, 40, 2000)]


@pytest.mark.parametrize("i8", [False, True])
@pytest.mark.parametrize("H,KV,D,N,start", DIMS)
def test_prefill_attention_rising_scores(H, KV, D, N, start, i8):
    """Scores that rise along the positions, by more than 2^4 in some tiles, by
    less in others and differently for each row, and one late key above all:
    every move of a row's reference point, in walks, wave groups and chunks."""
    print(f"rising scores H={H} KV={KV} D={D} N={N} start={start} int8={i8}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(7110 + D)
    S = start + N
    tile = torch.arange(S, device="cuda") // 64
    step = torch.tensor([0.0, 3.0, 0.5, -6.0, 4.5, 0.0, 2.0], device="cuda")
    height = step[tile % 7].masked_fill(torch.arange(S, device="cuda") % 64 != 5, 0.0).cumsum(0)
    height = height / max(1.0, float(height.max()) / 24)
    for late in (False, True):
        if late:
            height[S * 3 // 4] = float(height.max()) + 9
        q, k, v, ks = aligned_inputs(H, KV, D, N, S, height, g, i8)
        vs = torch.rand(S, KV, generator=g, device="cuda") * 0.02 + 0.005 if i8 else None
        out = torch.full((N, H * D), float("nan"), dtype=torch.float16, device="cuda")
        capi.attention_prefill_f16(out, q, k, v, H, KV, D, N, start, 1.0 / D, i8, ks, vs)
        ref = attention64(q, k, v, H, KV, D, N, start, 1.0 / D, ks, vs).cpu().numpy()
        assert util.rounded_ok(host16(out).reshape(ref.shape), ref).all(), late


@pytest.mark.parametrize("H,KV,D,N,start", DIMS)
def test_prefill_attention_small_probabilities(H, KV, D, N, start):
    """One position 2^26 above the rest whose V row is 0: what is left is made of
    probabilities below fp16's smallest."""
    print(f"small probabilities H={H} KV={KV} D={D} N={N} start={start}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(7120 + D)
    S = start + N
    height = torch.zeros(S, device="cuda")
    height[S // 3] = 26.0 * 0.6931
    q, k, v, _ = aligned_inputs(H, KV, D, N, S, height, g, False)
    q = torch.sign(q)  # every row's a is 1
    v *= 64
    v[S // 3] = 0
    out = torch.full((N, H * D), float("nan"), dtype=torch.float16, device="cuda")
    capi.attention_prefill_f16(out, q, k, v, H, KV, D, N, start, 1.0 / D)
    ref = attention64(q, k, v, H, KV, D, N, start, 1.0 / D).cpu().numpy()
    sees = slice(max(0, S // 3 - start), N)
    # 2^-11: half a unit of an fp16 output and as much again for the sums
    assert util.rounded_ok(host16(out).reshape(ref.shape)[sees], ref[sees], delta=2.0 ** -12).all()


@pytest.mark.parametrize("size", ["1e-6", "1e-4", "3e4", "mixed", "zeros"])
@pytest.mark.parametrize("H,KV,D,N,start", DIMS)
def test_prefill_attention_v_scales(H, KV, D, N, start, size):
    """int8 caches whose V scales are far from 1, with one position above the
    rest by up to 2^24: the probabilities keep their precision and, where it is
    below 2^4 and the reference point of the exponentials stays, their range."""
    print(f"V scales {size} H={H} KV={KV} D={D} N={N} start={start}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(7130 + D)
    S = start + N
    height = torch.rand(S, generator=g, device="cuda")
    height[S // 3] += (1.4 if size == "3e4" else 12) * 0.6931
    q, k, v, ks = aligned_inputs(H, KV, D, N, S, height, g, True)
    vs = torch.rand(S, KV, generator=g, device="cuda") + 0.5
    if size == "mixed":  # over 2^16 in every tile
        vs *= torch.exp2(torch.rand(S, KV, generator=g, device="cuda") * 16 - 14)
        vs *= torch.sign(torch.rand(S, KV, generator=g, device="cuda") - 0.05)
    elif size == "zeros":
        vs[: S // 2] = 0
    else:
        vs *= float(size)
        if size == "3e4":
            v = v % 2  # the outputs are fp16
    out = torch.full((N, H * D), float("nan"), dtype=torch.float16, device="cuda")
    capi.attention_prefill_f16(out, q, k, v, H, KV, D, N, start, 1.0 / D, True, ks, vs)
    ref = attention64(q, k, v, H, KV, D, N, start, 1.0 / D, ks, vs).cpu().numpy()
    assert util.rounded_ok(host16(out).reshape(ref.shape), ref).all()


@pytest.mark.parametrize("what", ["nan", "inf", "-inf", "k", "scale", "k scale"])
@pytest.mark.parametrize("H,KV,D,N,start", DIMS + [(2, 2, 80, 64, 500), (8, 1, 144, 200, 0), (4, 4, 48, 300, 1),
                                                  (32, 8, 128, 45, 8000)])
def test_prefill_attention_is_causal(H, KV, D, N, start, what):
    """Infinities and NaN in the caches reach the tokens that see them and no
    other: the earlier tokens' rows (and dims) are those of a clean cache."""
    print(f"causal {what} H={H} KV={KV} D={D} N={N} start={start}", flush=True)
    i8 = "scale" in what
    g = torch.Generator(device="cuda").manual_seed(7140 + D + N)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    S = start + N
    q, scale = rnd(N, H * D).half(), D ** -0.5
    if i8:
        k, v = (rnd(S, KV, D).mul(40).round().clamp(-127, 127).to(torch.int8) for _ in range(2))
        ks, vs = (rnd(S, KV).abs() * 0.01 + 0.02 for _ in range(2))
    else:
        k, v, ks, vs = rnd(S, KV, D).half(), rnd(S, KV, D).half(), None, None
    clean = torch.empty((N, H * D), dtype=torch.float16, device="cuda")
    capi.attention_prefill_f16(clean, q, k, v, H, KV, D, N, start, scale, i8, ks, vs)
    for token in sorted({0, 1, N // 2, N - 2, N - 1} & set(range(N))):
        p = start + token
        bk, bv, bks, bvs = (None if t is None else t.clone() for t in (k, v, ks, vs))
        dims = slice(0, D)
        if what == "k":
            bk[p, 0, D // 2] = float("nan")
        elif what == "scale":
            bvs[p, 0] = float("nan")
            bvs[p + 1:, 0] = float("inf")
        elif what == "k scale":
            bks[p, 0] = float("nan")
        else:
            dims = slice(3, 6)
            bv[p, 0, dims] = float(what)
        out = torch.full_like(clean, float("nan"))
        capi.attention_prefill_f16(out, q, bk, bv, H, KV, D, N, start, scale, i8, bks, bvs)
        o, c = out.view(N, H, D), clean.view(N, H, D)
        assert torch.equal(o[:token], c[:token])
        assert torch.equal(o[:, H // KV:], c[:, H // KV:])  # the other KV heads
        hit = o[token:, : H // KV, dims]
        assert not torch.isfinite(hit).any()
        rest = [d for d in range(D) if not dims.start <= d < dims.stop]
        assert torch.equal(o[token:, : H // KV, rest], c[token:, : H // KV, rest])


def test_prefill_attention_split_in_a_graph():
    """A split prefill captured on a stream without a workspace, replayed with
    other work between: every replay equals the eager result."""
    H, KV, D, N, start = 32, 8, 128, 20, 3000
    g = torch.Generator(device="cuda").manual_seed(7200)
    q = torch.randn(N, H * D, generator=g, device="cuda").half()
    k, v = (torch.randn(start + N, KV, D, generator=g, device="cuda").half() for _ in range(2))
    eager = torch.empty_like(q)
    capi.attention_prefill_f16(eager, q, k, v, H, KV, D, N, start, D ** -0.5)
    out = torch.empty_like(q)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        capi.attention_prefill_f16(out, q, k, v, H, KV, D, N, start, D ** -0.5)
    other = torch.empty_like(q)
    for _ in range(3):
        out.zero_()
        graph.replay()
        capi.attention_prefill_f16(other, q, k, v, H, KV, D, N, start // 2, D ** -0.5)
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    capi.release_workspace(stream)


def check_valu_attention():
    """Every kernel of RXQ4_ATTN_MFMA=0, in a process of its own."""
    g = torch.Generator(device="cuda").manual_seed(7250)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    for H, KV, D, N, start, i8 in [(32, 8, 128, 45, 100, False), (7, 1, 64, 130, 0, True), (4, 4, 128, 3, 700, True),
                                   (16, 1, 64, 20, 63, False), (8, 4, 256, 33, 200, False)]:
        q, ks, vs = rnd(N, H * D).half(), None, None
        if i8:
            k, v = (rnd(start + N, KV, D).mul(40).round().clamp(-127, 127).to(torch.int8) for _ in range(2))
            ks, vs = (rnd(start + N, KV).abs() * 0.01 + 0.005 for _ in range(2))
        else:
            k, v = rnd(start + N, KV, D).half(), rnd(start + N, KV, D).half()
        out = torch.full((N, H * D), float("nan"), dtype=torch.float16, device="cuda")
        capi.attention_prefill_f16(out, q, k, v, H, KV, D, N, start, D ** -0.5, i8, ks, vs)
        ref = attention64(q, k, v, H, KV, D, N, start, D ** -0.5, ks, vs).cpu().numpy()
        assert util.rounded_ok(host16(out).reshape(ref.shape), ref).all(), (H, KV, D, N, start, i8)


def test_valu_attention_for_every_shape():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = ("import sys; sys.path[:0] = [%r, %r]\nfrom tests import test_gpu_ranges as t\n"
            "t.check_valu_attention()\nprint('valu ok')\n" % (root, os.path.join(root, "reflex-infer_amd")))
    p = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, RXQ4_ATTN_MFMA="0"), capture_output=True,
                       text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-2000:]
    assert "valu ok" in p.stdout


# ------------------------------------------------------- 17..64 token products
# Token tiles of 32 and 64 on 128-row tiles (two wave groups share K) and, from
# 64 row tiles of 64 rows, on 64-row tiles (four groups): groups without
# super-blocks (K of one to three), uneven parts, K splits, partial row tiles,
# rows that no vector store covers, the first and last token count of a tile.
SHORT = [(12, 1, 17, 4352), (12, 130, 32, 4608), (12, 4700, 33, 512), (12, 3100, 64, 768), (12, 3075, 45, 2048),
         (12, 64, 20, 11008), (12, 9217, 17, 256), (12, 4100, 31, 1280), (12, 4101, 47, 256), (12, 4160, 64, 2816),
         (13, 130, 17, 5376), (13, 1400, 50, 2304), (13, 4099, 64, 768), (13, 200, 60, 5120), (13, 3000, 64, 256),
         (14, 1, 64, 4352), (14, 9300, 32, 768), (14, 1400, 33, 2304), (14, 6000, 17, 1280), (14, 60, 64, 11008),
         (14, 2400, 64, 256)]


def product_case(t, M, N, K, dt, seed):
    Wn = util.weights(seed, M, K) if t == 12 else kb.random_blocks(t, util.rng(seed), M, K)
    x32 = util.gaussian(seed + 1, (N, K))
    if dt == "bf16":
        bits = util.f32_to_bf16_bits(x32)
        x, xf = dev(bits).view(torch.bfloat16), orc.bits_bf16_to_f32(bits)
    else:
        bits = x32.astype(np.float16).view(np.uint16)
        x, xf = dev(bits).view(torch.float16), orc.bits_f16(bits).astype(np.float32)
    rows = np.unique(np.r_[0, np.arange(max(0, M - 40), M), util.rng(seed + 2).choice(M, min(M, 60), replace=False)])
    sub = np.ascontiguousarray(Wn[rows])
    ref = orc.gemm_f64(sub, K, xf, dt) if t == 12 else orc.kq_gemm_f64(sub, K, t, xf, dt)
    return dev(Wn), x, rows, ref


def check_product(call, W, x, rows, ref, t, M, N, K, dt):
    y = torch.full((N, M), float("nan"), dtype=torch.float32, device="cuda")
    call(y, W, x, M, N, K, ggml_type=t)
    assert util.rel_err(y.cpu().numpy()[:, rows], ref) <= util.TOL
    assert torch.isfinite(y).all()
    y16 = torch.empty((N, M), dtype=x.dtype, device="cuda")
    call(y16, W, x, M, N, K, ggml_type=t)
    assert util.rounded_ok(host16(y16)[:, rows], ref, dt).all()


@pytest.mark.parametrize("t,M,N,K", SHORT)
def test_short_prompt_products(t, M, N, K):
    print(f"short prompt type {t} [{M} x {K}] x {N}", flush=True)
    for dt in ("f16", "bf16"):
        case = product_case(t, M, N, K, dt, 7300 + M + N)
        check_product(capi.gemm, *case, t, M, N, K, dt)
        check_product(capi.gemm_noalloc, *case, t, M, N, K, dt)


# Small matrices, 16-token chunks: the last and first sizes of the rule (576
# workgroups of up to 8 super-blocks, 256 of up to 16), partial chunks and row
# tiles, many chunks.
CHUNKS = [(12, 256, 17, 2048), (12, 255, 500, 512), (12, 1, 1000, 256), (12, 1024, 144, 1024), (12, 1040, 144, 1024),
          (12, 1024, 64, 4096), (12, 1040, 64, 4096), (13, 130, 200, 2048), (13, 2303, 64, 768), (14, 256, 45, 2048),
          (14, 100, 333, 1280), (14, 2304, 49, 512), (14, 33, 129, 4096)]


@pytest.mark.parametrize("t,M,N,K", CHUNKS)
def test_small_matrices_in_chunks(t, M, N, K):
    print(f"chunks type {t} [{M} x {K}] x {N}", flush=True)
    for dt in ("f16", "bf16"):
        case = product_case(t, M, N, K, dt, 7450 + M + N)
        check_product(capi.gemm, *case, t, M, N, K, dt)
        check_product(capi.gemm_noalloc, *case, t, M, N, K, dt)


# 64-token tiles on more than 64 tokens: the last and first row and token counts
# of one round (256 tiles), the longest rows of the rule and the next, a last token
# tile of one token, a last row tile of one row.
MID = [(12, 8192, 65, 256), (12, 8193, 128, 512), (12, 4097, 130, 2048), (12, 2600, 384, 512), (12, 1025, 193, 4096),
       (12, 200, 321, 4352), (13, 1100, 450, 768), (13, 2049, 192, 3072), (13, 300, 257, 3328), (14, 8192, 128, 256),
       (14, 1601, 129, 2304), (14, 500, 640, 3072), (14, 65, 300, 3328)]


@pytest.mark.parametrize("t,M,N,K", MID)
def test_mid_prompt_products(t, M, N, K):
    print(f"mid prompt type {t} [{M} x {K}] x {N}", flush=True)
    for dt in ("f16", "bf16"):
        case = product_case(t, M, N, K, dt, 7600 + M + N)
        check_product(capi.gemm, *case, t, M, N, K, dt)
        check_product(capi.gemm_noalloc, *case, t, M, N, K, dt)


# Q4_K batches around the row counts from which x is staged in LDS.
STAGED = [(12, 8192, 5, 768), (12, 8193, 4, 768), (12, 8193, 8, 2048), (12, 5056, 16, 512), (12, 5057, 9, 512),
          (12, 5060, 16, 3840), (12, 9000, 3, 256)]


@pytest.mark.parametrize("t,M,N,K", STAGED)
def test_q4k_batches_staged(t, M, N, K):
    print(f"batch [{M} x {K}] x {N}", flush=True)
    for dt in ("f16", "bf16"):
        case = product_case(t, M, N, K, dt, 7350 + M + N)
        if dt == "f16" and util.gemv_path(N, M, K):
            continue
        check_product(capi.gemm, *case, t, M, N, K, dt)


# Q5_K / Q6_K batches whose rows are split over workgroups (20 blocks a row and
# up; parts of 2 to 11 blocks, the last one short), the largest unsplit row,
# and Q5_K batches large enough for the 32-token tiles.
BATCH = [(14, 100, 2, 5120), (14, 33, 16, 11008), (13, 33, 5, 11008), (13, 16, 16, 5376), (14, 64, 7, 4864),
         (14, 2049, 3, 5120), (13, 12501, 2, 4096), (13, 12500, 16, 4096)]


@pytest.mark.parametrize("t,M,N,K", BATCH)
def test_kquant_batches_split_and_large(t, M, N, K):
    print(f"kquant batch type {t} [{M} x {K}] x {N}", flush=True)
    for dt in ("f16", "bf16"):
        case = product_case(t, M, N, K, dt, 7400 + M + N)
        check_product(capi.gemm, *case, t, M, N, K, dt)
        check_product(capi.gemm_noalloc, *case, t, M, N, K, dt)


# --------------------------------------------------- decode GEMV, row groups
# 8, 16 and 32 lanes a row: partial last groups of rows, steps past a row's
# slots (a multiple of 4 only), several groups a wave, ranges of a pair and a
# triple ending inside a group, 1 to 4 tokens, the residual in place (70001 rows:
# more than 64 of them a wave).
ROWS = [((5120,), 5120), ((27649,), 1280), ((17919,), 1536), ((1537,), 1536), ((1536,), 8960), ((4099,), 3584),
        ((2047,), 3072), ((13823, 13825), 768), ((5121, 1, 1023), 5120), ((7, 9, 3), 2816), ((1,), 1792),
        ((37890,), 3584), ((4097,), 14336), ((3,), 65280), ((70001,), 768)]


@pytest.mark.parametrize("rows,K", ROWS)
def test_row_group_gemv(rows, K):
    print(f"row groups {rows} x {K}", flush=True)
    x = util.x_f16(7500, K)
    xd, xf = dev(x).view(torch.float16), orc.bits_f16(x).astype(np.float32)
    Ws = [util.weights(7501 + i, M, K) for i, M in enumerate(rows)]
    Wd = [dev(W) for W in Ws]
    ys = [torch.full((M,), float("nan"), dtype=torch.float16, device="cuda") for M in rows]
    capi.gemv_multi_f16([(y, W, M) for y, W, M in zip(ys, Wd, rows)], xd, K)
    picks = [np.unique(np.r_[0, M // 3, M // 2, np.arange(max(0, M - 70), M)]) for M in rows]
    refs = [orc.gemv_f64(np.ascontiguousarray(W[p]), K, xf) for W, p in zip(Ws, picks)]
    for y, p, ref in zip(ys, picks, refs):
        assert torch.isfinite(y).all()
        assert util.rounded_ok(host16(y)[p], ref).all()
    M, W, p, ref = rows[0], Wd[0], picks[0], refs[0]
    f32 = torch.empty(M, dtype=torch.float32, device="cuda")
    capi.gemv_f32(f32, W, xd, M, K)
    assert util.rel_err(f32.cpu().numpy()[p], ref) <= util.TOL
    res = util.x_f16(7510, M)
    rd = dev(res).view(torch.float16)
    one = torch.empty(M, dtype=torch.float16, device="cuda")
    capi.gemv_f16(one, W, xd, M, K)
    expect = (one.float() + rd.float()).half()  # the product rounded, then the sum
    capi.gemv_add_f16(rd, W, xd, rd, M, K)
    assert torch.equal(rd, expect)
    if K <= 8960:  # every token of a multi-token call equals its own call
        xs = dev(util.x_f16(7520, (3, K))).view(torch.float16)
        for N in (2, 3):
            if not util.gemv_path(N, M, K):
                continue
            many = torch.empty((N, M), dtype=torch.float16, device="cuda")
            capi.gemm_f16(many, W, xs, M, N, K)
            for t in range(N):
                capi.gemv_f16(one, W, xs[t], M, K)
                assert torch.equal(many[t], one), (N, t)


# Q5_K / Q6_K row groups (10240 rows and more; 32, 16 and 8 lanes a row): odd
# row counts, the first row count of the rule, rows on odd 2-byte boundaries.
@pytest.mark.parametrize("t,M,K", [(13, 10240, 2560), (13, 10243, 1536), (14, 10241, 1280), (14, 12345, 1536),
                                   (13, 20001, 3584), (14, 10247, 5120), (13, 11111, 3072), (14, 10241, 256 * 9)])
def test_kquant_row_groups(t, M, K):
    print(f"kquant row groups type {t} [{M} x {K}]", flush=True)
    Wn = kb.random_blocks(t, util.rng(7600 + K), M, K)
    x = util.x_f16(7601, K)
    W, xd = dev(Wn), dev(x).view(torch.float16)
    pick = np.unique(np.r_[0:9, M // 2, np.arange(M - 40, M), util.rng(7602).choice(M, 60, replace=False)])
    ref = orc.kq_gemm_f64(np.ascontiguousarray(Wn[pick]), K, t, orc.bits_f16(x).astype(np.float32)[None], None)[0]
    y = torch.full((M,), float("nan"), dtype=torch.float32, device="cuda")
    capi.gemv_f32(y, W, xd, M, K, ggml_type=t)
    assert torch.isfinite(y).all()
    assert util.rel_err(y.cpu().numpy()[pick], ref) <= util.TOL
    one = torch.empty(M, dtype=torch.float16, device="cuda")
    capi.gemv_f16(one, W, xd, M, K, ggml_type=t)
    assert util.rounded_ok(host16(one)[pick], ref).all()
    res = dev(util.x_f16(7603, M)).view(torch.float16)
    expect = (one.float() + res.float()).half()
    capi.gemv_add_f16(res, W, xd, res, M, K, ggml_type=t)
    assert torch.equal(res, expect)
