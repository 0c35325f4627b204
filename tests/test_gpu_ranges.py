"""GPU parity at the sizes where launch plans change: remainders of tiles,
splits and waves, and the smallest and largest of each plan's range, against
the CPU oracle (tests/util.py's tolerances) or a float64 product of the same
operands."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from rxq4 import capi
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
# waves without rows (they must not read past range 0).
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
