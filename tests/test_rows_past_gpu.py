"""Row kernels on streams larger than the caches, which they read and write past them: every row as in a launch of few rows."""
import pytest
import torch

from copilot_for_consensus_amd.ops import branch as N
from copilot_for_consensus_amd.ops import gated as G
from copilot_for_consensus_amd.ops import hyper as H
from copilot_for_consensus_amd.ops.cols import Cols

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed=0):
    return torch.randn(*shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed + len(shape)))


def same(a, b):
    """The same sums in the same order, contracted alike or not: a few units of 2^-24 of sums of terms up to 8 (32 bits), half a
    unit of 2^-8 where a bf16 result is rounded the other way."""
    d = (a.float() - b.float()).abs()
    assert float((d / b.float().abs().clamp_min(1.0)).max()) <= (2.0 ** -7 if a.dtype == torch.bfloat16 else 2.0 ** -18)


# a stream of 88 MB and a row more, and less; channels of one and of several vectors a thread
@pytest.mark.parametrize("T,W", [(4096, 4096), (4097, 4096), (2800, 6000), (16400, 1028), (5632, 4096), (5633, 4096), (3900, 6000), (1500, 16384), (22500, 1028)])
@pytest.mark.parametrize("split", [1, 3])
def test_branches(T, W, split):
    few = slice(T - 200, T)
    x, y, g = rnd(T, W), rnd(split, T, W, seed=1), rnd(T, W + 8, seed=2).bfloat16()
    w, b = rnd(W, seed=3), rnd(W, seed=4)
    parts = lambda s: (x[s].clone(), y[:, s].contiguous(), g[s])                       # noqa: E731
    for run in (lambda xs, ys, gs, h: G.gated_norm(xs, G.Branch(Cols(gs[:, :W]), b, w, 1e-5, y=ys), torch.bfloat16, h),
                lambda xs, ys, gs, h: N.branch_norm(xs, N.Branch(w, 1e-5, y=ys), b, 1e-5, h)):
        out = []
        for s in (slice(0, T), few):
            xs, ys, gs = parts(s)
            h = torch.empty(xs.shape, dtype=torch.bfloat16, device=DEV)
            run(xs, ys, gs, h)
            out.append((xs[-200:], h[-200:]))
        same(out[0][0], out[1][0])
        same(out[0][1], out[1][1])


# four streams: of 512 MB and less, of more rows than a launch of few; two and five; past the caches with two and four vectors a thread
@pytest.mark.parametrize("T,W,S", [(8200, 4096, 4), (300, 4096, 4), (16500, 4096, 2), (700, 5000, 3), (300, 4096, 5), (600, 1024, 4), (8200, 8192, 2), (9000, 5000, 3), (4100, 16384, 2)])
def test_streams(T, W, S):
    e, y, y2 = rnd(T, W), rnd(1, T, W, seed=1), rnd(2, T, W, seed=2)
    c = H.Connection(rnd(S, seed=3), rnd(S, S, seed=4), rnd(S, seed=5))
    w = rnd(W, seed=6)
    out = []
    for s in (slice(0, T), slice(T - 200, T)):
        xs = H.Streams(e[s].contiguous(), S)
        xs.done = (y[:, s].contiguous(), c)
        n = xs.e.shape[0]
        u, rstd = torch.empty(n, W, device=DEV), torch.empty(n, device=DEV)
        H.stats(xs, c.inp, 1e-5, u, rstd)
        xs.done = (y2[:, s].contiguous(), c)
        h = H.norm(xs, c.inp, w, 1e-5, torch.empty(n, W, dtype=torch.bfloat16, device=DEV))
        xs.done = (y[:, s].contiguous(), c)
        last = H.last_norm(xs, w, 1e-5, torch.float32)
        out.append([t[-200:] for t in (u, rstd, xs.x, h, last)])
    for a, b in zip(*out):
        same(a, b)
