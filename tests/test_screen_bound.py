"""The screened pass 1's error bound |a - log-joint| <= E, restated on the CPU: a from operands
rounded to bf16 and summed in float32, E from the float32 norms of the row and the block's
constants as the prologues form them, against the float64 log-joint, over the scales of the
rows and of the components at which both are finite."""

import math

import pytest
import torch

LOG2_E = math.log2(math.e)
LOG_2PI = math.log(2.0 * math.pi)
REL = float.fromhex("0x1.06p-8")   # of a product with an operand rounded to bf16
LIMIT = 1e30                       # constants from which on a component gets no finite bound


def bf16(t):
    return t.float().bfloat16().float()


def split3(t):
    """The nearest sum of three bf16 values."""
    t = t.float()
    a = bf16(t)
    b = bf16(t - a)
    return a.double() + b.double() + bf16(t - a - b).double()


def block_max(t):
    return t.view(-1, 32).max(dim=1).values.repeat_interleave(32)


def weight_error(w, h):
    return (w - h.double()).norm(dim=1) + REL * h.double().norm(dim=1)


def no_bound(A, *norms):
    """|C|, infinite where a constant is not an ordinary number."""
    for t in (A, *norms):
        A = torch.where(t < LIMIT, A, torch.full_like(A, math.inf))
    return A


def screen_iso(X, mu, lss, lpi):
    D = X.shape[1]
    b = 0.5 * torch.exp(-lss.double()) * LOG2_E
    musq = (mu.double() ** 2).sum(1)
    C = (lpi.double() - 0.5 * D * (LOG_2PI + lss.double())) * LOG2_E - b * musq
    x = X.double()
    exact = C - b * (x * x).sum(1)[:, None] + (x @ (2.0 * b[:, None] * mu.double()).t())
    s = (X * X).sum(1)
    w = 2.0 * b[:, None] * mu.double()
    h = bf16(mu * (2.0 * b).float()[:, None])
    a = (bf16(X) @ h.t()).double() + (C.float().double() - split3(s)[:, None] * split3(b))
    A = no_bound(C.abs(), b, h.double().norm(dim=1))
    e = [block_max(t).float() for t in (weight_error(w, h), b * 2.0 ** -14, A * 2.0 ** -14 + 1.0)]
    return exact, a.float(), s.sqrt()[:, None] * e[0] + s[:, None] * e[1] + e[2]


def screen_diag(X, mu, lss, lpi):
    D = X.shape[1]
    w = 0.5 * torch.exp(-lss.double()) * LOG2_E
    v = 2.0 * mu.double() * w
    C = (lpi.double() - 0.5 * (D * LOG_2PI + lss.double().sum(1))) * LOG2_E - (mu.double() ** 2 * w).sum(1)
    x = X.double()
    exact = C - (x * x) @ w.t() + x @ v.t()
    sq = X * X
    a = (bf16(X) @ bf16(v).t()).double() - (bf16(sq) @ bf16(w).t()).double() + C.float().double()
    xs, xq = sq.sum(1), (sq * sq).sum(1)
    ny = torch.where(xq < 2.0 ** -100, xs, xq.sqrt())
    A = no_bound(C.abs(), bf16(w).double().norm(dim=1), bf16(v).double().norm(dim=1))
    e = [block_max(t).float() for t in (weight_error(v, bf16(v)), weight_error(w, bf16(w)), A * 2.0 ** -14 + 1.0)]
    return exact, a.float(), xs.sqrt()[:, None] * e[0] + ny[:, None] * e[1] + e[2]


@pytest.mark.parametrize("model", ["iso", "diag"])
@pytest.mark.parametrize("D", [5, 96])
@pytest.mark.parametrize("sigma", [1e-14, 1e-12, 1e-5, 1.0, 1e6])
def test_bound_holds_at_every_scale(model, D, sigma):
    g = torch.Generator().manual_seed(D)
    N, K = 48, 128
    lpi = torch.log_softmax(torch.randn(K, generator=g), 0)
    base = torch.randn(N, D, generator=g)
    finite = 0
    for far in (0.0, 1.0, 60.0, 1e4):
        mu = 2.0 * torch.randn(K, D, generator=g) * sigma * max(far, 1.0)
        # One variance per component: bf16 roundings that add up over the dimensions.
        lss = (2.0 * torch.rand(K, generator=g) - 1.0) + 2.0 * math.log(sigma)
        if model == "diag":
            lss = lss[:, None].expand(K, D).clone()
        for e in range(-20, 19, 2):
            X = base * 10.0 ** e + mu[torch.randint(0, K, (N,), generator=g)]
            exact, a, E = (screen_iso if model == "iso" else screen_diag)(X, mu, lss, lpi)
            ok = torch.isfinite(E) & torch.isfinite(a)
            err = (a.double() - exact).abs()
            assert bool((err <= E.double())[ok].all()), (far, e, float((err / E)[ok].max()))
            # Beyond float32 the screening sees -inf: so is the log-joint.
            assert bool((exact <= -3e38)[torch.isfinite(E) & ~ok].all()), (far, e)
            finite += int(ok.sum())
    assert finite > 0.2 * 4 * 20 * N * K
