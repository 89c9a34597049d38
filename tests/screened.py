"""Calls of the isotropic and diagonal E-steps whose route the tests check: inputs, the call
with its workspace, and comparisons with the dense run (the unscreened exact passes)."""

import math

import torch

from flash_gmm import _lib, data, diag_estep_into, iso_estep_into
from parity import assert_close_stats, assert_dense_agrees
from routes import SCREEN, call_mode, listed_rows

KEYS = ("X", "mu", "log_sigma_sq", "log_pi")
INTO = {"iso": iso_estep_into, "diag": diag_estep_into}
CLUSTERED = {"iso": data.iso_clustered, "diag": data.diag_clustered}


def outputs(model, N, K, D, dev):
    return [torch.full((N,), math.nan, device=dev), torch.empty(K, device=dev), torch.empty(K, D, device=dev),
            torch.empty(K, device=dev) if model == "iso" else torch.empty(K, D, device=dev)]


def workspace(model, N, K, D, dev):
    nbytes = getattr(_lib.lib(), f"fgmm_{model}_workspace_bytes")(N, K, D)
    return torch.empty(nbytes, dtype=torch.uint8, device=dev)


def call(model, inp, dev, expect=None, **kw):
    """The default plan's outputs; expect: the route the probe must have chosen."""
    args = [inp[k].to(dev) for k in KEYS]
    N, D = args[0].shape
    K = args[1].shape[0]
    out, ws = outputs(model, N, K, D, dev), workspace(model, N, K, D, dev)
    INTO[model](*args, *out, workspace=ws, **kw)
    torch.cuda.synchronize()
    if expect is not None:
        mode = call_mode(model, ws, N, K, D)
        assert mode == expect, f"{model} N={N} K={K} D={D}: route {mode}, not {expect}"
    return out


def listed(model, inp, dev):
    """(rows a screened call puts on its list, the most that run one tile per workgroup)."""
    args = [inp[k].to(dev) for k in KEYS]
    N, D = args[0].shape
    K = args[1].shape[0]
    out, ws = outputs(model, N, K, D, dev), workspace(model, N, K, D, dev)
    INTO[model](*args, *out, workspace=ws, phase=1)
    torch.cuda.synchronize()
    assert call_mode(model, ws, N, K, D) == SCREEN
    return listed_rows(model, ws, N, K, D)


def check(model, inp, dev, what, oracle):
    """A screened call against the dense run and the oracle, twice the same."""
    print(what, flush=True)
    got = call(model, inp, dev, expect=SCREEN)
    assert_dense_agrees(got, call(model, inp, dev, dense=True), bitwise=False)
    again = call(model, inp, dev)
    assert all(torch.equal(u, v) for u, v in zip(got, again)), f"{what}: not deterministic"
    assert_close_stats(got, oracle(*[inp[k] for k in KEYS]), what)
    return got


def separated(model, N, K, D, seed):
    """The model's clustered rows with centres 1.75 times as far apart: in 31 dimensions, too, a row
    is near one component (and ||x|| no larger than in the others at 128)."""
    g = torch.Generator().manual_seed(seed)
    inp = CLUSTERED[model](8, K, D, seed=seed)   # the parameters' shapes and variances
    c = 3.5 * torch.randn(K, D, generator=g)
    sd = torch.exp(0.5 * inp["log_sigma_sq"].double()).float()
    a = torch.randint(0, K, (N,), generator=g)
    z = torch.randn(N, D, generator=g)
    inp["X"] = c[a] + (sd[a] * z if model == "diag" else z)
    inp["mu"] = c + 0.5 * torch.randn(K, D, generator=g)
    return inp


def paired(model, N, K, D, seed, share):
    """Clustered rows, a share of the clusters in close pairs half the components apart
    (so in two blocks): their rows are near both."""
    inp = CLUSTERED[model](N, K, D, seed=seed)
    g = torch.Generator().manual_seed(seed)
    n = int(K // 2 * share)
    inp["mu"][K // 2:K // 2 + n] = inp["mu"][:n] + (0.2 if model == "iso" else 0.1) * torch.randn(n, D, generator=g)
    if model == "diag":
        inp["log_sigma_sq"][K // 2:K // 2 + n] = inp["log_sigma_sq"][:n]
    return inp
