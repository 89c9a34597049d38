"""The full model's screened pass 1 (the drop-in call on clustered rows): against the
default plan, whose exact pass 1 sees every pair, and against the float64 oracle."""

import math

import pytest
import torch

from flash_gmm import _lib, data, full_estep_into
from oracle import gmm_oracle as O
from parity import assert_close_stats, assert_dense_agrees
from routes import SCREEN, call_mode, overflowed_tiles

pytestmark = pytest.mark.gpu
KEYS = ("X", "mu", "prec_chol", "log_pi")


def call(inp, dev, store, expect=None):
    """full_estep_into's outputs; expect: the route the probe must have chosen."""
    args = [inp[k].to(dev) for k in KEYS]
    N, D = args[0].shape
    K = args[1].shape[0]
    out = [torch.full((N,), math.nan, device=dev), torch.empty(K, device=dev), torch.empty(K, D, device=dev),
           torch.empty(K, D, D, device=dev)]
    flags = _lib.FLAG_STORE_LOGJOINT_AUTO if store == "auto" else 0
    ws = torch.empty(_lib.lib().fgmm_full_workspace_bytes_ex(N, K, D, flags), dtype=torch.uint8, device=dev)
    full_estep_into(*args, *out, store_log_joint=store, workspace=ws)
    torch.cuda.synchronize()
    if expect is not None:
        mode = call_mode("full", ws, N, K, D, flags)
        assert mode == expect, f"N={N} K={K} D={D}: route {mode}, not {expect}"
    return out


def same(got, want, what):
    """logZ bit for bit; the sums, whose terms the default plan's wider masks may group
    otherwise, as assert_dense_agrees takes two groupings; NaN where it is NaN."""
    for name, u, v in zip(("logZ", "Nk", "mu_acc", "sig_outer"), got, want):
        assert torch.equal(u.isnan(), v.isnan()), f"{what} {name}: NaN"
    assert_dense_agrees([u.nan_to_num(0.0) for u in got], [v.nan_to_num(0.0) for v in want], bitwise=False)


def separated(N, K, D, seed):
    """full_clustered's covariances around centres twice as far apart."""
    inp = data.full_clustered(8, K, D, seed=seed)
    g = torch.Generator().manual_seed(seed)
    inp["mu"] = 4.0 * torch.randn(K, D, generator=g)
    a, z = torch.randint(0, K, (N,), generator=g), torch.randn(N, D, generator=g)
    inp["X"] = torch.empty(N, D)
    for k in range(K):   # cov = (L L^T)^-1: x = mu + L^-T z
        r = (a == k).nonzero().flatten()
        inp["X"][r] = inp["mu"][k] + torch.linalg.solve_triangular(inp["prec_chol"][k].t(), z[r].t(), upper=True).t()
    return inp


# Widths 32 and 64, a last stage of 1, 4 and all of its components, a last tile of 1 row, a
# last workgroup of one tile, D that is no multiple of 4.
@pytest.mark.parametrize("N,K,D", [(5_153, 256, 32), (9_217, 301, 64), (40_033, 100, 39), (90_001, 17, 50),
                                   (30_001, 77, 17)])
def test_screened_sizes(N, K, D, gpu_device):
    print(f"full screen N={N} K={K} D={D}", flush=True)
    inp = (separated if D < 20 else data.full_clustered)(N, K, D, seed=K % 13)
    got = call(inp, gpu_device, "auto", SCREEN)
    same(got, call(inp, gpu_device, False), f"N={N} K={K} D={D}")
    assert_close_stats(got, O.estep_full(*[inp[k] for k in KEYS]), f"full screen N={N} K={K} D={D}")


def test_rows_of_several_and_special_components(gpu_device):
    """Components in close pairs and far away, zero weights, then NaN, infinite and huge rows."""
    inp = data.full_clustered(20_000, 128, 40, seed=5)
    g = torch.Generator().manual_seed(1)
    inp["mu"][64:100] = inp["mu"][:36] + 0.05 * torch.randn(36, 40, generator=g)
    inp["prec_chol"][64:100] = inp["prec_chol"][:36]
    inp["mu"][100:110] *= 50.0
    inp["log_pi"][110:120] = -math.inf
    inp["prec_chol"][120:124, 3, 37] = 5.0   # above the diagonal: taken as it is
    print("full screen paired", flush=True)
    got = call(inp, gpu_device, "auto", SCREEN)
    same(got, call(inp, gpu_device, False), "paired")
    assert (got[1][110:120] == 0).all()
    inp["X"][7, 3] = math.nan
    inp["X"][10_000, 39] = math.inf
    inp["X"][19_999] = 1e-25
    print("full screen special rows", flush=True)
    same(call(inp, gpu_device, "auto", SCREEN), call(inp, gpu_device, False), "special rows")
    inp["X"][7] = inp["X"][10_000] = 1e18   # finite; the screening's squares are not all
    print("full screen huge rows", flush=True)
    same(call(inp, gpu_device, "auto", SCREEN), call(inp, gpu_device, False), "huge rows")
    inp["X"][64:96] = math.nan   # a tile of which every pair is needed: the exact pass 1
    print("full screen full tile", flush=True)
    same(call(inp, gpu_device, "auto", SCREEN), call(inp, gpu_device, False), "full tile")


def test_a_tile_past_its_pool_costs_only_its_group(gpu_device):
    """Tiles whose needed pairs exceed their pool (every pair of NaN rows is needed): the call
    stays screened, and those tiles get the exact pass 1's results."""
    dev, N, K, D = gpu_device, 40_033, 100, 39
    inp = data.full_clustered(N, K, D, seed=2)
    inp["X"][64:80] = math.nan
    inp["X"][20_000] = math.nan   # alone in its tile: within the pool
    inp["X"][40_010:] = math.nan   # 22 rows of the last tile but one, and the last one's only row
    args = [inp[k].to(dev) for k in KEYS]
    out = [torch.empty(N, device=dev), torch.empty(K, device=dev), torch.empty(K, D, device=dev),
           torch.empty(K, D, D, device=dev)]
    nbytes = _lib.lib().fgmm_full_workspace_bytes_ex(N, K, D, _lib.FLAG_STORE_LOGJOINT_AUTO)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    print("full screen pools", flush=True)
    full_estep_into(*args, *out, store_log_joint="auto", workspace=ws, phase=1)
    assert call_mode("full", ws, N, K, D, _lib.FLAG_STORE_LOGJOINT_AUTO) == SCREEN
    assert overflowed_tiles(ws, N, K, D) == [2, 1250]
    full_estep_into(*args, None, *out[1:], store_log_joint="auto", workspace=ws, phase=2)
    same(out, call(inp, dev, False), "pools")
