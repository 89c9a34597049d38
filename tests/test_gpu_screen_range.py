"""The screened pass 1 over the range of its inputs' values: logZ bit for bit the dense run's
(the unscreened exact passes), the sums per component to 1e-5."""

import math

import pytest
import torch

from flash_gmm import data
from parity import assert_dense_agrees
from routes import SCREEN
from screened import call

pytestmark = pytest.mark.gpu
LOG2_E = math.log2(math.e)


def check(model, inp, dev, what):
    print(what, flush=True)
    got, dense = call(model, inp, dev, expect=SCREEN), call(model, inp, dev, dense=True)
    bad = (got[0] != dense[0]).nonzero().flatten()
    assert bad.numel() == 0, f"{what}: logZ of rows {bad[:8].tolist()}: {got[0][bad[:8]]} not {dense[0][bad[:8]]}"
    assert_dense_agrees(got[:2], dense[:2], bitwise=False)
    for u, v in zip(got[2:], dense[2:]):
        u, v = u.double().reshape(u.shape[0], -1), v.double().reshape(v.shape[0], -1)
        top = v.abs().max(dim=1).values
        assert bool(((u - v).abs().max(dim=1).values <= 1e-5 * top).all()), what
    return got


# A last block of 12 and of 8 components (the second with scattered zero weights too), and
# whole blocks of which one has no weight.
@pytest.mark.parametrize("N,K,D", [(400_031, 300, 64), (63_009, 1000, 128), (63_009, 1024, 128)])
def test_iso_rows_below_any_sentinel(N, K, D, gpu_device):
    """Finite rows whose every log-joint is below -1e28, beside components that weigh nothing
    (log_pi = -inf, or the padding of the last block)."""
    inp = data.iso_clustered(N, K, D, seed=K % 11)
    if K == 1024:
        inp["log_pi"][64:96] = -math.inf
    elif K == 1000:
        inp["log_pi"][5::37] = -math.inf
    for i, v in enumerate((1e14, 2e15, -2e15, 1e17, -9.22e18)):
        inp["X"][1000 * i + 17, 3 * i] = v
    check("iso", inp, gpu_device, f"iso range N={N} K={K} D={D}")


@pytest.mark.parametrize("N,K,D", [(42_017, 1000, 96), (42_017, 1024, 96)])
def test_diag_rows_below_any_sentinel(N, K, D, gpu_device):
    """Data in units of 1e-10 with outliers, beside components that weigh nothing."""
    inp = data.diag_clustered(N, K, D, seed=K % 11)
    if K == 1024:
        inp["log_pi"][64:96] = -math.inf
    elif K == 1000:
        inp["log_pi"][5::37] = -math.inf
    unit = 1e-10
    inp["X"] *= unit
    inp["mu"] *= unit
    inp["log_sigma_sq"] += 2.0 * math.log(unit)
    for i, v in enumerate((1e3, 1e5, -1e6, 1e7, -1e8)):
        inp["X"][1000 * i + 17, 3 * i] = v
    check("diag", inp, gpu_device, f"diag range N={N} K={K} D={D}")


@pytest.mark.parametrize("unit", [1e-14, 1e-12, 1.0])
def test_diag_squares_of_squares_that_underflow(unit, gpu_device):
    """Small units: the fourth powers of the rows' elements are 0 in float32.  Half of the
    components have one variance each, whose rounding to bf16 adds up over the dimensions,
    and a tenth of the rows is far out, nearest to those."""
    N, K, D = 42_017, 1024, 96
    inp = data.diag_clustered(N, K // 2, D, seed=3)
    g = torch.Generator().manual_seed(3)
    inp["mu"] = torch.cat([inp["mu"], 6.0 * torch.randn(K // 2, D, generator=g)])
    inp["log_sigma_sq"] = torch.cat([inp["log_sigma_sq"], (0.6 + 0.8 * torch.rand(K // 2, 1, generator=g)).expand(-1, D)])
    inp["log_pi"] = torch.full((K,), -math.log(K))
    inp["X"][::10] *= 50.0
    inp["X"] *= unit
    inp["mu"] *= unit
    inp["log_sigma_sq"] += 2.0 * math.log(unit)
    check("diag", inp, gpu_device, f"diag unit {unit}")


@pytest.mark.parametrize("model,N,D", [("iso", 63_009, 128), ("diag", 42_017, 96)])
def test_roundings_to_bf16_that_add_up(model, N, D, gpu_device):
    """Rows whose products with their component's operands are all rounded down by nearly 2^-7,
    and a second component, 20 (log2) behind, whose operands are 0: the first one's block must
    stay.  The other components are tight, so far behind."""
    K, e = 1024, 2.0 ** -8
    inp = (data.iso_clustered if model == "iso" else data.diag_clustered)(N, K, D, seed=8)
    inp["X"] *= 0.25
    inp["mu"] *= 0.25
    inp["log_sigma_sq"] -= 2.0 * math.log(4.0)
    for k, m in ((100, 64.0 * (1.0 + 0.97 * e)), (900, 0.0)):
        block = slice(k // 32 * 32, k // 32 * 32 + 32)
        inp["log_pi"][block] = -math.inf   # the block's bound is the component's
        inp["log_pi"][k] = -7.0
        inp["mu"][k] = m
        inp["log_sigma_sq"][k] = math.log(LOG2_E)   # exp(-lss) log2 e = 1: the operands are the mean's elements
    inp["X"][[33, 5000, N - 1]] = 32.0 * (1.0 + 0.99 * e)
    out = check(model, inp, gpu_device, f"{model} rounded down")
    assert abs(float(out[1][100]) - 3.0) < 1e-4
