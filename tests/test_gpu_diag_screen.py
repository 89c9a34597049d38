"""The diagonal default plan's screened pass 1 (large calls where most rows are near one
component block): results against the dense run (the unscreened exact passes) and the
float64 oracle, at the smallest sizes that take it."""

import math

import pytest
import torch

from flash_gmm import _lib, data, diag_estep_into, flash_gmm_estep_diag
from oracle import gmm_oracle as O
from parity import assert_dense_agrees
from routes import SCREEN
from screened import KEYS, call, check, listed, paired, separated

pytestmark = pytest.mark.gpu


# Widths 32 .. 128 (one and two blocks per stage), a last block of 1 and of 32 components, a
# last tile of 1 row, D that is no multiple of 4, an odd number of blocks.
@pytest.mark.parametrize("N,K,D", [(42_017, 1024, 96), (40_513, 1025, 90), (33_001, 993, 125), (111_201, 545, 61),
                                   (66_001, 2048, 31)])
def test_screened_sizes(N, K, D, gpu_device):
    inp = separated("diag", N, K, D, K % 13) if D < 40 else data.diag_clustered(N, K, D, seed=K % 13)
    check("diag", inp, gpu_device, f"diag screen N={N} K={K} D={D}", O.estep_diag)


@pytest.mark.parametrize("share,many", [(0.02, False), (0.4, True)])
def test_rows_near_two_blocks(share, many, gpu_device):
    """The listed rows: few (one tile per workgroup) and many (128 rows per workgroup)."""
    inp = paired("diag", 45_009, 1024, 96, 3, share)
    n, few = listed("diag", inp, gpu_device)
    assert n > 0 and (n > few) == many, f"{n} rows listed, a short list holds {few}"
    check("diag", inp, gpu_device, f"diag screen paired {share}", O.estep_diag)


def test_faint_and_special_components(gpu_device):
    """Components far from every row (responsibilities between 2^-160 and 2^-72 only) keep
    their sums as in the dense run (float32 sums of fewer than 2^8 terms a lane in another
    grouping: 2^-16); zero-weight components; NaN and infinite rows as in the dense run."""
    dev = gpu_device
    inp = data.diag_clustered(45_000, 1024, 96, seed=5)
    a, ls = inp["mu"][:40], inp["log_sigma_sq"][:40]
    inp["mu"][700:740] = a + 12.0 / math.sqrt(96.0) * torch.sign(a) * torch.exp(0.5 * ls)
    inp["log_sigma_sq"][700:740] = ls
    inp["log_pi"][300:310] = -math.inf
    print("diag screen faint", flush=True)
    got, dense = call("diag", inp, dev, expect=SCREEN), call("diag", inp, dev, dense=True)
    assert_dense_agrees(got, dense, bitwise=False)
    assert (got[1][300:310] == 0).all()
    small = (dense[1] > 1e-30) & (dense[1] < 1e-4)
    assert int(small.sum()) >= 10
    n = int(small.sum())
    for u, v in zip(got[1:3], dense[1:3]):
        u, v = u[small].double().reshape(n, -1), v[small].double().reshape(n, -1)
        assert float(((u - v).norm(dim=1) / v.norm(dim=1)).max()) <= 2.0 ** -16
    inp["X"][7, 3] = math.nan
    inp["X"][30_000, 95] = math.inf
    inp["X"][44_999] = 1e18
    print("diag screen special rows", flush=True)
    got, dense = call("diag", inp, dev, expect=SCREEN), call("diag", inp, dev, dense=True)
    assert torch.equal(got[0].isnan(), dense[0].isnan())
    fin = ~dense[0].isnan()
    assert torch.equal(got[0][fin], dense[0][fin])
    assert torch.equal(got[1].isnan(), dense[1].isnan())


def test_phase_split_strided_rows_and_lean_workspace(gpu_device):
    """PHASE1 then PHASE2, rows with a stride, and the drop-in call: bitwise one call's
    results.  A workspace too small for the screening: the exact pass 1, the same logZ."""
    dev = gpu_device
    N, K, D = 70_009, 1024, 60
    inp = paired("diag", N, K, D, 4, 0.1)
    one = call("diag", inp, dev, expect=SCREEN)
    L = _lib.lib()
    ws = torch.empty(L.fgmm_diag_workspace_bytes(N, K, D), dtype=torch.uint8, device=dev)
    args = [inp[k].to(dev) for k in KEYS]
    out = [torch.empty_like(t) for t in one]
    print("diag screen phases", flush=True)
    diag_estep_into(*args, *out, workspace=ws, phase=1)
    diag_estep_into(*args, None, *out[1:], workspace=ws, phase=2)
    assert all(torch.equal(u, v) for u, v in zip(out, one))
    wide = torch.zeros(N, 72, device=dev)
    wide[:, 8:68] = args[0]
    out = [torch.empty_like(t) for t in one]
    diag_estep_into(wide[:, 8:68], *args[1:], *out)
    assert all(torch.equal(u, v) for u, v in zip(out, one))
    assert all(torch.equal(u, v) for u, v in zip(flash_gmm_estep_diag(*args), one))
    out = [torch.empty_like(t) for t in one]
    print("diag screen lean workspace", flush=True)
    st = L.fgmm_diag_estep_f32(args[0].data_ptr(), D, N, D, args[1].data_ptr(), D, K, args[2].data_ptr(), D,
                               args[3].data_ptr(), *[t.data_ptr() for t in out], ws.data_ptr(), ws.numel() - 256, 0,
                               _lib.stream_handle(torch.device(dev)))
    torch.cuda.synchronize()
    assert st == 0
    assert_dense_agrees(out, one, bitwise=False)
