"""The isotropic default plan's screened pass 1 (large calls where most rows are near one
component block): results against the dense run (the unscreened exact passes) and the
float64 oracle, at the smallest sizes that take it."""

import math

import pytest
import torch

from flash_gmm import _lib, data, flash_gmm_estep, iso_estep_into
from oracle import gmm_oracle as O
from parity import assert_dense_agrees
from routes import SCREEN
from screened import KEYS, call, check, listed, paired, separated

pytestmark = pytest.mark.gpu


# Chunk counts 2 .. 8, a last block of 1 and of 32 components, a last tile of 1 row, D that is
# no multiple of 4, an odd number of blocks, and more blocks than one 32-word group.
@pytest.mark.parametrize("N,K,D", [(63_009, 1024, 128), (70_001, 993, 125), (90_017, 1025, 96), (236_001, 520, 64),
                                   (130_001, 2048, 31)])
def test_screened_sizes(N, K, D, gpu_device):
    inp = separated("iso", N, K, D, K % 13) if D < 40 else data.iso_clustered(N, K, D, seed=K % 13)
    check("iso", inp, gpu_device, f"screen N={N} K={K} D={D}", O.estep_iso)


@pytest.mark.parametrize("share,many", [(0.02, False), (0.4, True)])
def test_rows_near_two_blocks(share, many, gpu_device):
    """The listed rows: few (one tile per workgroup) and many (256 rows per workgroup)."""
    inp = paired("iso", 63_009, 1024, 128, 3, share)
    n, few = listed("iso", inp, gpu_device)
    assert n > 0 and (n > few) == many, f"{n} rows listed, a short list holds {few}"
    check("iso", inp, gpu_device, f"screen paired {share}", O.estep_iso)


def test_faint_components_keep_their_sums(gpu_device):
    """Components far from every row: responsibilities between 2^-160 and 2^-72 only, which
    their sums must still hold: the dense run adds the same responsibilities in another
    grouping (float32 sums of fewer than 2^8 terms a lane: 2^-16); and zero-weight
    components."""
    dev = gpu_device
    N, K, D = 70_000, 1024, 128
    inp = data.iso_clustered(N, K, D, seed=5)
    a = inp["mu"][:40].clone()
    inp["mu"][700:740] = a + 2.4 / math.sqrt(D) * torch.sign(a) * 5.0   # ||shift|| = 12
    inp["log_sigma_sq"][700:740] = inp["log_sigma_sq"][:40]
    inp["log_pi"][300:310] = -math.inf
    print("screen faint", flush=True)
    got = call("iso", inp, dev, expect=SCREEN)
    dense = call("iso", inp, dev, dense=True)
    assert_dense_agrees(got, dense, bitwise=False)
    assert (got[1][300:310] == 0).all()
    small = (dense[1] > 1e-30) & (dense[1] < 1e-4)
    assert int(small.sum()) >= 10
    for u, v in zip(got[1:], dense[1:]):
        u, v = u[small].double().reshape(int(small.sum()), -1), v[small].double().reshape(int(small.sum()), -1)
        assert float(((u - v).norm(dim=1) / v.norm(dim=1)).max()) <= 2.0 ** -16


def test_tight_components_beside_faint_rows(gpu_device):
    """Tight components of three rows each, with a row of another component at a distance at
    which its responsibility is about 2^-100: left out, since Nk is above 2^-10.  Their sums are
    the dense run's to float32 rounding and N 2^-72, also the one of a coordinate that is 0 in
    their own rows."""
    dev = gpu_device
    N, K, D = 63_009, 1024, 128
    inp = data.iso_clustered(N, K, D, seed=9)
    g = torch.Generator().manual_seed(9)
    sigma = 0.4
    inp["X"][0:20_000:1000, 0] = 1.0
    logZ2 = O.estep_iso(inp["X"][0:20_000:1000], *[inp[k] for k in KEYS[1:]])[0] * math.log2(math.e)
    half = 0.5 / sigma ** 2 * math.log2(math.e)
    tight = list(range(512, 532))
    for j, k in enumerate(tight):
        top = (float(inp["log_pi"][k]) - 0.5 * D * (math.log(2.0 * math.pi) + 2.0 * math.log(sigma))) * math.log2(math.e)
        d2 = (top - float(logZ2[j]) + 100.0) / half
        step = torch.randn(D, generator=g)
        step[0] = 0.0
        mu = inp["X"][1000 * j] + step / step.norm() * math.sqrt(d2 - 1.0)
        mu[0] = 0.0
        inp["mu"][k], inp["log_sigma_sq"][k] = mu, 2.0 * math.log(sigma)
        own = mu + sigma * torch.randn(3, D, generator=g)
        own[:, 0] = 0.0
        inp["X"][1000 * j + 1:1000 * j + 4] = own
    print("screen tight", flush=True)
    got, dense = call("iso", inp, dev, expect=SCREEN), call("iso", inp, dev, dense=True)
    assert_dense_agrees(got, dense, bitwise=False)
    assert bool(((got[1][tight] - 3.0).abs() < 1e-3).all())
    left_out = dense[2][tight, 0]
    assert int(((left_out > 0) & (left_out < N * 2.0 ** -72)).sum()) >= 10, left_out   # what the dense run adds
    for u, v in zip(got[1:], dense[1:]):
        u, v = u[tight].double().reshape(len(tight), -1), v[tight].double().reshape(len(tight), -1)
        assert bool(((u - v).abs() <= 2.0 ** -16 * v.abs().max(dim=1, keepdim=True).values).all())
    assert bool(((got[2] - dense[2])[tight, 0].abs() <= N * 2.0 ** -72).all())


def test_special_rows_and_components(gpu_device):
    """NaN and infinite rows, and a component whose constants overflow: as the dense run."""
    dev = gpu_device
    inp = data.iso_clustered(66_000, 1024, 128, seed=6)
    inp["X"][7, 3] = math.nan
    inp["X"][40_000, 127] = math.inf
    inp["X"][65_999] = 1e25
    print("screen special rows", flush=True)
    got, dense = call("iso", inp, dev, expect=SCREEN), call("iso", inp, dev, dense=True)
    assert torch.equal(got[0].isnan(), dense[0].isnan())
    fin = ~dense[0].isnan()
    assert torch.equal(got[0][fin], dense[0][fin])
    assert torch.equal(got[1].isnan(), dense[1].isnan())
    inp = data.iso_clustered(66_000, 1024, 128, seed=6)
    inp["log_sigma_sq"][5] = -90.0   # b ||x||^2 beyond float32
    print("screen special component", flush=True)   # (the probe finds every row near its block too)
    got, dense = call("iso", inp, dev), call("iso", inp, dev, dense=True)
    assert_dense_agrees(got, dense, bitwise=False)


def test_phase_split_strided_rows_and_lean_workspace(gpu_device):
    """PHASE1 then PHASE2, and rows with a stride: bitwise one call's results.  A workspace
    of the size that holds no screening: the exact pass 1, the same logZ bits."""
    dev = gpu_device
    N, K, D = 63_009, 1024, 100
    inp = paired("iso", N, K, D, 4, 0.1)
    one = call("iso", inp, dev, expect=SCREEN)
    L = _lib.lib()
    ws = torch.empty(L.fgmm_iso_workspace_bytes(N, K, D), dtype=torch.uint8, device=dev)
    args = [inp[k].to(dev) for k in KEYS]
    out = [torch.empty_like(t) for t in one]
    print("screen phases", flush=True)
    iso_estep_into(*args, *out, workspace=ws, phase=1)
    iso_estep_into(*args, None, *out[1:], workspace=ws, phase=2)
    assert all(torch.equal(u, v) for u, v in zip(out, one))
    wide = torch.zeros(N, 132, device=dev)
    wide[:, 8:108] = args[0]
    out = [torch.empty_like(t) for t in one]
    iso_estep_into(wide[:, 8:108], *args[1:], *out)
    assert all(torch.equal(u, v) for u, v in zip(out, one))
    auto = flash_gmm_estep(*args)
    assert all(torch.equal(u, v) for u, v in zip(auto, one))
    # One word per (tile, block) and one bit per row less than the query asks for.
    lean = ws.numel() - (N // 32 + 8) * (-(-K // 32)) * 4
    out = [torch.empty_like(t) for t in one]
    print("screen lean workspace", flush=True)
    st = L.fgmm_iso_estep_f32(args[0].data_ptr(), D, N, D, args[1].data_ptr(), D, K, args[2].data_ptr(),
                              args[3].data_ptr(), *[t.data_ptr() for t in out], ws.data_ptr(), lean, 0,
                              _lib.stream_handle(torch.device(dev)))
    torch.cuda.synchronize()
    assert st == 0
    assert_dense_agrees(out, one, bitwise=False)
