"""The gathering pass 2 above D = 64: each slab's float32 sums go out in two partials, one per
half of its rows, so that no sum runs over more rows than half a slab."""

import math

import pytest
import torch

from flash_gmm import diag_estep_into, iso_estep_into

pytestmark = pytest.mark.gpu


# 32 slabs of 42 and of 62 tiles (1024 components, 256 compute units).
@pytest.mark.parametrize("N,D,tiles", [(42_016, 96, 42), (63_009, 128, 62)])
# (An isotropic dense run's sums are the tile pass's.)
@pytest.mark.parametrize("model,dense", [("iso", False), ("diag", False), ("diag", True)])
def test_a_sum_ends_with_half_a_slab(model, N, D, tiles, dense, gpu_device):
    """Every row belongs to component 0.  Dimension 0 of the first row is 2^13, beside which
    the other rows' 2^-16 are lost, 32 rows at once too: as many as share its sum."""
    if torch.cuda.get_device_properties(gpu_device).multi_processor_count != 256:
        pytest.skip("slabs counted for 256 compute units")
    print(f"partials {model} N={N} D={D} dense={dense}", flush=True)
    dev, K = gpu_device, 1024
    g = torch.Generator(device=dev).manual_seed(D)
    X = 0.5 * torch.randn(N, D, generator=g, device=dev)
    mu = 50.0 * torch.randn(K, D, generator=g, device=dev)
    mu[0] = 0.0
    mu[:, 0] = 0.0
    X[:, 0] = 2.0 ** -16
    X[0, 0] = 2.0 ** 13
    shape = torch.zeros(K, device=dev) if model == "iso" else torch.zeros(K, D, device=dev)
    lpi = torch.full((K,), -math.log(K), device=dev)
    out = [torch.empty(N, device=dev), torch.empty(K, device=dev), torch.empty(K, D, device=dev),
           torch.empty_like(shape)]
    (iso_estep_into if model == "iso" else diag_estep_into)(X, mu, shape, lpi, *out, dense=dense)
    torch.cuda.synchronize()
    assert abs(float(out[1][0]) - N) <= 1e-5 * N
    lost = (N - 1) - (float(out[2][0, 0]) - 2.0 ** 13) * 2.0 ** 16
    # Half the tiles, and one more where they are computed in pairs; the sum of the partials
    # is rounded to a multiple of 2^-10.
    assert lost <= (tiles // 2 + 1) * 32 + 32, f"{lost} rows in the first row's sum"
    assert lost >= (tiles // 2 - 1) * 32 - 32   # (the other rows of its tile may not be)
