"""Calls that may screen, captured into a HIP graph: the route is the device's choice in every
replay, so the replays follow the data, and each equals the eager call on the same inputs."""

import pytest
import torch

from flash_gmm import _lib, data, diag_estep_into, full_estep_into, iso_estep_into
from routes import SCREEN, call_mode

pytestmark = pytest.mark.gpu
CALLS = {
    "iso": (iso_estep_into, data.iso_clustered, data.reference_smoke, (66_000, 1024, 128), "log_sigma_sq"),
    "diag": (diag_estep_into, data.diag_clustered, data.diag_reference_smoke, (45_003, 1024, 96), "log_sigma_sq"),
    "full": (full_estep_into, data.full_clustered, data.full_reference_smoke, (20_001, 128, 64), "prec_chol"),
}


@pytest.mark.parametrize("model", ["iso", "diag", "full"])
def test_replays_follow_the_data(model, gpu_device):
    fn, clustered, dense, (N, K, D), shape = CALLS[model]
    dev, flags = gpu_device, _lib.FLAG_STORE_LOGJOINT_AUTO
    keys = ("X", "mu", shape, "log_pi")
    sets = [[inp[k].to(dev) for k in keys] for inp in (clustered(N, K, D, seed=1), dense(N, K, D, seed=2),
                                                       clustered(N, K, D, seed=3))]
    nbytes = getattr(_lib.lib(), f"fgmm_{model}_workspace_bytes_ex")(N, K, D, flags)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    args = [t.clone() for t in sets[0]]
    sig = (K,) if model == "iso" else (K, D) if model == "diag" else (K, D, D)

    def outputs():
        return [torch.full(s, float("nan"), device=dev) for s in ((N,), (K,), (K, D), sig)]

    def call(a, o):
        fn(*a, *o, store_log_joint="auto", workspace=ws)

    out = outputs()
    call(args, out)   # warm-up: kernel attributes
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call(args, out)
    torch.cuda.synchronize()
    modes = []
    for rep in (0, 1, 2, 1, 0):
        print(f"capture {model} replay of set {rep}", flush=True)
        for dst, src in zip(args, sets[rep]):
            dst.copy_(src)
        for t in out:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        modes.append(call_mode(model, ws, N, K, D, flags))
        eager = outputs()
        call(sets[rep], eager)
        torch.cuda.synchronize()
        for u, v in zip(out, eager):
            assert torch.equal(u, v), f"{model} set {rep}"
    assert modes[0] == modes[2] == modes[4] == SCREEN and modes[1] == modes[3] != SCREEN
