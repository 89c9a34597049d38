"""Performance cases: calls that programs make through the package's public entry points.

A case is a dict of plain values:

  call       "estep" (one drop-in E-step), "em" (in-memory EM, `iters` iterations of E-step and
             M-step) or "stream" (EM over rows in host memory, in chunks of `chunk` rows)
  model      "iso", "diag" or "full" covariance
  data       "clustered" (rows drawn around K separated centres: a row has a few responsible
             components), "plain" (X ~ N(0, I), mu ~ N(0, 4I)) or "dense" (X, mu ~ N(0, I),
             unit-scale variances: every component is responsible for a part of every row)
  precision  "fp32", or "bf16" (the opt-in bf16 operand contract)
  N, K, D    rows, components, dimensions

prepare() makes the inputs on the GPU from the seed (the rows of "stream" in host memory),
run() is one pass, exact() the same outputs in float64 from plain torch.
"""

import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

# The package lives in flash-gmm_amd/ under the repository's root, the working folder.
_PKG = os.path.join(os.getcwd(), "flash-gmm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import flash_gmm  # noqa: E402

LOG2_E = math.log2(math.e)
LOG_2PI = math.log(2.0 * math.pi)


def _case(name, call, model, data, precision, N, K, D, iters=1, chunk=0):
    return dict(name=name, call=call, model=model, data=data, precision=precision, N=N, K=K, D=D,
                iters=iters, chunk=chunk)


def listed():
    return [
        # A toy mixture: a thousand 3-d points, five blobs.  Launches and host work are all of it.
        _case("iso_n1000_k5_d3", "estep", "iso", "clustered", "fp32", 1000, 5, 3),
        # The small golden workload of the tests: a quick experiment, or a codebook on a sample.
        _case("iso_n10k_k64_d32", "estep", "iso", "plain", "fp32", 10_000, 64, 32),
        # The GloVe-50 vocabulary (400,001 vectors) against a few hundred clusters: D is no
        # multiple of four, so the rows are not readable in place.
        _case("iso_n400k_k300_d50", "estep", "iso", "clustered", "fp32", 400_001, 300, 50),
        # The headline shape: SIFT-like vectors, 1024 clusters.
        _case("iso_n1m_k1024_d128", "estep", "iso", "clustered", "fp32", 1_000_000, 1024, 128),
        # The same shape on overlapping components (the first iterations of a fit).
        _case("iso_dense_n1m_k1024_d128", "estep", "iso", "dense", "fp32", 1_000_000, 1024, 128),
        # GIST-960 descriptors: the wide path.
        _case("iso_n100k_k256_d960", "estep", "iso", "clustered", "fp32", 100_000, 256, 960),
        # The headline shape under the bf16 operand contract.
        _case("iso_bf16_n1m_k1024_d128", "estep", "iso", "clustered", "bf16", 1_000_000, 1024, 128),
        # Deep-96 vectors, per-dimension variances.
        _case("diag_n1m_k1024_d96", "estep", "diag", "clustered", "fp32", 1_000_000, 1024, 96),
        # A diagonal mixture on a GloVe-25 sample with overlapping components, sizes all ragged.
        _case("diag_dense_n30k_k77_d25", "estep", "diag", "dense", "fp32", 30_011, 77, 25),
        # Full covariances at the benchmark shape.
        _case("full_n250k_k256_d64", "estep", "full", "clustered", "fp32", 250_000, 256, 64),
        # Fitting a full-covariance mixture on 39-d speech-like features: three EM iterations.
        _case("em_full_n100k_k32_d39", "em", "full", "clustered", "fp32", 100_003, 32, 39, iters=3),
        # Two EM iterations over rows that stay in host memory, fed from an array in chunks.
        _case("stream_iso_n1m_k256_d64", "stream", "iso", "clustered", "fp32", 1_000_000, 256, 64,
              iters=2, chunk=262_144),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the ranges above: N 500 .. 1M, K 2 .. 1024 (full 2 .. 256), D 2 .. 960 (bf16 and
    diagonal dense data to 128, full to 128), no more work than the largest listed E-step."""
    kind = rng.choice(["iso", "iso", "iso", "diag", "diag", "full", "full", "em", "stream"])
    data = rng.choice(["clustered", "clustered", "plain", "dense"])
    precision = "bf16" if kind in ("iso", "diag", "full") and rng.random() < 0.2 else "fp32"
    model = kind if kind in ("iso", "diag", "full") else rng.choice(["iso", "diag", "full"]) if kind == "em" else "iso"
    call = kind if kind in ("em", "stream") else "estep"
    if model == "full":
        D, K, data = _logint(rng, 2, 128), _logint(rng, 2, 256), "clustered" if data == "plain" else data
        per_row, most = K * D * D, 2.6e11 if data == "clustered" else 1.2e11
    else:
        wide = precision == "fp32" and call == "estep" and data == "clustered"
        D, K = _logint(rng, 2, 960 if wide else 128), _logint(rng, 2, 1024)
        per_row, most = K * D * (2 if model == "diag" else 1), 1.3e11 if D <= 128 else 5e10
    N = _logint(rng, 500, 1_000_000)
    iters, chunk = 1, 0
    if call != "estep":
        iters, most, N = rng.choice([2, 3]), most / 4, min(N, 500_000)
        data = "clustered"  # the rows a fit is run on
        if model == "full":
            D, K = min(D, 64), min(K, 64)
            per_row = K * D * D
        N = max(N, 50 * K, 20 * D * K if model == "full" else 0)  # enough rows for every component
    N = max(500, min(N, int(most / per_row)))
    if call == "stream":
        chunk = max(64, N // rng.choice([1, 3, 5]) + rng.choice([0, 1]))
    c = _case("", call, model, data, precision, N, K, D, iters, chunk)
    del c["name"]
    return c


# --------------------------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------------------------

def _inputs(case, seed):
    """(X, mu, shape, log_pi): shape is log_sigma_sq (iso K, diag K x D) or prec_chol (full)."""
    N, K, D, model, data = case["N"], case["K"], case["D"], case["model"], case["data"]
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    dense = data == "dense"
    c = randn(K, D) if dense else 2.0 * randn(K, D)
    lpi = torch.full((K,), -math.log(K), device=dev) if dense else torch.log_softmax(0.7 * randn(K).double(), 0).float()
    if model == "iso":
        shape = torch.zeros(K, device=dev) if data != "clustered" else torch.rand(K, generator=g, device=dev) - 0.5
    elif model == "diag":
        shape = 0.2 * randn(K, D) if data != "clustered" else 2.0 * torch.rand(K, D, generator=g, device=dev) - 1.0
    else:
        A = randn(K, D, D).double().cpu().numpy()
        AAt = np.matmul(A, np.ascontiguousarray(A.transpose(0, 2, 1))) / D
        cov = np.eye(D) + 0.2 * AAt if dense else AAt + 0.1 * np.eye(D)
        shape = torch.from_numpy(np.linalg.cholesky(np.linalg.inv(cov))).float().contiguous().to(dev)
        root = torch.from_numpy(np.linalg.cholesky(cov)).float().to(dev)
    if data != "clustered":
        return randn(N, D), c, shape, lpi
    X = torch.empty(N, D, device=dev)
    step = max(1, (1 << 27) // (D * (D if model == "full" else 1)))
    for n0 in range(0, N, step):
        n1 = min(N, n0 + step)
        a = torch.randint(0, K, (n1 - n0,), generator=g, device=dev)
        z = randn(n1 - n0, D)
        if model == "diag":
            z = z * torch.exp(0.5 * shape)[a]
        elif model == "full":
            z = (root[a] * z[:, None, :]).sum(dim=2)
        X[n0:n1] = c[a] + z
    # Parameters near the truth, as in the middle of a fit (full: the covariances are narrow
    # in some directions, so the means are closer).
    mu = c + (0.1 if model == "full" else 0.5) * randn(K, D)
    return X, mu, shape, lpi


def prepare(case, seed):
    X, mu, shape, lpi = _inputs(case, seed)
    s = SimpleNamespace(case=case, X=X, mu=mu, shape=shape, lpi=lpi)
    if case["call"] == "stream":
        s.rows = X.cpu().numpy()
        s.X = None
    return s


_ESTEP = {"iso": flash_gmm.flash_gmm_estep, "diag": flash_gmm.flash_gmm_estep_diag,
          "full": flash_gmm.flash_gmm_estep_full}
_EM = {"iso": flash_gmm.em_iso, "diag": flash_gmm.em_diag, "full": flash_gmm.em_full}


def run(state):
    case = state.case
    if case["call"] == "estep":
        return _ESTEP[case["model"]](state.X, state.mu, state.shape, state.lpi, precision=case["precision"])
    # EM updates its parameters in place: each pass is a fit from the same starting point.
    mu, shape, lpi = state.mu.clone(), state.shape.clone(), state.lpi.clone()
    if case["call"] == "em":
        loglik = _EM[case["model"]](state.X, mu, shape, lpi, case["iters"])
    else:
        rows = state.rows
        loglik = flash_gmm.stream_em_iso(lambda row0, nrows: rows[row0:row0 + nrows], case["N"], mu, shape, lpi,
                                         iterations=case["iters"], chunk_rows=case["chunk"])["loglik"]
    return mu, shape, lpi, loglik


# --------------------------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------------------------

def work(case):
    """Bytes: rows, parameters and outputs once per pass over the rows.  Flops: the log-joint of
    every (row, component) pair (2 D a pair for iso, 4 D for diag with its two features, D (D + 1)
    for the triangular whitening), and the statistics: of every pair on dense data, of one pair a
    row where responsibilities are concentrated."""
    N, K, D, model = case["N"], case["K"], case["D"], case["model"]
    shape = {"iso": K, "diag": K * D, "full": K * D * D}[model]
    joint = {"iso": 2 * D, "diag": 4 * D, "full": D * (D + 1)}[model]
    stats = {"iso": 2 * D, "diag": 4 * D, "full": D * (D + 1) + 2 * D}[model]
    pairs = K if case["data"] == "dense" else 1
    once = {"bytes": 4 * (N * D + N + 2 * (K * D + shape + K)), "flops": N * (K * joint + pairs * stats)}
    return {k: case["iters"] * v for k, v in once.items()}


def tolerance(case):
    """About four times the largest distance from exact() over the listed cases and 50 drawn ones."""
    if case["call"] != "estep":
        # log sigma^2 of an isotropic fit is near 0 (7.7e-5 of it is 1e-6 of sigma^2).
        return {"rel": 3e-4, "max": 8e-4} if case["model"] == "iso" else {"rel": 3e-5, "max": 2e-4}
    if case["precision"] == "bf16":
        # Responsibilities are rounded to bf16: the last bits of one decide its rounding (5.6e-6, 3.5e-5).
        return {"rel": 3e-5, "max": 2e-4}
    return {"rel": 1.4e-5, "max": 1e-4}  # 3.4e-6, 2.1e-5: dense data, responsibilities of every pair


# --------------------------------------------------------------------------------------------
# The outputs in float64
# --------------------------------------------------------------------------------------------

def _bf16(t):
    return t.float().bfloat16().double()


def _estep64(X, mu, shape, lpi, model, precision):
    """One E-step in float64 (X, mu, shape, lpi: float64 tensors holding the float32 inputs).  With
    "bf16" the operands that the contract rounds are rounded (rows, means or weights, the
    responsibilities of the weighted sums) and everything else is float64."""
    N, D = X.shape
    K = mu.shape[0]
    dev = X.device
    b16 = precision == "bf16"
    ln2 = math.log(2.0)
    logZ = torch.empty(N, dtype=torch.float64, device=dev)
    Nk = torch.zeros(K, dtype=torch.float64, device=dev)
    mu_acc = torch.zeros(K, D, dtype=torch.float64, device=dev)
    sig = torch.zeros((K,) if model == "iso" else (K, D) if model == "diag" else (K, D, D), dtype=torch.float64, device=dev)
    step = max(1, (1 << 28) // max(K, D))
    for n0 in range(0, N, step):
        x = X[n0:n0 + step]
        xb = _bf16(x) if b16 else x
        if model == "iso":
            half = 0.5 * torch.exp(-shape)
            mub = _bf16(mu) if b16 else mu
            dot = xb @ mub.t()
            sq = (xb * xb).sum(1)[:, None] - 2.0 * dot + (mu * mu).sum(1)[None, :]
            ll = (lpi - 0.5 * D * (LOG_2PI + shape))[None, :] - half[None, :] * sq
        elif model == "diag":
            w = 0.5 * torch.exp(-shape) * LOG2_E
            w1, w2 = (_bf16(w), _bf16(mu.float() * w.float())) if b16 else (w, mu * w)
            x2 = _bf16(x * x) if b16 else x * x
            const = (lpi - 0.5 * (D * LOG_2PI + shape.sum(1))) * LOG2_E - (mu * mu * w).sum(1)
            ll = (const[None, :] - x2 @ w1.t() + 2.0 * (xb @ w2.t())) * ln2
        else:
            L = _bf16(shape) if b16 else shape
            ll = torch.empty(x.shape[0], K, dtype=torch.float64, device=dev)
            logdet = torch.log(torch.diagonal(shape, dim1=1, dim2=2).abs() + 1e-30).sum(1)
            for k in range(K):
                y = xb @ L[k] - (mu[k] @ shape[k])[None, :]
                ll[:, k] = lpi[k] + logdet[k] - 0.5 * D * LOG_2PI - 0.5 * (y * y).sum(1)
        lz = torch.logsumexp(ll, dim=1)
        logZ[n0:n0 + step] = lz
        r = torch.exp(ll - lz[:, None])
        Nk += r.sum(0)
        rb = _bf16(r) if b16 else r
        if model == "iso":
            mu_acc += rb.t() @ xb
            sig += (r * sq).sum(0)
        elif model == "diag":
            first, second = rb.t() @ xb, rb.t() @ x2
            mu_acc += first
            sig += second - 2.0 * mu * first + mu * mu * r.sum(0)[:, None]
        else:
            mu_acc += rb.t() @ xb
            for k in range(K):
                rx = x * r[:, k:k + 1]
                sig[k] += (_bf16(rx) if b16 else rx).t() @ xb
    return logZ, Nk, mu_acc, sig


def exact(case, seed):
    N, K, D, model = case["N"], case["K"], case["D"], case["model"]
    X, mu, shape, lpi = (t.double() for t in _inputs(case, seed))
    if case["call"] == "estep":
        return _estep64(X, mu, shape, lpi, model, case["precision"])
    loglik = []
    for _ in range(case["iters"]):
        logZ, Nk, mu_acc, sig = _estep64(X, mu, shape, lpi, model, "fp32")
        loglik.append(float(logZ.sum()))
        lpi = torch.log(Nk / N)
        mu = mu_acc / Nk[:, None]
        if model == "iso":
            shape = torch.log(sig / (D * Nk))
        elif model == "diag":
            shape = torch.log(sig / Nk[:, None])
        else:
            cov = (sig / Nk[:, None, None] - mu[:, :, None] * mu[:, None, :]).cpu().numpy() + 1e-6 * np.eye(D)
            shape = torch.from_numpy(np.linalg.cholesky(np.linalg.inv(cov))).to(X.device)
    return mu, shape, lpi, loglik
