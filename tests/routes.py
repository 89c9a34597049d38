"""Which way a call went: its plan (the library's plan_info queries) and the choice and lists
it left in its workspace."""

import ctypes

from flash_gmm import _lib

DEFAULT, STORED, SCREEN = 0, 1, 2   # CallMode


def plan_info(model, N, K, D, flags=0):
    """iso, diag: (may screen, offset of the choice, offset of the list's length, a short list's
    rows, rows per slab, slabs).  full: (may screen, offset of the probe's counts, their number,
    the largest sum that screens, offset of the tiles' bytes, a pool's log-joints)."""
    info = (ctypes.c_int64 * 6)()
    fn = getattr(_lib.lib(), f"fgmm_{model}_plan_info")
    fn.restype = None
    fn.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_uint, ctypes.POINTER(ctypes.c_int64)]
    fn(N, K, D, flags, info)
    return list(info)


def _words(workspace, offset, n=1):
    return workspace[offset:offset + 4 * n].cpu().numpy().view("int32")


def call_mode(model, workspace, N, K, D, flags=0):
    """The CallMode of the last call on workspace; for iso and diag after phase 1 or a whole
    call, for full too."""
    info = plan_info(model, N, K, D, flags)
    if model == "full":
        if not flags & _lib.FLAG_STORE_LOGJOINT_AUTO:
            return DEFAULT
        total = int(_words(workspace, info[1], info[2]).sum())
        return SCREEN if info[0] and total <= info[3] else STORED if total >= 4 * info[3] else DEFAULT
    return DEFAULT if info[1] < 0 else int(_words(workspace, info[1])[0])


def listed_rows(model, workspace, N, K, D, flags=0):
    """(rows a screened call put on its list, the most that run one tile per workgroup), from
    the workspace of a phase-1 call (pass 2 writes over the list)."""
    info = plan_info(model, N, K, D, flags)
    return int(_words(workspace, info[2])[0]), info[3]


def overflowed_tiles(workspace, N, K, D):
    """The 32-row tiles whose needed pairs a screened full-covariance call found to exceed
    their pool, from the workspace of a phase-1 call."""
    info = plan_info("full", N, K, D, _lib.FLAG_STORE_LOGJOINT_AUTO)
    n = -(-N // 32)
    return workspace[info[4]:info[4] + n].cpu().nonzero().flatten().tolist()
