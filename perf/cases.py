"""The work a program has this library do, as cases to be measured.

Every call goes through the Python API (ozablas_amd): FP64 GEMMs emulated with INT8 products by
Scheme I (`ozaki_scheme1_gemm`) and Scheme II (`ozaki_scheme2_gemm`), the BLAS-style `gemm`, a planned
batch of unequal problems (`GroupScheme2`) and the request server (`ServerScheme2`).  Operands are
torch tensors resident on the GPU with the value distribution of the reference generator,
a = (U - 0.5) exp(phi Z); the outputs are the whole products.

A case's "kind" says which entry point it calls; the other keys are its sizes and options.
"""
import math

import torch

import ozablas_amd as oz
from ozablas_amd.workloads import batch_shapes, serve_requests

DEV = "cuda"
_EXECUTOR = None
_SERVER = None


def _executor():
    """A program keeps one library context per device."""
    global _EXECUTOR
    if _EXECUTOR is None:
        _EXECUTOR = oz.HipExecutor(0)
    return _EXECUTOR


def _server():
    """A serving program keeps one server, with its workspace arenas, for as long as it runs."""
    global _SERVER
    if _SERVER is None:
        _SERVER = oz.ServerScheme2(_executor(), 24 << 30, max_batch=64)
    return _SERVER


def listed():
    return [
        # The smallest call of the test configurations: six launches of a few microseconds each.
        {"name": "s2_256", "kind": "scheme2", "M": 256, "N": 256, "K": 256, "S": 4, "phi": 0.5},
        # One block of a factorisation or a solver's panel product at FP64 accuracy: still launch- and latency-bound.
        {"name": "s2_1024", "kind": "scheme2", "M": 1024, "N": 1024, "K": 1024, "S": 16, "phi": 1.0},
        # Odd, unequal sizes: nothing is a multiple of a tile, rows are not 16-byte aligned.
        {"name": "s2_ragged", "kind": "scheme2", "M": 777, "N": 1501, "K": 1003, "S": 14, "phi": 1.0},
        # A mid size of the raw-performance sweep at a moderate moduli count (reduced accuracy, top speed).
        {"name": "s2_2048", "kind": "scheme2", "M": 2048, "N": 2048, "K": 2048, "S": 6, "phi": 1.0},
        # The moduli sweep's size at the count that matches native FP64 accuracy.
        {"name": "s2_4096", "kind": "scheme2", "M": 4096, "N": 4096, "K": 4096, "S": 17, "phi": 1.0},
        # The headline: a large product at native FP64 accuracy.
        {"name": "s2_8192", "kind": "scheme2", "M": 8192, "N": 8192, "K": 8192, "S": 17, "phi": 1.0},
        # Gram-like products of tall operands: few output tiles, long K.
        {"name": "s2_long_k", "kind": "scheme2", "M": 512, "N": 512, "K": 32768, "S": 14, "phi": 1.0},
        # Scheme I on odd, unequal sizes.
        {"name": "s1_ragged", "kind": "scheme1", "M": 1499, "N": 1200, "K": 1801, "S": 8, "phi": 1.0},
        # Scheme I at the size of its slice sweep (the largest case: 36 INT8 products of 8192^3).
        {"name": "s1_8192", "kind": "scheme1", "M": 8192, "N": 8192, "K": 8192, "S": 8, "phi": 2.0},
        # BLAS-style update inside a larger matrix: column-major, A transposed, padded leading dimensions, alpha and beta.
        {"name": "blas_tn", "kind": "blas", "M": 3000, "N": 1000, "K": 2050, "S": 16, "phi": 1.0, "layout": oz.COL_MAJOR,
         "transA": oz.OP_T, "transB": oz.OP_N, "pad": 7, "alpha": 1.5, "beta": 0.5},
        # The batch of 512 unequal GEMMs (M, N, K log-uniform on [64, 2048]), planned once.
        {"name": "group_512", "kind": "group", "n": 512, "lo": 64, "hi": 2048, "shapes_seed": 20261202},
        # A burst of requests of the served stream (M, N, K log-uniform on [128, 8192]), submitted and drained.
        {"name": "serve_96", "kind": "serve", "n": 96, "lo": 128, "hi": 8192, "shapes_seed": 20261203},
    ]


# The listed cases' most costly product: 8192^3 times the 36 slice pairs of 8 slices.
_MOST = 8192.0 ** 3 * 36


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _least_slices(K):
    """The fewest moduli that leave both operands at least 10 bits."""
    return next(S for S in range(1, oz.MAX_SLICES + 1) if oz.scheme2_kparam(S, K) >= 10)


def draw(rng):
    kind = rng.choice(["scheme2", "scheme2", "scheme2", "scheme1", "scheme1", "blas", "blas", "group", "serve"])
    if kind in ("group", "serve"):
        lo, hi = ((64, rng.choice([512, 1024, 2048])) if kind == "group" else (128, rng.choice([2048, 4096, 8192])))
        return {"kind": kind, "n": _log_uniform(rng, 16, 512 if kind == "group" else 64), "lo": lo, "hi": hi,
                "shapes_seed": rng.randrange(1 << 30)}
    if rng.random() < 0.15:  # few output tiles, long K
        M, N, K = _log_uniform(rng, 64, 768), _log_uniform(rng, 64, 768), _log_uniform(rng, 8192, 65536)
    else:
        M, N, K = (_log_uniform(rng, 96, 8192) for _ in range(3))
        if rng.random() < 0.3:  # multiples of 64, as many programs' sizes are
            M, N, K = (max(64, x // 64 * 64) for x in (M, N, K))
    if kind == "scheme1":
        K = min(K, 32768)
        S = rng.randint(3, 10)
        while float(M) * N * K * S * (S + 1) / 2 > _MOST:
            S -= 1
    else:
        S = rng.randint(_least_slices(K), oz.MAX_SLICES)
    case = {"kind": kind, "M": M, "N": N, "K": K, "S": S, "phi": rng.choice([0.5, 1.0, 2.0])}
    if kind == "blas":
        case.update(layout=rng.choice([oz.ROW_MAJOR, oz.COL_MAJOR]), transA=rng.choice([oz.OP_N, oz.OP_T]),
                    transB=rng.choice([oz.OP_N, oz.OP_T]), pad=rng.choice([0, 0, 1, 8, 33]),
                    alpha=rng.choice([1.0, -1.0, 1.5]), beta=rng.choice([0.0, 0.5, -0.25]))
    return case


# ------------------------------------------------------------------------------------ inputs
def _matrix(gen, rows, cols, phi):
    u = torch.rand(rows, cols, dtype=torch.float64, device=DEV, generator=gen)
    z = torch.randn(rows, cols, dtype=torch.float64, device=DEV, generator=gen)
    return u.sub_(0.5).mul_(z.mul_(phi).exp_())


def _shapes(case):
    """[(M, N, K, S, phi)] of a batch or burst."""
    if case["kind"] == "group":
        return [sh[:5] for sh in batch_shapes(n=case["n"], seed=case["shapes_seed"], lo=case["lo"], hi=case["hi"])]
    return [r[1:6] for r in serve_requests(case["n"], 1.0, seed=case["shapes_seed"], lo=case["lo"], hi=case["hi"])]


def _inputs(case, seed):
    """The operand tensors, the same for prepare() and exact()."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    if case["kind"] in ("group", "serve"):
        return [(_matrix(gen, M, K, phi), _matrix(gen, K, N, phi)) for M, N, K, _, phi in _shapes(case)]
    M, N, K, phi = case["M"], case["N"], case["K"], case["phi"]
    if case["kind"] != "blas":
        return _matrix(gen, M, K, phi), _matrix(gen, K, N, phi)
    # Stored matrices, each row (of the row-major view of the storage) padded to its leading dimension.
    (ra, ca), (rb, cb), (rc, cc) = _stored(case)
    p = case["pad"]
    return _matrix(gen, ra, ca + p, phi), _matrix(gen, rb, cb + p, phi), _matrix(gen, rc, cc + p, phi)


def _stored(case):
    """(lines, line length) of A, B and C as stored: lines are rows (row-major) or columns (column-major)."""
    M, N, K = case["M"], case["N"], case["K"]
    a = (M, K) if case["transA"] == oz.OP_N else (K, M)
    b = (K, N) if case["transB"] == oz.OP_N else (N, K)
    c = (M, N)
    return (a, b, c) if case["layout"] == oz.ROW_MAJOR else (a[::-1], b[::-1], c[::-1])


class _Operand:
    """A tensor as the library's calls take it: its device address."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()


def _flat_outputs(shapes):
    """One buffer for all products of a batch, each starting on a 512-byte boundary, and their addresses."""
    offs, n = [], 0
    for M, N, *_ in shapes:
        offs.append(n)
        n += (M * N + 63) // 64 * 64
    out = torch.zeros(n, dtype=torch.float64, device=DEV)
    return out, offs


def prepare(case, seed):
    ex = _executor()
    kind = case["kind"]
    inputs = _inputs(case, seed)
    if kind in ("group", "serve"):
        shapes = _shapes(case)
        out, offs = _flat_outputs(shapes)
        st = {"kind": kind, "inputs": inputs, "out": out, "shapes": [sh[:4] for sh in shapes],
              "A": [a.data_ptr() for a, _ in inputs], "B": [b.data_ptr() for _, b in inputs],
              "C": [out.data_ptr() + 8 * o for o in offs]}
        if kind == "group":
            st["group"] = oz.GroupScheme2(ex, st["shapes"])
        else:
            st["server"] = _server()
        return st
    if kind == "blas":
        A, B, C = inputs
        return {"kind": kind, "ex": ex, "case": case, "A": A, "B": B, "C": C,
                "ws": ex.alloc(oz.gemm_workspace_bytes(2, case["M"], case["N"], case["K"], case["S"]))}
    A, B = inputs
    C = torch.empty(case["M"], case["N"], dtype=torch.float64, device=DEV)
    ws = (oz.WorkspaceScheme1 if kind == "scheme1" else oz.WorkspaceScheme2)(ex, case["M"], case["N"], case["K"], case["S"])
    return {"kind": kind, "ws": ws, "A": _Operand(A), "B": _Operand(B), "C": _Operand(C)}


def run(state):
    kind = state["kind"]
    if kind == "scheme2":
        oz.ozaki_scheme2_gemm(state["ws"], state["A"], state["B"], state["C"])
        return state["C"].t
    if kind == "scheme1":
        oz.ozaki_scheme1_gemm(state["ws"], state["A"], state["B"], state["C"])
        return state["C"].t
    if kind == "blas":
        c, A, B, C = state["case"], state["A"], state["B"], state["C"]
        oz.gemm(state["ex"], c["M"], c["N"], c["K"], c["alpha"], A.data_ptr(), A.shape[1], B.data_ptr(), B.shape[1],
                c["beta"], C.data_ptr(), C.shape[1], transA=c["transA"], transB=c["transB"], layout=c["layout"],
                scheme=2, slices=c["S"], workspace=state["ws"])
        return C
    if kind == "group":
        state["group"].run(state["A"], state["B"], state["C"])
        return state["out"]
    server = state["server"]
    for (M, N, K, S), a, b, c in zip(state["shapes"], state["A"], state["B"], state["C"]):
        server.submit(M, N, K, S, a, b, c)
    server.drain()  # the burst's results are in memory
    return state["out"]


def work(case):
    """FP64 operands read and results written once; the INT8 operations of the scheme's products."""
    if case["kind"] in ("group", "serve"):
        sh = _shapes(case)
        return {"bytes": sum(8.0 * (M * K + K * N + M * N) for M, N, K, _, _ in sh),
                "flops": sum(2.0 * M * N * K * S for M, N, K, S, _ in sh)}
    M, N, K, S = (case[k] for k in ("M", "N", "K", "S"))
    products = S * (S + 1) / 2 if case["kind"] == "scheme1" else S
    c_passes = 2 if case.get("beta", 0.0) != 0.0 else 1
    return {"bytes": 8.0 * (M * K + K * N + c_passes * M * N), "flops": 2.0 * M * N * K * products}


def exact(case, seed):
    inputs = _inputs(case, seed)
    if case["kind"] in ("group", "serve"):
        out, offs = _flat_outputs(_shapes(case))
        for (a, b), o in zip(inputs, offs):
            c = a @ b
            out[o:o + c.numel()] = c.reshape(-1)
        return out
    if case["kind"] != "blas":
        return inputs[0] @ inputs[1]
    A, B, C = inputs
    (_, ca), (_, cb), (_, cc) = _stored(case)
    a, b, c = A[:, :ca], B[:, :cb], C[:, :cc]
    if case["layout"] == oz.COL_MAJOR:
        a, b, c = a.T, b.T, c.T
    a = a.T if case["transA"] == oz.OP_T else a
    b = b.T if case["transB"] == oz.OP_T else b
    c.copy_(case["alpha"] * (a @ b) + case["beta"] * c)  # in place: the padding stays as it was
    return C
