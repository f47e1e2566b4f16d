"""The work a user of this library has it do, as measurable cases.

Each case is one call (or one batch launch) through a public entry point:
the DM-QR factorisation of a matrix resident on the device
(qrdm_amd.dgeqrdm_dev), the drop-in module on numpy arrays (QRDM.QRDM), the
batched form (qrdm_amd.BatchPlan), the unpivoted QR and the application of
its Q (qrdm_dgeqrf_dev, qrdm_dormqr_dev).  All of them are float64.

The inputs have pivots that the data decides, not its rounding: Gaussian
entries, spectra graded over a few decades, or a low rank plus a small noise
with the stopping test on (a rank-revealing use, which ends at the rank).
The reduced-precision trailing updates and the learned thresholds are left
out: on this device they are not faster than the plain path, so they are not
what a program that wants its result would call.
"""
import ctypes
import math

import numpy as np
import torch

DELTA, TAU = 0.9, 0.15  # the reference's demo and the benchmark


def listed():
    """The named cases; `draw` spreads over the ranges they stand for."""
    return [
        # A small solve inside a larger program: launches and latency only.
        _dm("small_64x48", 64, 48),
        # The reference's demo: the drop-in module on a 128 x 128 numpy array.
        _dm("host_128x128", 128, 128, kind="host", family="graded"),
        # The 1024 x 512 fixture shape through the drop-in module: the copies
        # of pageable memory count, as they do for its user.
        _dm("host_1024x512", 1024, 512, kind="host"),
        # An ordinary matrix of odd sizes, packed (the leading dimension is m).
        _dm("ragged_3001x1777", 3001, 1777),
        # Least squares: many more rows than columns, graded spectrum.
        _dm("tall_16384x1024", 16384, 1024, family="graded"),
        # Rank revealing: rank 1024 plus noise, the stopping test ends the loop.
        _dm("lowrank_8192x4096", 8192, 4096, family="lowrank", rank=1024, stop=3),
        # The benchmark's shape, factorised to the last column.
        _dm("square_8192", 8192, 8192),
        # Wider DM blocks than one register tile (the entry points take up to 256).
        _dm("nb128_2048x1024", 2048, 1024, nb=128),
        # The batched form: one launch over many uneven matrices.
        {"name": "batch_1024", "kind": "batch", "count": 1024, "mmax": 1024, "nmax": 512, "nb": 64},
        # The unpivoted QR that the module offers beside the pivoted one.
        {"name": "qrf_1024x1024", "kind": "qrf", "m": 1024, "n": 1024, "lda": 1024},
        {"name": "qrf_4096x2048", "kind": "qrf", "m": 4096, "n": 2048, "lda": 4096},
        # Q formed from the reflectors: what every check and every use of Q does.
        {"name": "formq_4096x2048", "kind": "ormqr", "m": 4096, "k": 2048, "nc": 2048, "trans": 0},
    ]


def _dm(name, m, n, kind="dm", family="gauss", nb=64, rank=0, stop=0, lda=0):
    c = {"kind": kind, "m": m, "n": n, "lda": lda or m, "nb": nb, "family": family, "rank": rank,
         "stop": stop}
    return dict(c, name=name) if name else c


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind, then its sizes over the range (logarithmic)."""
    kind = rng.choice(["dm", "dm", "dm", "dm", "host", "nb", "batch", "qrf", "ormqr"])
    if kind in ("dm", "host", "nb"):
        if kind == "dm":  # square, tall and wide, up to the benchmark's elements
            m = _log(rng, 48, 16384)
            n = min(_log(rng, 32, 8192), 8192 * 8192 // m)
        elif kind == "host":
            m, n = _log(rng, 48, 2048), _log(rng, 32, 1024)
        else:
            m, n = _log(rng, 256, 4096), _log(rng, 192, 2048)
        nb = rng.randint(65, 256) if kind == "nb" else rng.choice([16, 32, 48, 64, 64, 64])
        lda = m + rng.choice([0, 0, -m % 32, rng.randint(1, 40)])  # packed, padded, a part of more
        family = rng.choice(["gauss", "graded", "lowrank"]) if min(m, n) >= 128 else "gauss"
        rank = rng.randint(min(m, n) // 6, min(m, n) // 2) if family == "lowrank" else 0
        return _dm("", m, n, kind="host" if kind == "host" else "dm", family=family, nb=nb,
                   rank=rank, stop=3 if rank else 0, lda=lda)
    if kind == "batch":
        return {"kind": "batch", "count": _log(rng, 16, 1024), "mmax": _log(rng, 128, 1024),
                "nmax": _log(rng, 64, 512), "nb": rng.choice([16, 32, 64, 64])}
    if kind == "qrf":
        m, n = _log(rng, 48, 4096), _log(rng, 32, 2048)
        return {"kind": "qrf", "m": m, "n": n, "lda": m + rng.choice([0, 0, -m % 32])}
    m = _log(rng, 64, 4096)
    k = _log(rng, 16, min(m, 2048))
    return {"kind": "ormqr", "m": m, "k": k, "nc": _log(rng, 1, 2048), "trans": rng.choice([0, 1])}


# ---------------------------------------------------------------- the inputs

def _generator(seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _matrix(case, seed):
    """The m x n matrix as an (n, lda) row-major tensor: its memory is the
    column-major matrix with leading dimension lda."""
    m, n, dev = case["m"], case["n"], _device()
    g = _generator(seed, dev)

    def randn(*shape):
        return torch.randn(*shape, generator=g, dtype=torch.float64, device=dev)

    a = randn(n, case["lda"])
    family = case.get("family", "gauss")
    if family == "graded":  # singular values that fall over about three decades
        k = 2 * min(m, n)
        s = 10.0 ** (-3.0 * torch.arange(k, dtype=torch.float64, device=dev) / k)
        a[:, :m] = (randn(n, k) * s) @ randn(k, m) / math.sqrt(k)
    elif family == "lowrank":
        r = case["rank"]
        a[:, :m] = randn(n, r) @ randn(r, m) + 1e-10 * a[:, :m]
    return a


def _thres(case):
    # stop mode 3: the loop ends once the remaining block is 1e-5 of the
    # largest column (far above the noise, far below the rank's last pivots)
    return np.array([DELTA, TAU, 1e-5])


def _ncols(case):
    nc = np.zeros(case["n"], np.int32)
    nc[0] = case["stop"]
    return nc


def _batch_shapes(case):
    rng = np.random.default_rng(1000003 * case["count"] + 1009 * case["mmax"] + case["nmax"])
    ms = rng.integers(64, case["mmax"] + 1, case["count"])
    ns = [int(rng.integers(32, min(int(m), case["nmax"]) + 1)) for m in ms]
    return [(int(m), n) for m, n in zip(ms, ns)]


def _reflectors(case, seed):
    """k reflectors and their tau as a QR of an m x k matrix leaves them: unit
    lower trapezoidal vectors with entries of the size that Gaussian columns
    give, H = I - tau v v^T orthogonal; R above them.  (k, m) row-major."""
    m, k, dev = case["m"], case["k"], _device()
    g = _generator(seed, dev)
    a = torch.randn(k, m, generator=g, dtype=torch.float64, device=dev)
    col = torch.arange(k, device=dev)[:, None]
    below = torch.arange(m, device=dev)[None, :] > col
    v = torch.where(below, a / torch.sqrt((m - col).to(torch.float64)), torch.zeros_like(a))
    tau = 2.0 / (1.0 + (v * v).sum(1))
    if m == k:
        tau[-1] = 0.0
    return torch.where(below, v, a), tau


def prepare(case, seed):
    """The matrix, the arrays the call fills, and the batch's plan."""
    import qrdm_amd
    kind, s = case["kind"], {"case": case}
    if kind == "batch":
        shapes = _batch_shapes(case)
        s["plan"] = p = qrdm_amd.BatchPlan(shapes, nb=case["nb"])
        g = _generator(seed, "cuda")
        # Gaussian matrices whose column norms spread over a decade
        scale = 10.0 ** -torch.rand(p.col_size, generator=g, dtype=torch.float64, device="cuda")
        rows = torch.repeat_interleave(torch.tensor([m for m, _ in shapes]),
                                       torch.tensor([n for _, n in shapes])).cuda()
        s["a0"] = torch.randn(p.a_size, generator=g, dtype=torch.float64, device="cuda")
        s["a0"] *= torch.repeat_interleave(scale, rows)
        s["a"] = torch.empty_like(s["a0"])
        s["tau"] = torch.zeros(p.tau_size, dtype=torch.float64, device="cuda")
        s["jpvt"], s["ncols"], s["info"] = (
            torch.zeros(k, dtype=torch.int32, device="cuda")
            for k in (p.col_size, p.col_size, len(shapes)))
        return s
    if kind == "ormqr":
        s["v"], s["tau"] = _reflectors(case, seed)
        g = _generator(seed + 1, "cuda")
        m, nc = case["m"], case["nc"]
        if case["trans"]:  # Q^T B, as a least-squares solve does
            s["c0"] = torch.randn(nc, m, generator=g, dtype=torch.float64, device="cuda")
        else:  # Q's leading columns
            s["c0"] = torch.eye(nc, m, dtype=torch.float64, device="cuda")
        s["c"] = torch.empty_like(s["c0"])
        return s
    a = _matrix(case, seed)
    k = min(case["m"], case["n"])
    if kind == "host":
        s["a0"] = a.cpu().numpy()
        s["tau"] = np.zeros(k)
        s["thres"] = _thres(case)
        return s
    s["a0"], s["a"] = a, torch.empty_like(a)
    s["tau"] = torch.zeros(k, dtype=torch.float64, device="cuda")
    if kind == "dm":
        s["thres"] = _thres(case)
    return s


def run(s):
    """One call; in-place entry points get a fresh copy of the matrix."""
    import qrdm_amd
    case = s["case"]
    kind = case["kind"]
    if kind == "host":
        import QRDM
        a, jpvt, ncols = s["a0"].copy(), np.zeros(case["n"], np.int32), _ncols(case)
        info = QRDM.QRDM(102, case["m"], case["n"], a, case["lda"], jpvt, s["tau"], ncols,
                         s["thres"], case["nb"])
        return {"info": info, "a": a[:, :case["m"]], "tau": s["tau"], "jpvt": jpvt, "ncols": ncols}
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "ormqr":
        s["c"].copy_(s["c0"])
        info = qrdm_amd.lib().qrdm_dormqr_dev(
            case["trans"], case["m"], case["nc"], case["k"], s["v"].data_ptr(), case["m"],
            s["tau"].data_ptr(), s["c"].data_ptr(), case["m"], ctypes.c_void_p(stream))
        return {"info": info, "c": s["c"]}
    s["a"].copy_(s["a0"])
    if kind == "qrf":
        info = qrdm_amd.lib().qrdm_dgeqrf_dev(case["m"], case["n"], s["a"].data_ptr(), case["lda"],
                                              s["tau"].data_ptr(), ctypes.c_void_p(stream))
        return {"info": info, "a": s["a"][:, :case["m"]], "tau": s["tau"]}
    if kind == "batch":
        s["plan"].run(s["a"], s["tau"], s["jpvt"], s["ncols"], s["info"], thres=(DELTA, TAU, 0.0),
                      stream=stream)
        return {k: s[k] for k in ("a", "tau", "jpvt", "info")}
    jpvt, ncols = np.zeros(case["n"], np.int32), _ncols(case)
    info, _ = qrdm_amd.dgeqrdm_dev(s["a"], case["m"], s["tau"], jpvt, ncols, s["thres"],
                                   nb=case["nb"], stream=stream)
    return {"info": info, "a": s["a"][:, :case["m"]], "tau": s["tau"], "jpvt": jpvt, "ncols": ncols}


def work(case):
    """The matrix read and written once; the flops of a Householder QR (of the
    leading rank columns where the stopping test ends it), or of Q's use."""
    kind = case["kind"]

    def qr(m, n, k):  # k reflectors applied to an m x n matrix: 4 (m - j)(n - j) each
        return 4.0 * (m * n * k - (m + n) * k * k / 2.0 + k * k * k / 3.0)

    if kind == "batch":
        sh = _batch_shapes(case)
        return {"bytes": sum(16.0 * m * n for m, n in sh), "flops": sum(qr(m, n, n) for m, n in sh)}
    if kind == "ormqr":
        m, k, nc = case["m"], case["k"], case["nc"]
        return {"bytes": 8.0 * (m * k - k * k / 2.0) + 16.0 * m * nc,
                "flops": 4.0 * nc * (m * k - k * k / 2.0)}
    m, n = case["m"], case["n"]
    return {"bytes": 16.0 * m * n, "flops": qr(m, n, case.get("rank") or min(m, n))}


# ------------------------------------------------- the same results, plainly

def _householder(x):
    """LAPACK's reflector of the vector x (in place): returns tau."""
    alpha, below = float(x[0]), float(torch.linalg.vector_norm(x[1:])) if len(x) > 1 else 0.0
    if below == 0.0:
        return 0.0
    beta = -math.copysign(math.hypot(alpha, below), alpha if alpha else 1.0)
    x[1:] /= alpha - beta
    x[0] = beta
    return (beta - alpha) / beta


def _panel(a, j, width, tau, truncate):
    """Householder QR of columns j.. of the (n, m) tensor a (columns are its
    rows), at most `width` of them, then their block reflector on the rest.
    With truncate it ends before a column (not the first) whose part below
    the diagonal is under TAU |R(j, j)|.  Returns the columns reduced."""
    kept, limit = 0, math.inf
    for i in range(width):
        x = a[j + i, j + i:]
        if i and truncate and len(x) > 1 and float(torch.linalg.vector_norm(x[1:])) < limit:
            break
        t = _householder(x)
        tau[j + i] = t
        kept += 1
        if i == 0 and width > 1:
            limit = TAU * abs(float(x[0]))
        v = x.clone()
        v[0] = 1.0
        c = a[j + i + 1:j + width, j + i:]
        c -= torch.outer(c @ v, t * v)
    _apply(a[j:j + kept, j:], tau[j:j + kept], a[j + width:, j:], 1)
    return kept


def _apply(a, tau, c, trans):
    """c (columns as rows) := Q^T c or Q c, Q the k reflectors of a (k, m)."""
    k = len(a)
    v = torch.triu(a, 1)
    v[:, :k].diagonal().fill_(1.0)
    # T^-1 + T^-T = V^T V with tau^-1 on the diagonal (tau = 0: no reflector)
    on = tau != 0
    s = torch.triu(v @ v.T, 1) * on[:, None] * on[None, :]
    s.diagonal().copy_(torch.where(on, 1.0 / torch.where(on, tau, torch.ones_like(tau)),
                                   torch.ones_like(tau)))
    w = (c @ v.T) * on
    w = torch.linalg.solve_triangular(s, w.T, upper=True) if not trans else \
        torch.linalg.solve_triangular(s.T, w.T, upper=False)
    c -= (w.T * on) @ v


def _swaps(selected, n):
    """The reference's walk that brings the accepted columns of n to the
    front, as position swaps: an accepted last column goes forward first, then
    each accepted one to the first position that is still free."""
    marked, swaps = set(selected), []
    free, last = 0, n - 1
    for c in selected:
        while free < last and last in marked:
            swaps.append((last, free))
            if free not in marked:
                marked ^= {last, free}
            while free in marked:
                free += 1
        if c in marked:
            while free in marked:
                free += 1
            if c > free and c >= len(selected):
                swaps.append((c, free))
                marked ^= {c, free}
                free += 1
    return swaps


def _dm_qr(a, nb, stop, eta):
    """Deviation maximisation QR of the (n, m) tensor a, in place."""
    n, m = a.shape
    k = min(m, n)
    jpvt, ncols = list(range(1, n + 1)), []
    tau = torch.zeros(k, dtype=a.dtype, device=a.device)
    first = float(torch.linalg.vector_norm(a, dim=1).max())
    j = 0
    while j < k:
        norms = torch.linalg.vector_norm(a[j:, j:], dim=1)
        val, idx = torch.sort(norms, descending=True, stable=True)
        top = min(nb, m - j, n - j)
        nc = max(1, int((val[:top] > TAU * val[0]).sum()))
        u = a[j + idx[:nc], j:] / val[:nc, None]
        cos = (u @ u.T).abs().cpu().numpy()
        ranks = [0]
        for i in range(1, nc):
            if cos[ranks, i].max() < DELTA:
                ranks.append(i)
        order = idx.cpu().numpy()
        selected = [int(order[r]) for r in ranks]
        where = np.arange(n)
        for p, q in _swaps(selected, n - j):
            jpvt[j + p], jpvt[j + q] = jpvt[j + q], jpvt[j + p]
            where[j + p], where[j + q] = where[j + q], where[j + p]
        moved = np.nonzero(where != np.arange(n))[0]
        if len(moved):
            to = torch.from_numpy(moved).to(a.device)
            a[to] = a[torch.from_numpy(where[moved]).to(a.device)]
        kept = _panel(a, j, len(selected), tau, True)
        ncols.append(kept)
        j += kept
        if stop and j < n:
            rest = float(torch.linalg.vector_norm(a[j:, j:], dim=1).max()) if j < m else 0.0
            if rest * math.sqrt(n - j) <= eta * first:
                break
    return tau, np.array(jpvt, np.int32), ncols


def exact(case, seed):
    """What run() returns, by plain torch operations in 64 bits; None for the
    batch and for sizes whose column-by-column loop takes too long."""
    kind = case["kind"]
    if kind == "batch":
        return None
    if kind == "ormqr":
        v, tau = _reflectors(case, seed)
        m, k, nc = case["m"], case["k"], case["nc"]
        g = _generator(seed + 1, v.device)
        c = torch.randn(nc, m, generator=g, dtype=torch.float64, device=v.device) \
            if case["trans"] else torch.eye(nc, m, dtype=torch.float64, device=v.device)
        blocks = range(0, k, 64)
        for b in blocks if case["trans"] else reversed(blocks):
            e = min(b + 64, k)
            _apply(v[b:e, b:], tau[b:e], c[:, b:], case["trans"])
        return {"info": 0, "c": c}
    m, n = case["m"], case["n"]
    k = min(m, n)
    if k > 4096:
        return None
    a = _matrix(case, seed)[:, :m].contiguous()
    if kind == "qrf":
        tau = torch.zeros(k, dtype=torch.float64, device=a.device)
        for j in range(0, k, 64):
            _panel(a, j, min(64, k - j), tau, False)
        return {"info": 0, "a": a, "tau": tau}
    tau, jpvt, nc = _dm_qr(a, case["nb"], case["stop"], _thres(case)[2])
    ncols = _ncols(case)
    ncols[:len(nc)] = nc
    if kind == "host":
        a, tau = a.cpu().numpy(), tau.cpu().numpy()
    return {"info": 0, "a": a, "tau": tau, "jpvt": jpvt, "ncols": ncols}
