"""Timing cases of the per-peer matrix pipeline, through the device C ABI (excalibur_amd.hip) and
the host-pointer drop-in (excalibur_amd.bbtsvd).

Each case is one step that a peer runs on data it already holds: masks, local and global QR, the
bidiagonal SVD, the combine, the mixed form's FP32 passes, the SVD of the shared factor, the stage
of many peers on one device, and the bracket network's training step. listed() holds the sizes of
the repository's workloads, draw() gives others of the same ranges, prepare() what a program keeps
on the GPU (inputs, plans, workspaces), run() one pass, work() the bytes and operations the pass
cannot do without, and exact() the same outputs from plain torch or numpy in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

from excalibur_amd import bbtsvd, hip

DEV = "cuda:0"
F64, F32, I32 = torch.float64, torch.float32, torch.int32
PASSES = 32  # mask_times of every mask in the pipeline
lib = hip.lib


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # both masks of one peer's block at the smallest workload (A 1,000 x 100, two peers, N(0,1))
        {"name": "mask-100", "kind": "mask", "m": 100, "n": 100, "f32": False, "mask": True},
        # the same on the 1,000 x 1,000 factor of a 50,000 x 1,000 block (plain form)
        {"name": "mask-1000", "kind": "mask", "m": 1000, "n": 1000, "f32": False, "mask": True},
        # both masks of an FP32 Gram matrix at the short-wide workload (mixed form, A 2,000 x 200,000)
        {"name": "mask-2000-f32", "kind": "mask", "m": 2000, "n": 2000, "f32": True, "mask": True},
        # local QR of one peer's 50,000 x 1,000 block, Q kept, singular values over six decades
        {"name": "local-qr-1000", "kind": "local_qr", "m": 1000, "r": 50000},
        # the two panels of the global QR that merges two peers' 1,000 x 1,000 factors, and its Q
        {"name": "global-qr-1000", "kind": "global_qr", "m": 1000, "peers": 2},
        # the whole SVD of the m x m factor that every peer of the mixed form runs by itself
        {"name": "factor-svd-1000", "kind": "factor_svd", "m": 1000},
        # bidiagonal SVD of the short-wide workload's order, every triplet
        {"name": "bidiag-svd-2000", "kind": "bidiag_svd", "n": 2000, "k": 2000},
        # the drop-in of bidiagonal_bisection_twisted_svd on host arrays, at the smallest workload
        {"name": "bidiag-svd-host-100", "kind": "bidiag_svd_host", "n": 100},
        # combine and unmask of one of two peers: its rows of U, and all of its V (50,000 columns)
        {"name": "combine-1000", "kind": "combine", "m": 1000, "r": 50000},
        # FP32 passes of the mixed form at the short-wide workload: Gram matrix and L^-1 X
        {"name": "fp32-passes-2000", "kind": "fp32_passes", "m": 2000, "r": 100000},
        # local QR and masks of 32 peers' uneven blocks on one device, and the merge of their factors
        {"name": "batched-32x512", "kind": "batched", "peers": 32, "m": 512, "lo": 2000, "hi": 60000},
        # one training step of the bracket network (its minibatch) and its BF16 inference
        {"name": "bracket-net-4096", "kind": "bracket_net", "batch": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mask", "mask", "local_qr", "global_qr", "factor_svd", "bidiag_svd", "bidiag_svd_host",
                       "combine", "fp32_passes", "batched", "bracket_net"])
    if kind == "mask":
        return {"kind": kind, "m": _log_int(rng, 48, 3000), "n": _log_int(rng, 48, 3000),
                "f32": rng.random() < 0.4, "mask": rng.random() < 0.6}
    if kind == "local_qr":
        m = _log_int(rng, 40, 1200)
        return {"kind": kind, "m": m, "r": int(m * math.exp(rng.uniform(math.log(6), math.log(40))))}
    if kind == "global_qr":
        return {"kind": kind, "m": _log_int(rng, 40, 1200), "peers": rng.randint(2, 4)}
    if kind == "factor_svd":
        return {"kind": kind, "m": _log_int(rng, 40, 1200)}
    if kind == "bidiag_svd":
        n = _log_int(rng, 40, 2200)
        return {"kind": kind, "n": n, "k": n if rng.random() < 0.6 else max(1, _log_int(rng, 8, n))}
    if kind == "bidiag_svd_host":
        return {"kind": kind, "n": _log_int(rng, 16, 400)}
    if kind == "combine":
        m = _log_int(rng, 40, 1200)
        return {"kind": kind, "m": m, "r": int(m * math.exp(rng.uniform(math.log(6), math.log(40))))}
    if kind == "fp32_passes":
        m = _log_int(rng, 64, 2000)
        return {"kind": kind, "m": m, "r": int(m * math.exp(rng.uniform(math.log(6), math.log(50))))}
    if kind == "batched":
        m = _log_int(rng, 64, 512)
        return {"kind": kind, "peers": rng.randint(2, 32), "m": m, "lo": 6 * m, "hi": _log_int(rng, 12 * m, 100 * m)}
    return {"kind": kind, "batch": _log_int(rng, 64, 65536)}


# ------------------------------------------------------------------ helpers
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=F64)


def _orthogonal(g, n):
    return torch.linalg.qr(_randn(g, n, n))[0].contiguous()


def _empty(*shape, dtype=F64):
    return torch.zeros(*shape, device=DEV, dtype=dtype)


def _work(nbytes):
    return torch.empty(max(int(nbytes), 256), device=DEV, dtype=torch.uint8)


def _p(t, offset=0):
    """Device address of element `offset` of a contiguous tensor."""
    return t.data_ptr() + offset * t.element_size()


def _plan(K, mask, seed):
    """The public or private mask's plan for K lines on the GPU: pairs and (c, s) of every pass."""
    pairs, cs = hip.givens_plan(K, PASSES, mask, seed & 0x7FFFFFFF)
    return torch.from_numpy(pairs).to(DEV), torch.from_numpy(cs).to(DEV)


def _sweep(x, plan, mask, is_left):
    name = "exc_givens_apply_f32" if x.dtype == F32 else "exc_givens_apply"
    hip.call(name, _p(x), x.shape[0], x.shape[1], _p(plan[0]), _p(plan[1]), PASSES, int(mask), int(is_left), None)


def _rotate(x, plan, mask, is_left):
    """The sweep in plain torch: the pairs of one pass are disjoint, except that for an odd number
    of lines one pair repeats a line, which comes last (mask) or first (unmask)."""
    x = x.to(F64).clone() if is_left else x.to(F64).t().contiguous()
    pairs, cs = plan[0].long(), plan[1]
    K = x.shape[0]
    half = pairs.shape[1]
    if K % 2 == 0:
        steps = [slice(0, half)]
    else:
        steps = [slice(0, half - 1), slice(half - 1, half)] if mask else [slice(0, 1), slice(1, half)]
    sgn = 1.0 if mask else -1.0
    for p in range(pairs.shape[0]):
        for st in steps:
            i, j = pairs[p, st, 0], pairs[p, st, 1]
            c, s = cs[p, st, 0][:, None], sgn * cs[p, st, 1][:, None]
            a, b = x[i], x[j]
            x[i] = c * a + s * b
            x[j] = c * b - s * a
    return x if is_left else x.t().contiguous()


def _householders(g, m):
    """House (m x m, reflector j in column j below the diagonal) and tau of m orthogonal reflectors."""
    v = torch.tril(_randn(g, m, m), -1)
    v = v / torch.sqrt(torch.tensor(float(m), device=DEV, dtype=F64))
    tau = 2.0 / (1.0 + (v * v).sum(0))
    v = v + torch.triu(_randn(g, m, m))  # what the bidiagonalization leaves above is not part of H
    tau[0] = 0.0  # the bidiagonalization's first reflector is the identity
    return v.contiguous(), tau.contiguous()


def _split(m, peers):
    """m_part of the run: m lines over the peers, the last one taking the rest."""
    return [m // peers] * (peers - 1) + [m - (m // peers) * (peers - 1)]


# ------------------------------------------------------------------ prepare / run / exact by kind
def _mask_prepare(c, seed):
    g = _gen(seed)
    x = _randn(g, c["m"], c["n"])
    return {"x": x.to(F32) if c["f32"] else x, "left": _plan(c["m"], c["mask"], seed),
            "right": _plan(c["n"], c["mask"], seed + 1), "mask": c["mask"]}


def _mask_run(s):
    for left in (True, False) if s["mask"] else (False, True):
        _sweep(s["x"], s["left" if left else "right"], s["mask"], left)
    return s["x"]


def _mask_exact(c, seed):
    s = _mask_prepare(c, seed)
    x = s["x"]
    for left in (True, False) if c["mask"] else (False, True):
        x = _rotate(x, s["left" if left else "right"], c["mask"], left)
    return x


def _graded(g, m, r):
    """An m x r block whose singular values fall over about six decades."""
    sigma = 10.0 ** (-6.0 * torch.arange(m, device=DEV, dtype=F64) / max(1, m - 1))
    return torch.mm(_orthogonal(g, m) * sigma, _randn(g, m, r)) / math.sqrt(r)


def _local_qr_prepare(c, seed):
    m, r = c["m"], c["r"]
    return {"m": m, "r": r, "x": _graded(_gen(seed), m, r), "rt": _empty(m, m), "qt": _empty(m, r),
            "ws": _work(lib.exc_qr_t_workspace(m, r, 1))}


def _local_qr_run(s):
    hip.call("exc_qr_t", s["m"], s["r"], _p(s["x"]), s["r"], _p(s["rt"]), _p(s["qt"]), s["r"], None, 0, None, None, 0,
             _p(s["ws"]), s["ws"].numel(), None)
    return {"rt": s["rt"], "qt": s["qt"]}


def _local_qr_exact(c, seed):
    q, r = np.linalg.qr(_graded(_gen(seed), c["m"], c["r"]).cpu().numpy().T)
    return {"rt": np.ascontiguousarray(r.T), "qt": np.ascontiguousarray(q.T)}


def _global_qr_prepare(c, seed):
    m, P = c["m"], c["peers"]
    R = m * P
    wb = max(max(lib.exc_qr_t_workspace(k, R, 0) for k in set(_split(m, P))), lib.exc_wy_workspace(m, R, m))
    return {"m": m, "R": R, "parts": _split(m, P), "a": _randn(_gen(seed), m, R), "p": _empty(m, R),
            "rt": _empty(m, m), "vt": _empty(m, R), "tau": _empty(m), "qt": _empty(m, R), "ws": _work(wb)}


def _global_qr_run(s):
    m, R, p, vt, tau, rt = s["m"], s["R"], s["p"], s["vt"], s["tau"], s["rt"]
    ws, wb = _p(s["ws"]), s["ws"].numel()
    hip.call("exc_memcpy_d2d", _p(p), _p(s["a"]), m * R * 8, None)
    pos = 0
    for i, ci in enumerate(s["parts"]):
        L, at = R - pos, pos * R + pos
        hip.call("exc_qr_t", ci, L, _p(p, at), R, _p(rt), None, 0, _p(vt, at), R, _p(tau, pos), None, 1, ws, wb, None)
        hip.call("exc_copy2d", ci, ci, _p(rt), ci, _p(p, at), R, None)
        hip.call("exc_fill2d", ci, L - ci, 0.0, _p(p, at + ci), R, None)
        nxt = pos + ci
        for cj in s["parts"][i + 1:]:  # every later peer's panel
            hip.call("exc_apply_q_right", cj, L, ci, _p(p, nxt * R + pos), R, _p(vt, at), R, _p(tau, pos), ws, wb, None)
            nxt += cj
        pos += ci
    hip.call("exc_orgqr_t", m, R, _p(vt), R, _p(tau), _p(s["qt"]), R, ws, wb, None)
    return {"rt": p, "qt": s["qt"], "tau": tau}


def _global_qr_exact(c, seed):
    m, R = c["m"], c["m"] * c["peers"]
    a = _randn(_gen(seed), m, R).cpu().numpy().T
    tau = np.linalg.qr(a, mode="raw")[1]
    q, r = np.linalg.qr(a)
    rt = np.zeros((m, R))
    rt[:, :m] = r.T
    return {"rt": rt, "qt": np.ascontiguousarray(q.T), "tau": tau}


def _factor(seed, m):
    """The lower-triangular factor L (A A^T = L L^T) of N(0,1) rows."""
    a = _randn(_gen(seed), m, 3 * m)
    return torch.linalg.cholesky(torch.mm(a, a.t())).contiguous()


def _factor_svd_prepare(c, seed):
    m = c["m"]
    link = ctypes.c_void_p()
    hip.call("exc_ralha_link_alloc", m, ctypes.byref(link))
    wb = max(lib.exc_bidiag_local_workspace(m, m), lib.exc_bidiag_svd_workspace(m, m),
             lib.exc_ormqr_house_workspace(m, m), lib.exc_gemm_workspace(m, m, m), lib.exc_oa_refine_workspace(m))
    s = {k: _empty(m, m) for k in ("f", "u0", "house", "bu", "bv", "pm", "u", "w")}
    s.update({k: _empty(n) for k, n in (("tau", m), ("alpha", m), ("beta", m), ("cs", 2 * m), ("flip", m),
                                       ("sigma", m))})
    s.update(m=m, lt=_factor(seed, m), link=_Link(link), ws=_work(wb))
    return s


class _Link:
    """A loop link buffer, freed with the state that holds it."""

    def __init__(self, ptr):
        self.ptr = ptr

    def __del__(self):
        lib.exc_ralha_link_free(self.ptr)


def _factor_svd_run(s):
    m, ws, wb = s["m"], _p(s["ws"]), s["ws"].numel()
    hip.call("exc_memcpy_d2d", _p(s["f"]), _p(s["lt"]), m * m * 8, None)
    hip.call("exc_bidiag_local", m, m, _p(s["f"]), _p(s["u0"]), _p(s["house"]), _p(s["tau"]), _p(s["alpha"]),
             _p(s["beta"]), _p(s["cs"]), s["link"].ptr, 1, ws, wb, 30.0, None)
    hip.call("exc_bidiag_svd", m, _p(s["alpha"]), _p(s["beta"]), _p(s["bu"]), _p(s["bv"]), _p(s["sigma"]), m, None, ws,
             wb, None)
    hip.call("exc_sign_normalize", m, m, _p(s["bu"]), _p(s["bv"]), _p(s["flip"]), None)
    hip.call("exc_dgemm", 0, 1, m, m, m, 1.0, _p(s["u0"]), m, _p(s["bv"]), m, 0.0, _p(s["u"]), m, ws, wb, None)
    hip.call("exc_fill2d", m, m, 0.0, _p(s["pm"]), m, None)
    hip.call("exc_add_diag", m, _p(s["pm"]), m, 1.0, None)
    hip.call("exc_rot_back", m, m, _p(s["pm"]), _p(s["cs"]), None)
    hip.call("exc_ormqr_house_ln", m, m, _p(s["house"]), _p(s["tau"]), _p(s["pm"]), m, ws, wb, None)
    hip.call("exc_dgemm", 0, 0, m, m, m, 1.0, _p(s["pm"]), m, _p(s["bu"]), m, 0.0, _p(s["w"]), m, ws, wb, None)
    hip.call("exc_oa_refine", m, _p(s["lt"]), m, 1, _p(s["u"]), m, _p(s["w"]), m, _p(s["sigma"]), 2, 1e-6, 1e-4, ws, wb,
             None)
    return {"sigma": s["sigma"], "u": s["u"], "w": s["w"]}


def _factor_svd_exact(c, seed):
    # the signs of a pair of vectors follow from the bidiagonal form, so only the values are given
    return {"sigma": np.linalg.svd(_factor(seed, c["m"]).cpu().numpy(), compute_uv=False), "u": None, "w": None}


def _bidiagonal(seed, n):
    """The upper bidiagonal form of an n x n matrix of N(0,1) entries: chi-distributed entries."""
    rng = np.random.default_rng(seed)
    return np.sqrt(rng.chisquare(np.arange(n, 0, -1))), np.sqrt(rng.chisquare(np.arange(n - 1, 0, -1)))


def _bidiag_svd_prepare(c, seed):
    n, k = c["n"], c["k"]
    a, b = _bidiagonal(seed, n)
    return {"n": n, "k": k, "a": torch.from_numpy(a).to(DEV), "b": torch.from_numpy(np.append(b, 0.0)).to(DEV),
            "u": _empty(n, k), "v": _empty(k, n), "sigma": _empty(k), "twists": _empty(2 * k, dtype=I32),
            "ws": _work(lib.exc_bidiag_svd_workspace(n, k))}


def _bidiag_svd_run(s):
    hip.call("exc_bidiag_svd", s["n"], _p(s["a"]), _p(s["b"]), _p(s["u"]), _p(s["v"]), _p(s["sigma"]), s["k"],
             _p(s["twists"]), _p(s["ws"]), s["ws"].numel(), None)
    return {k: s[k] for k in ("sigma", "u", "v", "twists")}


def _bidiag_values(n, k, seed):
    a, b = _bidiagonal(seed, n)
    return np.linalg.svd(np.diag(a) + np.diag(b, 1), compute_uv=False)[:k]


def _bidiag_svd_exact(c, seed):
    # a vector's sign follows from the bidiagonal's own recurrences, so only the values are given
    return {"sigma": _bidiag_values(c["n"], c["k"], seed), "u": None, "v": None, "twists": None}


def _bidiag_svd_host_prepare(c, seed):
    return (c["n"],) + _bidiagonal(seed, c["n"])


def _bidiag_svd_host_run(s):
    n, a, b = s
    return bbtsvd.bidiagonal_bisection_twisted_svd(n, a, b, n)


def _bidiag_svd_host_exact(c, seed):
    return None, None, _bidiag_values(c["n"], c["n"], seed)


def _combine_prepare(c, seed):
    m, r = c["m"], c["r"]
    g = _gen(seed)
    half = m // 2
    angle = _randn(g, m - 1)
    house, tau = _householders(g, m)
    return {"m": m, "r": r, "c": half, "u0": _orthogonal(g, m)[:half].contiguous(), "bv": _orthogonal(g, m),
            "received": _orthogonal(g, m)[half:].contiguous(), "bu0": _orthogonal(g, m), "bu": _empty(m, m),
            "cs": torch.stack([torch.cos(angle), torch.sin(angle)], 1).reshape(-1).contiguous(), "house": house,
            "tau": tau, "qg": _randn(g, m, 2 * m) / math.sqrt(2.0 * m), "qt": _randn(g, m, r) / math.sqrt(r),
            "u": _empty(m, m), "tmp": _empty(m, m), "vt": _empty(m, r), "left": _plan(m, False, seed),
            "right": _plan(m, False, seed + 1),
            "ws": _work(max(lib.exc_ormqr_house_workspace(m, m), lib.exc_gemm_workspace(m, m, m)))}


def _combine_run(s):
    m, r, c, ws, wb = s["m"], s["r"], s["c"], _p(s["ws"]), s["ws"].numel()
    hip.call("exc_dgemm", 0, 1, c, m, m, 1.0, _p(s["u0"]), m, _p(s["bv"]), m, 0.0, _p(s["u"]), m, ws, wb, None)
    hip.call("exc_memcpy_d2d", _p(s["u"], c * m), _p(s["received"]), (m - c) * m * 8, None)
    _sweep(s["u"], s["left"], False, True)
    hip.call("exc_memcpy_d2d", _p(s["bu"]), _p(s["bu0"]), m * m * 8, None)
    hip.call("exc_rot_back", m, m, _p(s["bu"]), _p(s["cs"]), None)
    hip.call("exc_ormqr_house_ln", m, m, _p(s["house"]), _p(s["tau"]), _p(s["bu"]), m, ws, wb, None)
    hip.call("exc_dgemm", 1, 0, m, m, m, 1.0, _p(s["bu"]), m, _p(s["qg"], m), 2 * m, 0.0, _p(s["tmp"]), m, ws, wb, None)
    _sweep(s["tmp"], s["right"], False, False)
    hip.call("exc_dgemm", 0, 0, m, r, m, 1.0, _p(s["tmp"]), m, _p(s["qt"]), r, 0.0, _p(s["vt"]), r, None, 0, None)
    return {"u": s["u"], "vt": s["vt"]}


def _combine_exact(c, seed):
    s = _combine_prepare(c, seed)
    m = s["m"]
    own = torch.mm(s["u0"], s["bv"].t().contiguous())
    u = _rotate(torch.cat([own, s["received"]]), s["left"], False, True)
    b, cs = s["bu0"].clone(), s["cs"].cpu().numpy()
    for i in range(m - 2, -1, -1):
        x, y = b[i].clone(), b[i + 1].clone()
        b[i] = cs[2 * i] * x - cs[2 * i + 1] * y
        b[i + 1] = cs[2 * i] * y + cs[2 * i + 1] * x
    v = torch.tril(s["house"], -1) + torch.eye(m, device=DEV, dtype=F64)
    for j in range(m - 1, -1, -1):
        h = v[j:, j]
        b[j:] -= s["tau"][j] * torch.outer(h, torch.mv(b[j:].t().contiguous(), h))
    t = _rotate(torch.mm(b.t().contiguous(), s["qg"][:, m:].contiguous()), s["right"], False, False)
    return {"u": u, "vt": torch.mm(t, s["qt"])}


def _fp32_passes_prepare(c, seed):
    m, r = c["m"], c["r"]
    x = _randn(_gen(seed), m, r)
    low = torch.linalg.cholesky(torch.mm(x, x.t()))
    li = torch.linalg.solve_triangular(low, torch.eye(m, device=DEV, dtype=F64), upper=False)
    return {"m": m, "r": r, "x": x, "li": li.to(F32).contiguous(), "x32": _empty(m, r, dtype=F32),
            "g": _empty(m, m, dtype=F32), "packed": _empty(m * (m + 1) // 2, dtype=F32), "y": _empty(m, r, dtype=F32),
            "ws": _work(lib.exc_gemm_workspace(m, m, r))}


def _fp32_passes_run(s):
    m, r, ws, wb = s["m"], s["r"], _p(s["ws"]), s["ws"].numel()
    hip.call("exc_convert_f64_f32", m, r, _p(s["x"]), r, _p(s["x32"]), r, None)
    hip.call("exc_sgemm", 0, 1, m, m, r, 1.0, _p(s["x32"]), r, _p(s["x32"]), r, 0.0, _p(s["g"]), m, ws, wb, None)
    hip.call("exc_pack_lower_f32", m, _p(s["g"]), m, _p(s["packed"]), None)
    hip.call("exc_sgemm", 0, 0, m, r, m, 1.0, _p(s["li"]), m, _p(s["x32"]), r, 0.0, _p(s["y"]), r, None, 0, None)
    return {"gram": s["packed"], "y": s["y"]}


def _fp32_passes_exact(c, seed):
    s = _fp32_passes_prepare(c, seed)
    x = s["x"].to(F32).to(F64)
    i, j = torch.tril_indices(c["m"], c["m"], device=DEV)
    return {"gram": torch.mm(x, x.t())[i, j], "y": torch.mm(s["li"].to(F64), x)}


def _batched_cols(c):
    return np.random.default_rng([c["peers"], c["m"], c["lo"], c["hi"]]).integers(c["lo"], c["hi"] + 1, c["peers"])


def _batched_blocks(c, seed):
    g, m = _gen(seed), c["m"]
    return [_randn(g, m, int(k)) * torch.exp(_randn(g, 1)) for k in _batched_cols(c)]


def _batched_prepare(c, seed):
    P, m = c["peers"], c["m"]
    x = _batched_blocks(c, seed)
    cols = (ctypes.c_long * P)(*[b.shape[1] for b in x])
    qt = _empty(m * sum(b.shape[1] for b in x))
    starts = np.cumsum([0] + [m * b.shape[1] for b in x[:-1]])
    rt, masked = _empty(P, m, m), _empty(P, m, m)
    public, private = _plan(m, True, seed), [_plan(m, True, seed + 1 + b) for b in range(P)]

    def device(addresses):
        return torch.tensor(addresses, dtype=torch.int64, device=DEV)

    return {"peers": P, "m": m, "x": x, "cols": cols, "qt": qt, "rt": rt, "masked": masked,
            "hx": (ctypes.c_void_p * P)(*[_p(b) for b in x]),
            "hr": (ctypes.c_void_p * P)(*[_p(rt, b * m * m) for b in range(P)]),
            "hq": (ctypes.c_void_p * P)(*[_p(qt, int(o)) for o in starts]),
            "plans": [public] + private, "xs": device([_p(masked, b * m * m) for b in range(P)]),
            "left": (device([_p(public[0])] * P), device([_p(public[1])] * P)),
            "right": (device([_p(q[0]) for q in private]), device([_p(q[1]) for q in private])),
            "cat": _empty(m, P * m), "merged": _empty(m, m),
            "ws": _work(max(lib.exc_batched_local_qr_workspace(P, m, cols), lib.exc_qr_t_workspace(m, P * m, 0)))}


def _batched_run(s):
    P, m, ws, wb = s["peers"], s["m"], _p(s["ws"]), s["ws"].numel()
    hip.call("exc_batched_local_qr", P, m, s["cols"], s["hx"], s["hr"], s["hq"], None, ws, wb, None)
    hip.call("exc_memcpy_d2d", _p(s["masked"]), _p(s["rt"]), P * m * m * 8, None)
    for left in (True, False):
        plan = s["left" if left else "right"]
        hip.call("exc_givens_apply_batched", P, _p(s["xs"]), m, m, _p(plan[0]), _p(plan[1]), PASSES, 1, int(left), None)
    for b in range(P):
        hip.call("exc_copy2d", m, m, _p(s["masked"], b * m * m), m, _p(s["cat"], b * m), P * m, None)
    hip.call("exc_qr_t", m, P * m, _p(s["cat"]), P * m, _p(s["merged"]), None, 0, None, 0, None, None, 0, ws, wb, None)
    return {"rt": s["rt"], "qt": s["qt"], "masked": s["masked"], "merged": s["merged"]}


def _batched_exact(c, seed):
    P, m = c["peers"], c["m"]
    public, private = _plan(m, True, seed), [_plan(m, True, seed + 1 + b) for b in range(P)]
    rt, qt, masked = [], [], []
    for b, x in enumerate(_batched_blocks(c, seed)):
        low = torch.linalg.cholesky(torch.mm(x, x.t()))
        rt.append(low)
        qt.append(torch.linalg.solve_triangular(low, x, upper=False).reshape(-1))
        masked.append(_rotate(_rotate(low, public, True, True), private[b], True, False))
    r = np.linalg.qr(torch.cat(masked, 1).cpu().numpy().T, mode="r")
    return {"rt": torch.stack(rt), "qt": torch.cat(qt), "masked": torch.stack(masked),
            "merged": np.ascontiguousarray(r.T)}


_LAYERS = ((32, 256), (256, 256), (256, 2))
_ADAM = (1e-3, 0.9, 0.999, 1e-8)


def _net_inputs(c, seed):
    g, B = _gen(seed), c["batch"]
    parts = []
    for rows, cols in _LAYERS:
        parts += [(_randn(g, rows * cols) * math.sqrt(2.0 / rows)), 0.01 * _randn(g, cols)]
    p = torch.cat(parts).to(F32)
    # features: a falling counting function at 29 shifts, the rank fraction, its position, one
    x = torch.rand(B, 32, generator=g, device=DEV, dtype=F64)
    x[:, :29] = torch.sort(x[:, :29], 1, descending=True)[0]
    x[:, 30] = -x[:, 30]
    x[:, 31] = 1.0
    y = x[:, 30] + 0.05 * _randn(g, B)
    return p, x.to(F32).contiguous(), y.to(F32).contiguous(), (1e-2 * _randn(g, p.numel())).to(F32), (
        1e-4 * (1.0 + torch.rand(p.numel(), generator=g, device=DEV, dtype=F64))).to(F32)


def _bracket_net_prepare(c, seed):
    B = c["batch"]
    p, x, y, m, v = _net_inputs(c, seed)
    return {"B": B, "p": p, "x": x, "y": y, "m": m, "v": v, "step": 100,
            "acts": _empty(lib.exc_mlp_acts_floats(B), dtype=F32), "out": _empty(2 * B, dtype=F32),
            "grad": _empty(p.numel(), dtype=F32), "loss": _empty(1, dtype=F32),
            "scratch": _empty(lib.exc_mlp_backward_scratch_floats(B), dtype=F32),
            "bf16": _empty(p.numel(), dtype=torch.bfloat16), "infer": _empty(2 * B, dtype=F32),
            "ws": _work(lib.exc_gemm_workspace(256, 256, B))}


def _bracket_net_run(s):
    B, x, ws, wb = s["B"], _p(s["x"]), _p(s["ws"]), s["ws"].numel()
    hip.call("exc_mlp_to_bf16", _p(s["p"]), _p(s["bf16"]), None)
    hip.call("exc_mlp_infer_bf16", B, x, _p(s["bf16"]), _p(s["infer"]), None)
    hip.call("exc_mlp_forward", B, x, _p(s["p"]), _p(s["acts"]), _p(s["out"]), ws, wb, None)
    hip.call("exc_mlp_backward", B, x, _p(s["y"]), _p(s["p"]), _p(s["acts"]), _p(s["out"]), _p(s["grad"]),
             _p(s["scratch"]), _p(s["loss"]), ws, wb, None)
    s["step"] += 1
    hip.call("exc_mlp_adam", _p(s["p"]), _p(s["grad"]), _p(s["m"]), _p(s["v"]), *_ADAM, s["step"], None)
    return {k: s[k] for k in ("infer", "out", "loss", "grad", "p", "m", "v")}


def _bracket_net_exact(c, seed):
    p, x, y, m, v = (t.to(F64) for t in _net_inputs(c, seed))
    p.requires_grad_(True)
    h, o = x, 0
    for i, (rows, cols) in enumerate(_LAYERS):
        w, b = p[o:o + rows * cols].reshape(rows, cols), p[o + rows * cols:o + (rows + 1) * cols]
        h = torch.mm(h, w) + b
        h = torch.relu(h) if i < 2 else h
        o += (rows + 1) * cols
    loss = (torch.abs(y - h[:, 0]) * torch.exp(-h[:, 1]) + h[:, 1]).mean()
    g, = torch.autograd.grad(loss, p)
    lr, b1, b2, eps = _ADAM
    m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
    p = p.detach() - lr * (m / (1 - b1 ** 101)) / (torch.sqrt(v / (1 - b2 ** 101)) + eps)
    return {"infer": h.detach().reshape(-1), "out": h.detach().reshape(-1), "loss": loss.detach().reshape(1), "grad": g, "p": p, "m": m,
            "v": v}


# ------------------------------------------------------------------ work of one pass
def _mask_work(c):
    m, n, s = c["m"], c["n"], 4 if c["f32"] else 8
    rot = PASSES * (((m + 1) // 2) * n + ((n + 1) // 2) * m)
    return 2 * s * m * n + 24 * PASSES * ((m + 1) // 2 + (n + 1) // 2), 6 * rot


def _local_qr_work(c):
    m, r = c["m"], c["r"]
    return 8 * (2 * m * r + m * m), 4.0 * m * m * r - 4.0 * m ** 3 / 3  # R, then Q


def _global_qr_work(c):
    m, R = c["m"], c["m"] * c["peers"]
    return 8 * (3 * m * R + m), 4.0 * m * m * R - 4.0 * m ** 3 / 3


def _factor_svd_work(c):
    m = c["m"]
    # bidiagonal form, its SVD (55 bisection levels and the twisted vectors), U, W and one refinement
    return 8 * (3 * m * m + m), 8.0 * m ** 3 / 3 + 365.0 * m * m + 4.0 * m ** 3 + 10.0 * m ** 3


def _bidiag_svd_work(c):
    n, k = c["n"], c.get("k", c["n"])
    return 8 * (2 * n + 2 * n * k + k), 365.0 * n * k


def _combine_work(c):
    m, r = c["m"], c["r"]
    return 8 * (2 * m * r + 5 * m * m + m * (m // 2) * 2), 2.0 * m * m * r + 5.0 * m ** 3


def _fp32_passes_work(c):
    m, r = c["m"], c["r"]
    return 8 * m * r + 4 * m * r + 4 * m * m, 2.0 * m * m * r  # both products are triangular


def _batched_work(c):
    m, P, r = c["m"], c["peers"], c["peers"] * (c["lo"] + c["hi"]) // 2
    return 8 * (2 * m * r + 2 * P * m * m + m * m), 4.0 * m * m * r + P * 12.0 * PASSES * m * m / 2 + 2.0 * P * m ** 3


def _bracket_net_work(c):
    w = sum(a * b for a, b in _LAYERS)
    return 4 * (34 * c["batch"] + 4 * c["batch"]) + 4 * 8 * w, 8.0 * c["batch"] * w


# ------------------------------------------------------------------ dispatch
def prepare(case, seed):
    """The state a program holds before the call: a dict (or tuple) with the case's kind."""
    return case["kind"], globals()["_%s_prepare" % case["kind"]](case, seed)


def run(state):
    return globals()["_%s_run" % state[0]](state[1])


def exact(case, seed):
    return globals()["_%s_exact" % case["kind"]](case, seed)


def work(case):
    kind = "bidiag_svd" if case["kind"] == "bidiag_svd_host" else case["kind"]
    nbytes, flops = globals()["_%s_work" % kind](case)
    return {"bytes": float(nbytes), "flops": float(flops)}
