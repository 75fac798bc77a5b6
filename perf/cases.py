"""The work that is timed when this library's speed is looked at.

Each case is a dict of plain values; prepare() builds its inputs on the GPU
from a seed, run() makes one pass through the library's public entry points
and returns what they compute, exact() gives the same results in 64 bits with
plain torch / numpy, and work() the bytes and operations a pass cannot do
without.  listed() holds one or two sizes of every kind, draw() gives more
of the same ranges.

The kinds, and what each stands for:

  action   one resolvent action of a small operator, host sketch in and host
           response out (set_sketch, direct or adjoint, get_Y): the whole
           engine, bound by launches and serial time steps
  step     RK4 steps (four Horner stages each) of the N x k test-vector block
           of a discretised flow operator: the inner loop of every large
           action; with several blocks and no forcing, the e^{A dT} steps of
           the transient removal
  coef     the small-coefficient product that makes a chunk of forcing
           samples from the frequency blocks, or the snapshot DFT
  qr       QR of every frequency block (between the actions of a power
           iteration)
  svd      the SVDs of the k x k factors of all frequencies
  project  the Galerkin projection of the transient removal for a group of
           test vectors: relayout, inner products, shifted solves, products
  weights  a sparse weight, input or output matrix times all frequency blocks
  layer    one layer of the learned-sketch network: forward, backward,
           weight and bias gradients
"""
import ctypes
import functools
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG_DIR = os.path.join(ROOT, "rsvd-delta-t_amd")
DEV = "cuda"

V = ctypes.c_void_p
I64 = ctypes.c_int64
INT = ctypes.c_int
DBL = ctypes.c_double


# --------------------------------------------------------------------------
# the library
def _load(name, path):
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def _pkg():
    return _load("rsvdt_amd", os.path.join(PKG_DIR, "__init__.py"))


def _workloads():
    return _load("rsvdt_workloads", os.path.join(PKG_DIR, "workloads.py"))


class SpmmDesc(ctypes.Structure):
    """rsvdt_spmm_desc of include/rsvdt_hip.h."""
    _fields_ = [("nrows", I64), ("k", I64), ("nb", I64), ("rowptr", V), ("col", V), ("val", V), ("a_real", INT),
                ("prec", INT), ("lanes", INT), ("xcd_remap", INT), ("variant", INT), ("group", INT), ("gptr", V),
                ("gword", V), ("gval", V), ("tile_rows", INT), ("tile_hmax", INT), ("tile_emax", INT), ("tptr", V),
                ("tcol", V), ("lidx", V), ("tile_bpw", INT)]


@functools.lru_cache(None)
def _lib():
    """The kernel-level C ABI (include/rsvdt_hip.h) with its argument types."""
    L = _pkg().lib()
    proto = {
        "rsvdt_hip_init": [INT],
        "rsvdt_hip_horner_stage": [ctypes.POINTER(SpmmDesc), V, V, V, V, DBL, V, V, V],
        "rsvdt_hip_coef_gemm": [I64, I64, I64, V, I64, I64, I64, INT, I64, DBL, V, I64, V, I64, INT, DBL, V],
        "rsvdt_hip_bgram": [I64] * 4 + [V, I64, I64, I64, V, I64, I64, I64, V, V, V],
        "rsvdt_hip_bgram_work_bytes": [I64] * 4,
        "rsvdt_hip_bapply": [I64] * 4 + [V, I64, I64, I64, V, DBL, V, I64, I64, I64, V, I64, I64, I64, V],
        "rsvdt_hip_bjacobi_svd": [I64, I64, V, V, V, V],
        "rsvdt_hip_bshift_solve": [I64, I64, I64, V, V, V, V, V, V, V],
        "rsvdt_hip_bshift_solve_work_bytes": [I64] * 3,
        "rsvdt_hip_transpose_rows": [I64] * 5 + [V, V, INT, V],
        "rsvdt_hip_zscale": [I64, DBL, V, V, V],
        "rsvdt_hip_spmm_blocks": [I64] * 3 + [V, V, V, V, I64, V, I64, V],
        "rsvdt_hip_gemm_bf16": [I64] * 3 + [V, I64, I64, V, I64, I64, V, I64, INT, V, V, I64, V],
        "rsvdt_hip_colsum": [I64, I64, V, I64, V, V],
        "rsvdt_qr_blocks_noalloc": [V, I64, I64, I64, V],
    }
    for name, types in proto.items():
        getattr(L, name).argtypes = types
    L.rsvdt_hip_bgram_work_bytes.restype = ctypes.c_size_t
    L.rsvdt_hip_bshift_solve_work_bytes.restype = ctypes.c_size_t
    _ok(L.rsvdt_hip_init(0))
    return L


def _ok(rc):
    if rc:
        raise RuntimeError("code %d: %s" % (rc, _pkg().lib().rsvdt_hip_last_error().decode()))


def _stream():
    return torch.cuda.current_stream().cuda_stream


# --------------------------------------------------------------------------
# inputs
def _gen(seed):
    return torch.Generator(DEV).manual_seed(int(seed))


def _zrandn(gen, *shape):
    return torch.randn(*shape, dtype=torch.complex128, device=DEV, generator=gen)


def _stencil(case, gen):
    """A flow operator as the workloads have them: nf coupled fields per point
    of an nx x ny (x nz) grid, field index fastest.  2D: 9-point diffusion and
    advection, periodic; 3D: 7-point, periodic in x and z, walls in y; dense
    random coupling of the fields of a point.  Returns (cols, vals), N x w
    with the row's columns ascending and missing entries (column N, value 0)
    last."""
    nx, ny, nz, nf = case["nx"], case["ny"], case["nz"], case["nf"]
    three = nz > 1
    npt = nx * ny * nz
    pt = torch.arange(npt, device=DEV)
    ii, jj, kk = pt % nx, (pt // nx) % ny, pt // (nx * ny)
    h = 1.0 / 64 if three else 2.0 / nx
    y = (jj + 0.5) / ny
    u = 1.0 + (0.3 * torch.tanh(y.double() - 0.5) if three else 0.5 * torch.sin(2 * math.pi * y.double()))
    if three:
        offs = [(1, 0, 0, 1.0), (-1, 0, 0, 1.0), (0, 1, 0, 1.0), (0, -1, 0, 1.0), (0, 0, 1, 1.0), (0, 0, -1, 1.0)]
        nu, scale, centre = 5e-4, 1.0 / (h * h), -6.0
    else:
        offs = [(1, 0, 0, 4.0), (-1, 0, 0, 4.0), (0, 1, 0, 4.0), (0, -1, 0, 4.0),
                (1, 1, 0, 1.0), (1, -1, 0, 1.0), (-1, 1, 0, 1.0), (-1, -1, 0, 1.0)]
        nu, scale, centre = 1e-3, 1.0 / (6 * h * h), -20.0
    N = nf * npt
    f = torch.arange(nf, device=DEV)
    cols, vals = [], []
    for di, dj, dk, w in offs:
        j2 = jj + dj
        ok = (j2 >= 0) & (j2 < ny) if three else torch.ones_like(jj, dtype=torch.bool)
        nbr = (((kk + dk) % nz) * ny + j2 % ny) * nx + (ii + di) % nx
        v = torch.full((npt,), nu * w * scale, dtype=torch.float64, device=DEV)
        if di and not dj:
            v = v - u * di / (2 * h)
        v = torch.where(ok, v, torch.zeros_like(v))
        c = torch.where(ok[:, None], nf * nbr[:, None] + f, torch.full_like(f, N)[None])
        cols.append(c[:, :, None])
        vals.append(v[:, None, None].expand(npt, nf, 1))
    R = 0.1 * torch.randn(npt, nf, nf, dtype=torch.float64, device=DEV, generator=gen)
    R = R + torch.eye(nf, dtype=torch.float64, device=DEV) * (nu * centre * scale - 0.05)
    cols.append((nf * pt[:, None, None] + f).expand(npt, nf, nf))
    vals.append(R)
    cols, vals = torch.cat(cols, 2).reshape(N, -1), torch.cat(vals, 2).reshape(N, -1)
    cols, order = torch.sort(cols, dim=1)
    return cols, vals.gather(1, order)


def _csr(cols, vals):
    """int32 CSR arrays of the (cols, vals) form."""
    N = cols.shape[0]
    keep = cols < N
    rowptr = torch.zeros(N + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(keep.sum(1), 0, out=rowptr[1:])
    return rowptr.int(), cols[keep].int(), vals[keep]


def _tiles(rowptr, col, N, TR):
    """The tiled form of include/rsvdt_hip.h (tile_rows, tptr, tcol, lidx)."""
    counts = (rowptr[1:] - rowptr[:-1]).long()
    tile = torch.repeat_interleave(torch.arange(N, device=DEV), counts) // TR
    nt = (N + TR - 1) // TR
    uniq, inv = torch.unique(tile * N + col, return_inverse=True)
    per = torch.bincount(uniq // N, minlength=nt)
    tptr = torch.zeros(nt + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(per, 0, out=tptr[1:])
    lidx = (inv - tptr[tile]).to(torch.int16)
    ends = rowptr[torch.clamp(torch.arange(0, nt + 1, device=DEV) * TR, max=N)].long()
    return tptr.int(), (uniq % N).int(), lidx, int(per.max()), int((ends[1:] - ends[:-1]).max())


def _idft_table(nwe, nt2, real):
    """nt2 x nwe: exp(2 pi i m_alias j / nt2) 2/nt2."""
    m = torch.arange(nwe, dtype=torch.int64, device=DEV)
    if not real:
        m = torch.where(m > (nwe - 1) // 2, m - nwe + nt2, m)
    ph = (torch.arange(nt2, device=DEV)[:, None] * m) % nt2
    a = ph.double() * (2 * math.pi / nt2)
    return torch.complex(torch.cos(a), torch.sin(a)) * (2.0 / nt2)


def _dft_table(nw, nwe):
    """nw x nwe: exp(-2 pi i m s / nw)."""
    ph = (torch.arange(nw, device=DEV)[:, None] * torch.arange(nwe, device=DEV)) % nw
    a = ph.double() * (-2 * math.pi / nw)
    return torch.complex(torch.cos(a), torch.sin(a))


def _graded(gen, n, decades):
    """n singular values over the given decades, jittered, descending."""
    j = torch.arange(n, dtype=torch.float64, device=DEV)
    r = torch.rand(n, dtype=torch.float64, device=DEV, generator=gen)
    return 10.0 ** (-decades * (j + 0.3 * r) / n)


# --------------------------------------------------------------------------
# action: Session(...).set_sketch / direct / adjoint / get_Y
def _action_operator(case):
    W = _workloads()
    if case["op"] == "gl":
        return W.gl(case["N"], L=85.0 * case["N"] / 500 if case["N"] < 500 else 85.0)
    A0 = W._flow2d_unshifted(nx=2 * case["ny"], ny=case["ny"])
    return W.shifted(A0, -0.3, 0.0)[0].astype(np.complex128)


def _action_size(case):
    return case["N"] if case["op"] == "gl" else 6 * case["ny"] * case["ny"]


def _action_prepare(case, seed):
    w = case["w"]
    s = _pkg().Session(_action_operator(case), k=case["k"], q=0, Nw=case["Nw"], w=w, TL=case["TL"],
                       dt=2 * math.pi / w / case["steps"], transient_removal=case["removal"])
    g = np.random.default_rng(seed)
    shape = (s.N, s.k * s.Nw_eff)
    F = np.asfortranarray(g.standard_normal(shape) + 1j * g.standard_normal(shape))
    return {"case": case, "s": s, "F": F}


def _action_run(st):
    s = st["s"]
    s.set_sketch(st["F"])
    if st["case"]["direct"]:
        s.direct()
    else:
        s.adjoint()
    return s.get_Y()


def _action_grid(case):
    """(dt, Ns, Nt, RR) of the time grid."""
    T = 2 * math.pi / case["w"]
    dtw = T / case["Nw"]
    dt = dtw / math.ceil(dtw / (T / case["steps"]))
    Ns = int(round(T / dt))
    return dt, Ns, int(round(case["TL"] / dt)), Ns // case["Nw"]


def _action_exact(case, seed):
    """The forced RK4 recursion from rest, its snapshots, and the DFT or the
    Galerkin removal of the transient, with dense 64-bit products."""
    A = torch.from_numpy(np.asarray(_action_operator(case).todense())).to(DEV)
    N, k, Nw = A.shape[0], case["k"], case["Nw"]
    real = case["op"] != "gl"
    nwe = Nw // 2 if real else Nw
    g = np.random.default_rng(seed)
    F = g.standard_normal((N, k * nwe)) + 1j * g.standard_normal((N, k * nwe))
    F = torch.from_numpy(F).to(DEV).reshape(N, nwe, k)
    dt, Ns, Nt, RR = _action_grid(case)
    direct, sgn = case["direct"], 1 if case["direct"] else -1
    if not direct:
        A = A.conj().T.contiguous()
    idft = _idft_table(nwe, 2 * Ns, real)
    n = Nw + 1 if case["removal"] else Nw
    rend = Nt + Ns + (RR if case["removal"] else 0)
    Fm = F.permute(1, 0, 2).reshape(nwe, N * k)
    snaps = torch.zeros(n, N, k, dtype=torch.complex128, device=DEV)
    y = torch.zeros(N, k, dtype=torch.complex128, device=DEV)
    chunk = 256
    for i0 in range(0, rend, chunk):
        c = min(chunk, rend - i0)
        pos = (sgn * (2 * i0 + torch.arange(2 * c + 1, device=DEV))) % (2 * Ns)
        f = (idft[pos] @ Fm).reshape(2 * c + 1, N, k)
        for t in range(c):
            k1 = A @ y + f[2 * t]
            k2 = A @ (y + (dt / 2) * k1) + f[2 * t + 1]
            k3 = A @ (y + (dt / 2) * k2) + f[2 * t + 1]
            k4 = A @ (y + dt * k3) + f[2 * t + 2]
            y = y + (dt / 6) * (k1 + 2 * k2 + 2 * k3 + k4)
            i = i0 + t + 1
            if i > Nt and (i - Nt) % RR == 0:
                p = ((i - Nt) // RR - 1) % n
                snaps[p if direct else n - 1 - p] = y
    dft = _dft_table(Nw, nwe) * RR
    if not case["removal"]:
        Y = torch.einsum("snk,sm->nmk", snaps, dft)
        return Y.reshape(N, nwe * k).cpu().numpy()
    I = torch.eye(N, dtype=torch.complex128, device=DEV)
    hA = dt * A
    P = I + hA @ (I + hA @ (I + hA @ (I + hA / 4) / 3) / 2)
    out = torch.zeros(N, nwe, k, dtype=torch.complex128, device=DEV)
    ang = sgn * case["w"] * dt * RR * torch.arange(nwe, dtype=torch.float64, device=DEV)
    ph = torch.complex(torch.cos(ang), torch.sin(ang))
    w1, w2 = (0, 1) if direct else (1, 0)
    for ik in range(k):
        X = snaps[:, :, ik].T.contiguous()
        Q = torch.from_numpy(np.linalg.qr(X.cpu().numpy())[0]).to(DEV)
        MV = Q
        for _ in range(RR):
            MV = P @ MV
        M = Q.conj().T @ MV
        y1, y2 = X[:, w1:w1 + Nw] @ dft, X[:, w2:w2 + Nw] @ dft
        b = Q.conj().T @ (ph * y1 - y2)
        S = ph[:, None, None] * torch.eye(M.shape[0], dtype=torch.complex128, device=DEV) - M
        a = torch.from_numpy(np.linalg.solve(S.cpu().numpy(), b.T.cpu().numpy()[:, :, None])).to(DEV)
        out[:, :, ik] = y1 - Q @ a[:, :, 0].T
    return out.reshape(N, nwe * k).cpu().numpy()


def _action_work(case):
    N, k = _action_size(case), case["k"]
    nwe = case["Nw"] if case["op"] == "gl" else case["Nw"] // 2
    nnz = (3 if case["op"] == "gl" else 11) * N
    dt, Ns, Nt, RR = _action_grid(case)
    steps = Nt + Ns + (RR if case["removal"] else 0)
    per = 8 if case["op"] == "gl" else 4
    return {"bytes": 32.0 * N * k * nwe + 20.0 * nnz, "flops": float(steps) * 4 * per * nnz * k}


# --------------------------------------------------------------------------
# step: RK4 steps on nb blocks of N x k, four rsvdt_hip_horner_stage calls each
def _step_dt(case):
    return 0.012 if case["nz"] > 1 else 0.8 * 2.0 / case["nx"]


def _step_prepare(case, seed):
    _lib()
    gen = _gen(seed)
    N, k, nb = case["nx"] * case["ny"] * case["nz"] * case["nf"], case["k"], case["nb"]
    rowptr, col, val = _csr(*_stencil(case, gen))
    st = {"case": case, "keep": [rowptr, col, val]}
    d = SpmmDesc(nrows=N, k=k, nb=nb, rowptr=rowptr.data_ptr(), col=col.data_ptr(), val=val.data_ptr(), a_real=1,
                 prec=case["prec"], lanes=case["lanes"], xcd_remap=case["remap"], variant=case["variant"])
    if case["variant"] >= 9:
        tptr, tcol, lidx, hmax, emax = _tiles(rowptr, col, N, case["tile_rows"])
        st["keep"] += [tptr, tcol, lidx]
        d.tile_rows, d.tile_hmax, d.tile_emax = case["tile_rows"], hmax, emax
        d.tptr, d.tcol, d.lidx, d.tile_bpw = tptr.data_ptr(), tcol.data_ptr(), lidx.data_ptr(), case["bpw"]
    dtype = torch.complex128 if case["prec"] == 64 else torch.complex64
    y0 = torch.randn(nb, N, k, dtype=dtype, device=DEV, generator=gen)
    st.update(d=d, y0=y0, y=torch.empty_like(y0), u1=torch.empty_like(y0), u2=torch.empty_like(y0))
    if case["forced"]:
        st["g"] = 0.01 * torch.randn(case["steps"], nb, N, k, dtype=dtype, device=DEV, generator=gen)
        st["snap"] = torch.empty(nb, N, k, dtype=torch.complex128, device=DEV)
    return st


def _step_run(st):
    case, L, d, s = st["case"], _lib(), ctypes.byref(st["d"]), _stream()
    h = _step_dt(case)
    y, u1, u2 = st["y"].data_ptr(), st["u1"].data_ptr(), st["u2"].data_ptr()
    src = st["y0"].data_ptr()
    stage = L.rsvdt_hip_horner_stage
    for i in range(case["steps"]):
        g = st["g"][i].data_ptr() if case["forced"] else None
        snap = st["snap"].data_ptr() if case["forced"] and i == case["steps"] - 1 else None
        _ok(stage(d, src, src, None, None, h / 4, u1, None, s))
        _ok(stage(d, u1, src, None, None, h / 3, u2, None, s))
        _ok(stage(d, u2, src, None, None, h / 2, u1, None, s))
        _ok(stage(d, u1, src, None, g, h, y, snap, s))
        src = y
    return {"y": st["y"], "snap": st["snap"]} if case["forced"] else {"y": st["y"]}


def _step_exact(case, seed):
    gen = _gen(seed)
    cols, vals = _stencil(case, gen)
    N, k, nb = cols.shape[0], case["k"], case["nb"]
    cols = torch.where(cols < N, cols, torch.zeros_like(cols))
    dtype = torch.complex128 if case["prec"] == 64 else torch.complex64
    y = torch.randn(nb, N, k, dtype=dtype, device=DEV, generator=gen).to(torch.complex128)
    g = None
    if case["forced"]:
        g = 0.01 * torch.randn(case["steps"], nb, N, k, dtype=dtype, device=DEV, generator=gen)
    h = _step_dt(case)
    for b in range(nb):
        x = y[b].clone()
        for i in range(case["steps"]):
            v = x
            for c in (h / 4, h / 3, h / 2, h):
                t = torch.zeros_like(x)
                for e in range(cols.shape[1]):
                    t += vals[:, e, None] * v[cols[:, e]]
                v = x + c * t
            x = v if g is None else v + g[i, b]
        y[b] = x
    return {"y": y, "snap": y} if case["forced"] else {"y": y}


def _step_work(case):
    N = case["nx"] * case["ny"] * case["nz"] * case["nf"]
    nnz = N * ((6 if case["nz"] > 1 else 8) + case["nf"])
    s = 16 if case["prec"] == 64 else 8
    vec = float(N) * case["k"] * case["nb"] * s
    return {"bytes": case["steps"] * (4 * (12.0 * nnz + 4 * N) + (12 if case["forced"] else 11) * vec),
            "flops": case["steps"] * 16.0 * nnz * case["k"] * case["nb"]}


# --------------------------------------------------------------------------
# coef: rsvdt_hip_coef_gemm
def _coef_table(case):
    """(table, cq, cp, p0, sgn, cmod, alpha): the forcing reads the iDFT table
    at every second of its 2 Ns samples, the DFT its Nw x Nw_eff table."""
    if case["dft"]:
        return _dft_table(case["K"], case["P"]), case["P"], 1, 0, 1, case["P"], float(case["rr"])
    nt2 = 2 * case["rr"] * case["K"] * 2
    return _idft_table(case["K"], nt2, True), 1, case["K"], case["sgn"] * (nt2 // 3), 2 * case["sgn"], nt2, 1.0


def _coef_prepare(case, seed):
    _lib()
    st = {"case": case, "table": _coef_table(case), "x": _zrandn(_gen(seed), case["K"], case["L"])}
    st["out"] = torch.empty(case["P"], case["L"], dtype=torch.complex128 if case["prec"] == 64 else torch.complex64,
                            device=DEV)
    return st


def _coef_run(st):
    c = st["case"]
    t, cq, cp, p0, sgn, cmod, alpha = st["table"]
    _ok(_lib().rsvdt_hip_coef_gemm(c["P"], c["K"], c["L"], t.data_ptr(), cq, cp, p0, sgn, cmod, alpha,
                                   st["x"].data_ptr(), c["L"], st["out"].data_ptr(), c["L"], c["prec"], 0.0, _stream()))
    return st["out"]


def _coef_exact(case, seed):
    t, cq, cp, p0, sgn, cmod, alpha = _coef_table(case)
    col = (p0 + sgn * torch.arange(case["P"], device=DEV)) % cmod
    C = t[:, col].T if case["dft"] else t[col]
    return alpha * (C.contiguous() @ _zrandn(_gen(seed), case["K"], case["L"]))


def _coef_work(case):
    return {"bytes": case["L"] * (16.0 * case["K"] + (16 if case["prec"] == 64 else 8) * case["P"]),
            "flops": 8.0 * case["P"] * case["K"] * case["L"]}


# --------------------------------------------------------------------------
# qr: rsvdt_qr_blocks_noalloc on frequency blocks of graded responses
def _qr_input(case, seed):
    gen = _gen(seed)
    nb, N, k = case["nb"], case["N"], case["k"]
    mix = _zrandn(gen, nb, k, k) * _graded(gen, k, case["decades"])[:, None]
    return torch.stack([_zrandn(gen, N, k) @ mix[b] for b in range(nb)])


def _qr_prepare(case, seed):
    _lib()
    y0 = _qr_input(case, seed)
    return {"case": case, "y0": y0, "y": torch.empty_like(y0)}


def _qr_run(st):
    c = st["case"]
    st["y"].copy_(st["y0"])          # the QR is in place; the response is kept, as a program that stores it does
    _ok(_lib().rsvdt_qr_blocks_noalloc(st["y"].data_ptr(), c["N"], c["k"], c["nb"], _stream()))
    return st["y"]


def _qr_exact(case, seed):
    """Gram-Schmidt, each column orthogonalised twice."""
    y = _qr_input(case, seed)
    for b in range(case["nb"]):
        q = y[b].T.contiguous()
        for j in range(case["k"]):
            for _ in range(2):
                if j:
                    q[j] -= q[:j].T @ (q[:j].conj() @ q[j])
            q[j] /= torch.linalg.vector_norm(q[j])
        y[b] = q.T
    return y


def _qr_work(case):
    el = float(case["nb"]) * case["N"] * case["k"]
    return {"bytes": 32.0 * el, "flops": 16.0 * el * case["k"]}


# --------------------------------------------------------------------------
# svd: rsvdt_hip_bjacobi_svd of triangular factors
def _svd_input(case, seed):
    gen = _gen(seed)
    nb, n = case["nb"], case["n"]
    s = torch.stack([_graded(gen, n, case["decades"]) for _ in range(nb)]).cpu().numpy()
    a, b = _zrandn(gen, nb, n, n).cpu().numpy(), _zrandn(gen, nb, n, n).cpu().numpy()
    X = (np.linalg.qr(a)[0] * s[:, None, :]) @ np.linalg.qr(b)[0]
    return np.triu(np.linalg.qr(X)[1])


def _svd_prepare(case, seed):
    _lib()
    R = torch.from_numpy(_svd_input(case, seed)).to(DEV).contiguous()
    return {"case": case, "R": R, "U": torch.empty_like(R),
            "sig": torch.empty(case["nb"], case["n"], dtype=torch.float64, device=DEV)}


def _svd_run(st):
    c = st["case"]
    _ok(_lib().rsvdt_hip_bjacobi_svd(c["nb"], c["n"], st["R"].data_ptr(), st["U"].data_ptr(), st["sig"].data_ptr(),
                                     _stream()))
    return {"U": st["U"], "sig": st["sig"]}


def _svd_exact(case, seed):
    U, s, _ = np.linalg.svd(_svd_input(case, seed))
    t = U.sum(axis=1, keepdims=True)
    return {"U": U * (np.abs(t) / t), "sig": s}


def _svd_work(case):
    n = float(case["n"])
    return {"bytes": case["nb"] * (32.0 * n * n + 8 * n), "flops": case["nb"] * 8 * 12.0 * n ** 3}


# --------------------------------------------------------------------------
# project: the Galerkin projection of kb test vectors
def _project_input(case, seed):
    gen = _gen(seed)
    kb, N, nw, nwe, kt = case["kb"], case["N"], case["Nw"], case["Nwe"], case["kt"]
    n = nw + 1
    Y = _zrandn(gen, n, N, kt)
    Vb = _zrandn(gen, kb, N, n) / math.sqrt(2 * N)
    M = 0.5 * _zrandn(gen, kb, n, n) / math.sqrt(2 * n)
    dft = _dft_table(nw, nw)[:, :nwe] * 8.0
    z = torch.zeros(1, nwe, dtype=torch.complex128, device=DEV)
    a = torch.arange(nwe, dtype=torch.float64, device=DEV) * (2 * math.pi / nw)
    ph = torch.complex(torch.cos(a), torch.sin(a))
    C1 = torch.cat([dft, z])
    Ct = ph * C1 - torch.cat([z, dft])
    return Y, Vb, M, ph, C1, Ct


def _project_prepare(case, seed):
    L = _lib()
    kb, N, nwe, kt, n = case["kb"], case["N"], case["Nwe"], case["kt"], case["Nw"] + 1
    Y, Vb, M, ph, C1, Ct = _project_input(case, seed)
    z = functools.partial(torch.zeros, dtype=torch.complex128, device=DEV)
    rep = lambda x: x.expand(kb, *x.shape).contiguous()      # noqa: E731
    return {"case": case, "Y": Y, "V": Vb, "M": M, "ph": rep(ph), "C1": rep(C1), "Ct": rep(Ct),
            "X": z(kb, N, n), "W": z(kb, n, n), "B": z(kb, n, nwe), "Yb": z(kb, N, nwe), "out": z(nwe, N, kt),
            "work": torch.empty(L.rsvdt_hip_bgram_work_bytes(kb, N, n, n), dtype=torch.uint8, device=DEV),
            "lw": torch.empty(L.rsvdt_hip_bshift_solve_work_bytes(kb, n, nwe), dtype=torch.uint8, device=DEV),
            "info": torch.zeros(64, dtype=torch.int32, device=DEV)}


def _project_run(st):
    c, L, s = st["case"], _lib(), _stream()
    kb, N, nwe, kt, b0, n = c["kb"], c["N"], c["Nwe"], c["kt"], c["b0"], c["Nw"] + 1
    p = {k: v.data_ptr() for k, v in st.items() if k != "case"}
    xs = N * n
    _ok(L.rsvdt_hip_transpose_rows(N, n, kt, b0, kb, p["Y"], p["X"], 0, s))
    _ok(L.rsvdt_hip_bgram(kb, N, n, n, p["V"], xs, n, 1, p["X"], xs, n, 1, p["W"], p["work"], s))
    _ok(L.rsvdt_hip_bapply(kb, n, n, nwe, p["W"], n * n, n, 1, p["Ct"], 0.0, None, 0, 0, 0, p["B"], n * nwe, nwe, 1, s))
    _ok(L.rsvdt_hip_bshift_solve(kb, n, nwe, p["M"], p["ph"], p["B"], p["B"], p["lw"], p["info"], s))
    _ok(L.rsvdt_hip_zscale(kb * n * nwe, -1.0, p["B"], p["B"], s))
    _ok(L.rsvdt_hip_bapply(kb, N, n, nwe, p["X"], xs, n, 1, p["C1"], 0.0, None, 0, 0, 0, p["Yb"], N * nwe, nwe, 1, s))
    _ok(L.rsvdt_hip_bapply(kb, N, n, nwe, p["V"], xs, n, 1, p["B"], 1.0, p["Yb"], N * nwe, nwe, 1, p["Yb"], N * nwe,
                           nwe, 1, s))
    _ok(L.rsvdt_hip_transpose_rows(N, nwe, kt, b0, kb, p["Yb"], p["out"], 1, s))
    return {"Y": st["out"], "W": st["W"], "a": st["B"]}


def _project_exact(case, seed):
    Y, Vb, M, ph, C1, Ct = _project_input(case, seed)
    kb, N, nwe, kt, b0, n = case["kb"], case["N"], case["Nwe"], case["kt"], case["b0"], case["Nw"] + 1
    out = torch.zeros(nwe, N, kt, dtype=torch.complex128, device=DEV)
    Wa, a = [], []
    for b in range(kb):
        X = Y[:, :, b0 + b].T.contiguous()
        W = Vb[b].conj().T.contiguous() @ X
        rhs = (W @ Ct).T.cpu().numpy()[:, :, None]
        S = ph[:, None, None] * torch.eye(n, dtype=torch.complex128, device=DEV) - M[b]
        x = -torch.from_numpy(np.linalg.solve(S.cpu().numpy(), rhs)).to(DEV)[:, :, 0].T.contiguous()
        out[:, :, b0 + b] = (X @ C1 + Vb[b] @ x).T
        Wa.append(W)
        a.append(x)
    return {"Y": out, "W": torch.stack(Wa), "a": torch.stack(a)}


def _project_work(case):
    kb, N, nwe, n = case["kb"], float(case["N"]), case["Nwe"], case["Nw"] + 1
    return {"bytes": kb * N * 16.0 * (2 * n + nwe),
            "flops": kb * (8.0 * N * n * (n + 2 * nwe) + nwe * 8.0 * n ** 3 / 3)}


# --------------------------------------------------------------------------
# weights: rsvdt_hip_spmm_blocks
def _weights_input(case, seed):
    """A rows x cols matrix with 1 .. wmax entries in a row near the scaled
    diagonal (wmax = 1: a diagonal weight or a selection), as (cols, vals,
    counts)."""
    gen = _gen(seed)
    rows, ncol, wmax = case["rows"], case["cols"], case["wmax"]
    base = torch.arange(rows, device=DEV) * (ncol - wmax) // rows
    col = base[:, None] + torch.arange(wmax, device=DEV)
    val = _zrandn(gen, rows, wmax)
    cnt = torch.randint(1, wmax + 1, (rows,), device=DEV, generator=gen)
    x = _zrandn(gen, case["nb"], ncol, case["k"])
    return col, val, cnt, x


def _weights_prepare(case, seed):
    _lib()
    col, val, cnt, x = _weights_input(case, seed)
    keep = torch.arange(case["wmax"], device=DEV) < cnt[:, None]
    rp = torch.zeros(case["rows"] + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(cnt, 0, out=rp[1:])
    return {"case": case, "rp": rp.int(), "ci": col[keep].int(), "v": val[keep].contiguous(), "x": x,
            "out": torch.empty(case["nb"], case["rows"], case["k"], dtype=torch.complex128, device=DEV)}


def _weights_run(st):
    c = st["case"]
    _ok(_lib().rsvdt_hip_spmm_blocks(c["rows"], c["k"], c["nb"], st["rp"].data_ptr(), st["ci"].data_ptr(),
                                     st["v"].data_ptr(), st["x"].data_ptr(), c["cols"] * c["k"], st["out"].data_ptr(),
                                     c["rows"] * c["k"], _stream()))
    return st["out"]


def _weights_exact(case, seed):
    col, val, cnt, x = _weights_input(case, seed)
    out = torch.zeros(case["nb"], case["rows"], case["k"], dtype=torch.complex128, device=DEV)
    for e in range(case["wmax"]):
        v = torch.where(cnt > e, val[:, e], torch.zeros_like(val[:, e]))
        for b in range(case["nb"]):
            out[b] += v[:, None] * x[b][col[:, e]]
    return out


def _weights_work(case):
    nnz = case["rows"] * (case["wmax"] + 1) / 2
    return {"bytes": 20.0 * nnz + 4 * case["rows"] + 16.0 * case["nb"] * case["k"] * (case["rows"] + case["cols"]),
            "flops": 8.0 * nnz * case["nb"] * case["k"]}


# --------------------------------------------------------------------------
# layer: rsvdt_hip_gemm_bf16 with its epilogues, rsvdt_hip_colsum
def _layer_input(case, seed):
    gen = _gen(seed)
    M, N, K = case["M"], case["N"], case["K"]
    f = functools.partial(torch.randn, device=DEV, generator=gen)
    return f(M, K), f(N, K) / math.sqrt(K), 0.1 * f(N), f(M, N) / math.sqrt(M), f(M, K)


def _layer_prepare(case, seed):
    _lib()
    M, N, K = case["M"], case["N"], case["K"]
    a, w, b, dz, zin = _layer_input(case, seed)
    e = functools.partial(torch.empty, device=DEV)
    return {"case": case, "a": a, "w": w, "b": b, "dz": dz, "zin": zin, "c": e(M, N), "z": e(M, N), "dw": e(N, K),
            "db": e(N), "da": e(M, K)}


def _layer_run(st):
    c, L, s = st["case"], _lib(), _stream()
    M, N, K = c["M"], c["N"], c["K"]
    p = {k: v.data_ptr() for k, v in st.items() if k != "case"}
    _ok(L.rsvdt_hip_gemm_bf16(M, N, K, p["a"], K, 1, p["w"], 1, K, p["c"], N, 1, p["b"], p["z"], N, s))
    _ok(L.rsvdt_hip_gemm_bf16(N, K, M, p["dz"], 1, N, p["a"], K, 1, p["dw"], K, 0, None, None, 0, s))
    _ok(L.rsvdt_hip_colsum(M, N, p["dz"], N, p["db"], s))
    _ok(L.rsvdt_hip_gemm_bf16(M, K, N, p["dz"], N, 1, p["w"], K, 1, p["da"], K, 3, None, p["zin"], K, s))
    return {k: st[k] for k in ("c", "z", "dw", "db", "da")}


def _layer_exact(case, seed):
    a, w, b, dz, zin = (x.double() for x in _layer_input(case, seed))
    z = a @ w.T + b
    sg = torch.sigmoid(zin)
    return {"c": z * torch.sigmoid(z), "z": z, "dw": dz.T @ a, "db": dz.sum(0),
            "da": (dz @ w) * sg * (1 + zin * (1 - sg))}


def _layer_work(case):
    M, N, K = float(case["M"]), case["N"], case["K"]
    return {"bytes": 4 * (3 * M * K + 3 * M * N + 2 * N * K + 2 * N), "flops": 6.0 * M * N * K}


# --------------------------------------------------------------------------
KINDS = {"action": (_action_prepare, _action_run, _action_exact, _action_work),
         "step": (_step_prepare, _step_run, _step_exact, _step_work),
         "coef": (_coef_prepare, _coef_run, _coef_exact, _coef_work),
         "qr": (_qr_prepare, _qr_run, _qr_exact, _qr_work),
         "svd": (_svd_prepare, _svd_run, _svd_exact, _svd_work),
         "project": (_project_prepare, _project_run, _project_exact, _project_work),
         "weights": (_weights_prepare, _weights_run, _weights_exact, _weights_work),
         "layer": (_layer_prepare, _layer_run, _layer_exact, _layer_work)}


def _step(nx, ny, nz, nf, k, nb, prec, steps, forced):
    """A step case with the launch shape that the engine takes for it: the
    tiled form on 3D grids and for several blocks, two columns per lane on
    2D grids, column pairs in FP32 where k allows."""
    c = {"kind": "step", "nx": nx, "ny": ny, "nz": nz, "nf": nf, "k": k, "nb": nb, "prec": prec, "steps": steps,
         "forced": forced, "tile_rows": 0, "bpw": 0, "remap": 0}
    half = 4
    while 2 * half < k:
        half *= 2
    if nb > 1:
        c.update(variant=9, lanes=8, tile_rows=32, bpw=8)
    elif prec == 32 and k in (16, 32, 64):
        c.update(variant=8, lanes=k // 4, remap=1 if nz == 1 else 3)
    elif prec == 64 and nz > 1:
        c.update(variant=10, lanes=8, tile_rows=32, bpw=1, remap=3)
    else:
        c.update(variant=3, lanes=half)
    return c


def listed():
    return [
        # the smallest run anyone makes: a first check of an installation
        {"name": "gl_action_n64", "kind": "action", "op": "gl", "N": 64, "k": 2, "Nw": 8, "w": 0.3, "TL": 1.0,
         "steps": 1048, "removal": True, "direct": True},
        # the Ginzburg-Landau case users start from
        {"name": "gl_action_n500", "kind": "action", "op": "gl", "N": 500, "k": 10, "Nw": 64, "w": 0.05, "TL": 10.0,
         "steps": 4096, "removal": True, "direct": True},
        # the inner loop on the 2D flow workload, double and single precision state
        dict(_step(512, 256, 1, 3, 16, 1, 64, 4, True), name="step_flow2d"),
        dict(_step(512, 256, 1, 3, 16, 1, 32, 4, True), name="step_flow2d_fp32"),
        # the inner loop on the 3D flow workload
        dict(_step(128, 64, 48, 5, 32, 1, 64, 2, True), name="step_flow3d"),
        # e^{A dT} on the 65 basis blocks of 8 test vectors, a reduced 3D grid
        dict(_step(64, 32, 24, 5, 8, 65, 64, 2, False), name="removal_steps_flow3d"),
        # 64 forcing samples from the 64 frequency blocks of the 2D flow workload
        {"name": "forcing_chunk_flow2d", "kind": "coef", "P": 64, "K": 64, "L": 393216 * 16, "rr": 16, "sgn": 1,
         "prec": 64, "dft": False},
        # QR of frequency blocks between the actions of a power iteration
        {"name": "qr_freqs", "kind": "qr", "N": 393216, "k": 16, "nb": 16, "decades": 3.0},
        # the k x k SVDs of the 3D workload's 32 frequencies
        {"name": "svd_freqs", "kind": "svd", "nb": 32, "n": 32, "decades": 4.0},
        # the projection of 8 of 16 test vectors, 65 snapshots each
        {"name": "removal_projection", "kind": "project", "N": 98304, "kb": 8, "kt": 16, "b0": 8, "Nw": 64, "Nwe": 32},
        # an output matrix with a few entries in a row
        {"name": "output_weights", "kind": "weights", "rows": 393216, "cols": 393216, "wmax": 5, "k": 16, "nb": 8},
        # a hidden layer of the learned-sketch network, 32 frequencies x 500 points
        {"name": "sketch_layer", "kind": "layer", "M": 16000, "N": 256, "K": 256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["action", "action", "step", "step", "step", "coef", "qr", "svd", "project", "weights", "layer"])
    if kind == "action":
        if rng.random() < 0.75:
            N = _log(rng, 40, 700)
            c = {"op": "gl", "N": N, "k": rng.randint(1, 16), "Nw": rng.choice([8, 15, 16, 32, 33, 64]),
                 "w": rng.choice([0.05, 0.1, 0.3]), "TL": round(rng.uniform(1.0, 12.0), 2),
                 "removal": rng.random() < 0.6}
            c["Nw"] = min(c["Nw"], max(8, N // 4)) if c["removal"] else c["Nw"]
            c["steps"] = int(2 * math.pi / c["w"] / rng.uniform(0.025, 0.035))
        else:
            ny = rng.randint(4, 9)
            c = {"op": "flow2d", "N": 0, "ny": ny, "k": rng.randint(1, 16), "Nw": rng.choice([8, 16, 32]), "w": 0.5,
                 "TL": round(rng.uniform(2.0, 20.0), 2), "removal": False, "steps": rng.randint(200, 900)}
        return dict(c, kind="action", direct=rng.random() < 0.5)
    if kind == "step":
        k = rng.choice([4, 7, 8, 10, 13, 16, 16, 24, 32, 32, 48])
        if rng.random() < 0.3:
            nb, k, prec, forced = rng.choice([9, 17, 33, 65]), rng.choice([4, 6, 8, 8, 16]), 64, False
        else:
            nb, prec, forced = 1, rng.choice([64, 64, 32]), True
        points = _log(rng, 2000, 240000)
        points = max(64, min(points, 12_000_000 // (k * nb)))
        if rng.random() < 0.5:
            ny = max(4, int(math.sqrt(points / 2) * rng.uniform(0.7, 1.4)))
            dims = (max(4, points // ny), ny, 1, rng.choice([1, 3, 4]))
        else:
            ny = max(4, int(points ** (1 / 3) * rng.uniform(0.7, 1.4)))
            nz = max(3, int(points ** (1 / 3) * rng.uniform(0.6, 1.0)))
            dims = (max(4, points // (ny * nz)), ny, nz, rng.choice([2, 5, 5]))
        return _step(*dims, k, nb, prec, rng.randint(1, 3), forced)
    if kind == "coef":
        dft = rng.random() < 0.4
        K = rng.choice([16, 32, 33, 64, 100, 128]) if dft else rng.choice([4, 8, 15, 16, 32, 64])
        P = max(1, K // rng.choice([1, 2])) if dft else rng.choice([16, 31, 37, 64, 64, 128, 256])
        return {"kind": "coef", "P": P, "K": K, "L": max(500, min(_log(rng, 500, 4_000_000), 10 ** 10 // (P * K))),
                "rr": rng.randint(8, 64), "sgn": rng.choice([1, -1]), "prec": 64 if dft else rng.choice([64, 64, 32]),
                "dft": dft}
    if kind == "qr":
        k, nb = rng.randint(2, 48), rng.randint(1, 64)
        return {"kind": "qr", "N": max(500, min(_log(rng, 500, 400_000), 60_000_000 // (k * nb))), "k": k, "nb": nb,
                "decades": round(rng.uniform(0.5, 4.0), 2)}
    if kind == "svd":
        return {"kind": "svd", "nb": rng.randint(1, 128), "n": rng.randint(2, 64),
                "decades": round(rng.uniform(2.0, 6.0), 2)}
    if kind == "project":
        Nw, kb = rng.choice([8, 15, 16, 32, 64, 64]), rng.randint(1, 8)
        kt = kb + rng.randint(0, 8)
        return {"kind": "project", "N": min(_log(rng, 500, 100_000), 40_000_000 // (kt * Nw)), "kb": kb, "kt": kt,
                "b0": rng.randint(0, kt - kb), "Nw": Nw, "Nwe": max(1, Nw // rng.choice([1, 2]))}
    if kind == "weights":
        rows, k = _log(rng, 500, 500_000), rng.randint(1, 40)
        return {"kind": "weights", "rows": rows, "cols": max(16, int(rows * rng.choice([1.0, 1.0, 0.3, 2.5]))),
                "wmax": rng.choice([1, 1, 3, 5, 11]), "k": k, "nb": max(1, min(rng.randint(1, 64), 60_000_000 // (rows * k)))}
    return {"kind": "layer", "M": _log(rng, 500, 40_000), "N": rng.choice([16, 64, 128, 200, 256]),
            "K": rng.choice([64, 96, 128, 256])}


def prepare(case, seed):
    return KINDS[case["kind"]][0](case, seed)


def run(state):
    return KINDS[state["case"]["kind"]][1](state)


def exact(case, seed):
    return KINDS[case["kind"]][2](case, seed)


def work(case):
    return KINDS[case["kind"]][3](case)
