"""The work a user of this framework has it do, as measurable cases.

Every case is one pass through the public entry points of movfem_amd on
synthetic models of the repository's own families (movfem_amd.model,
movfem_amd.learned).  Kinds:

  solve     one frequency step of the program: re-integration and assembly of K
            and M (GpuVfem.assemble), right-hand side, factorization and GMRES
            (solve_frequencies, direct preconditioner, every listed frequency
            factored), then the readout of each frequency: nodal E and H and the
            receivers' E, H, Z, rho_a and phase.  Elements whose nodes are all
            air carry no mass, so the system leaves E arbitrary there (any
            gradient solves it), and with 20-node elements its curl too: the
            nodal E, and at 20 nodes the nodal H, are read out by the call but
            are no answer to compare, and are not returned.
  boundary  the reference's own call sequence through host arrays: assemble,
            set_frequency, global_vfem (coordinate form and right-hand side into
            host arrays that are kept from pass to pass, as the reference
            allocates them once) and the zmumps-shaped solve.
  krylov    assembly, Jacobi-preconditioned COCG over all frequencies in one
            batch (no factorization), readout.
  batch     several models through solve_batch (host threads, one stream each).
  train     one optimizer step of the learned-guess network: forward, backward,
            gradients to the host, Adam, updated parameters.
  predict   the network's forward pass.

The models' sizes follow the workloads of bench.py, tests/ and the example input
(a 20^3 Dirichlet half-space, 32..48 cells a side at 20 nodes, 58 x 58 x 43 at 8
nodes, 64 x 64 x 48 voxels for the network) and odd sizes between; receivers lie
on a 5 x 5 grid as in tests/test_gpu_configs.py.
"""
import math

import numpy as np
import torch

from movfem_amd import _lib as L
from movfem_amd import learned
from movfem_amd import model as M
from movfem_amd.vfem import GpuVfem, solve_batch


def listed():
    return [
        # the smallest call: a test-sized model through the reference's host-array sequence
        {"name": "boundary8_small", "kind": "boundary", "nodes": 8, "nx": 12, "ny": 11, "nz": 10, "air": 1,
         "dirichlet": True, "tensor": False, "freq": 1.0, "nf": 1, "model": 1},
        # the 8-node 20 x 20 x (16 + 4) Dirichlet workload: launches and latency dominate
        {"name": "solve8_20", "kind": "solve", "nodes": 8, "nx": 20, "ny": 20, "nz": 20, "air": 4,
         "dirichlet": True, "tensor": False, "freq": 1.0, "nf": 1, "model": 2},
        # the lattice of the example input (58 x 58 x 43 cells), 8-node Dirichlet, 0.1 Hz
        {"name": "solve8_58", "kind": "solve", "nodes": 8, "nx": 58, "ny": 58, "nz": 43, "air": 8,
         "dirichlet": True, "tensor": False, "freq": 0.1, "nf": 1, "model": 3},
        # odd sides, GPML, full tensor: the boundary type of the flagship workload on a small grid
        {"name": "solve20_odd_gpml", "kind": "solve", "nodes": 20, "nx": 21, "ny": 19, "nz": 17, "air": 4,
         "dirichlet": False, "tensor": True, "freq": 0.72, "nf": 1, "model": 4},
        # a member of the many-model workload (20-node, 33 x 33 x 25), two of its frequencies
        {"name": "solve20_33_nf2", "kind": "solve", "nodes": 20, "nx": 33, "ny": 33, "nz": 25, "air": 4,
         "dirichlet": True, "tensor": True, "freq": 2.15, "nf": 2, "model": 5},
        # quadratic Lagrange elements under a tensor earth
        {"name": "solve27_16", "kind": "solve", "nodes": 27, "nx": 16, "ny": 16, "nz": 12, "air": 2,
         "dirichlet": True, "tensor": True, "freq": 3.0, "nf": 1, "model": 6},
        # the flagship 20-node GPML workload at three quarters of its side: 1.0M unknowns
        {"name": "solve20_48_gpml", "kind": "solve", "nodes": 20, "nx": 48, "ny": 48, "nz": 36, "air": 6,
         "dirichlet": False, "tensor": False, "freq": 3.73, "nf": 1, "model": 7},
        # 8-node 64 x 64 x 48, two frequencies of plain COCG in one batch
        {"name": "krylov8_64", "kind": "krylov", "nodes": 8, "nx": 64, "ny": 64, "nz": 48, "air": 8,
         "dirichlet": True, "tensor": False, "freq": 50.0, "nf": 2, "model": 8},
        # the same on a small odd grid, where the iteration's launches count
        {"name": "krylov8_23", "kind": "krylov", "nodes": 8, "nx": 23, "ny": 22, "nz": 19, "air": 3,
         "dirichlet": True, "tensor": True, "freq": 50.0, "nf": 1, "model": 9},
        # many small models in flight, both element types (the reduced many-model workload)
        {"name": "batch_6", "kind": "batch", "nodes": 8, "nx": 16, "ny": 16, "nz": 12, "air": 4,
         "dirichlet": True, "tensor": True, "freq": 1.0, "nf": 2, "count": 6, "model": 10},
        # the learned-guess network: a training step and an inference at its own grid
        {"name": "train_64", "kind": "train", "nx": 64, "ny": 64, "nz": 48, "batch": 2},
        {"name": "predict_64", "kind": "predict", "nx": 64, "ny": 64, "nz": 48, "batch": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges, never dearer than the dearest of them."""
    kind = rng.choice(["solve", "solve", "solve", "solve", "boundary", "krylov", "batch", "train", "predict"])
    if kind in ("train", "predict"):
        nx, ny, nz = (8 * rng.randint(2, 8) for _ in range(3))
        return {"kind": kind, "nx": nx, "ny": ny, "nz": min(nz, 48), "batch": rng.randint(1, 2)}
    nodes = 8 if kind == "krylov" else rng.choice([8, 20, 20, 27] if kind == "solve" else [8, 20])
    top = {"solve": {8: 58, 20: 42, 27: 18}, "boundary": {8: 40, 20: 22}, "krylov": {8: 56},
           "batch": {8: 20, 20: 16}}[kind][nodes]
    nx = _log(rng, 9, top)
    ny = max(9, min(top, nx + rng.randint(-3, 3)))
    nz = max(9, min(int(0.8 * top), nx + rng.randint(-8, 2)))
    air = 1 if kind == "boundary" else rng.randint(1, 2 if nz < 14 else 6)
    gpml = kind == "solve" and rng.random() < 0.4
    out = {"kind": kind, "nodes": nodes, "nx": nx, "ny": ny, "nz": nz, "air": air, "dirichlet": not gpml,
           "tensor": rng.random() < 0.5,
           "freq": round(math.exp(rng.uniform(math.log(30.0 if kind == "krylov" else 0.1), math.log(100.0))), 3),
           "nf": rng.randint(1, 2) if kind != "boundary" else 1, "model": rng.randint(100, 10 ** 6)}
    if kind == "batch":
        out["count"] = rng.randint(2, 6)
    return out


# ------------------------------------------------------------------ models --
def _freqs(case):
    return [case["freq"] * 4.0 ** k for k in range(case["nf"])]


def _earth(case, seed):
    """Anisotropic blocks (bench.py, the many-model workload) of the case's size."""
    m = M.anisotropic_blocks(nx=case["nx"], ny=case["ny"], nz_earth=case["nz"] - case["air"], nz_air=case["air"],
                             h=500.0, nodes=case["nodes"], freqs=tuple(_freqs(case)), block=4,
                             seed=1000003 * case["model"] + seed, full_tensor=case["tensor"],
                             dirichlet=case["dirichlet"], nextd=2 if case["dirichlet"] else 4)
    return m


def _receivers(m):
    cx, cy = 0.5 * (m.xp[0] + m.xp[-1]), 0.5 * (m.yp[0] + m.yp[-1])
    off = np.arange(-2, 3) * 100.0
    xx, yy = np.meshgrid(cx + off, cy + off, indexing="ij")
    return xx.ravel(), yy.ravel()


def _handle(m):
    # update_sigma over the whole array, as bench.py: with the reference's index range no
    # solver reaches 1e-8 after the first frequency
    return GpuVfem(m, emulate=L.MVF_EMU_GPML_PREV_FLAGS)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "predict"):
        rng = np.random.default_rng(seed)
        shape = (case["batch"], case["nx"], case["ny"], case["nz"])
        net = learned.Net(case["nx"], case["ny"], case["nz"], batch=case["batch"], seed=4)
        # features as learned.features makes them: normalised log sigma, air mask, log f
        x = np.empty(shape + (learned.CIN,), np.float32)
        x[..., 0] = rng.uniform(-1.0, 1.0, shape)
        x[..., 1] = np.arange(case["nz"]) >= case["nz"] * 5 // 6
        x[..., 2] = rng.uniform(-1.2, 0.8)
        st = {"kind": kind, "net": net, "x": x}
        if kind == "train":
            st["t"] = rng.standard_normal(shape + (learned.COUT,), dtype=np.float32)
            st["mask"] = (rng.random(shape + (learned.COUT,), dtype=np.float32) < 0.9).astype(np.float32)
        return st
    if kind == "batch":
        ms = []
        for q in range(case["count"]):
            c = dict(case, nodes=8 if q % 2 == 0 else 20, nx=case["nx"] + q % 3, ny=case["ny"] + q % 2,
                     model=case["model"] + 17 * q)
            ms.append(_earth(c, seed))
        return {"kind": kind, "gs": [_handle(m) for m in ms], "freqs": _freqs(case), "air": case["air"],
                "rx": [_receivers(m) for m in ms]}
    m = _earth(case, seed)
    g = _handle(m)
    st = {"kind": kind, "g": g, "freqs": _freqs(case), "ke_top": case["nz"] - case["air"], "rx": _receivers(m)}
    if kind == "boundary":
        st["coo"] = (np.zeros(g.nnze, np.int32), np.zeros(g.nnze, np.int32), np.zeros(g.nnze, np.complex128),
                     np.zeros(2 * g.nne, np.complex128))
    return st


DIRECT = {"method": "gmres", "precond": "direct", "tol": 1e-8}


def _readout(g, freqs, ke_top, rx, nodal):
    out = []
    for f in range(len(freqs)):
        fields = g.readout(None, f=f, ke_top=ke_top, rx=rx[0], ry=rx[1])
        out.append(fields[1 if nodal else 2:])
    return out


def run(state):
    kind = state["kind"]
    if kind == "train":
        net = state["net"]
        loss = net.forward_backward(state["x"], state["t"], state["mask"])
        grads = net.grads()
        net.adam(1e-4)
        return {"loss": loss, "grads": grads, "params": net.params()}
    if kind == "predict":
        return state["net"].predict(state["x"])
    if kind == "batch":
        gs = state["gs"]
        for g in gs:
            g.assemble()
        solve_batch(gs, state["freqs"], **DIRECT)
        return [_readout(g, state["freqs"], g.m.nz - state["air"], rx, False) for g, rx in zip(gs, state["rx"])]
    g = state["g"]
    g.assemble()
    if kind == "boundary":
        g.set_frequency_hz(state["freqs"][0])
        ia, ja, a, b = g.global_vfem(out=state["coo"])
        x, _ = g.solve(b, **DIRECT)
        return {"ia": ia, "ja": ja, "a": a, "b": b, "x": x}
    if kind == "krylov":
        g.solve_frequencies(state["freqs"], method="cocg", tol=1e-8, maxit=20000, check_every=25, use_graph=True)
    else:
        g.solve_frequencies(state["freqs"], **DIRECT)
    return _readout(g, state["freqs"], state["ke_top"], state["rx"], g.m.nodes_per_elem != 20)


# ---------------------------------------------------------------- the work --
def _unknowns(case):
    """Edge unknowns and pattern entries of a large grid, per element type."""
    ne = case["nx"] * case["ny"] * case["nz"]
    return {8: 3, 20: 12, 27: 24}[case["nodes"]] * ne, {8: 99, 20: 1013, 27: 2500}[case["nodes"]] * ne


def _conv_macs(case):
    """Multiply-adds per forward pass of the U-Net (16/32/64/96 channels)."""
    ch, v, macs = [16, 32, 64, 96], case["nx"] * case["ny"] * case["nz"] * case["batch"], 0
    for k in range(4):
        cin = 3 if k == 0 else ch[k - 1]
        macs += 27 * (cin * ch[k] + ch[k] * ch[k]) * v / 8 ** k
        if k < 3:
            macs += 27 * ((ch[k] + ch[k + 1]) * ch[k] + ch[k] * ch[k]) * v / 8 ** k
    return macs + 16 * 12 * v


def work(case):
    kind = case["kind"]
    if kind in ("train", "predict"):
        v = case["nx"] * case["ny"] * case["nz"] * case["batch"]
        macs = _conv_macs(case)
        if kind == "predict":
            return {"bytes": 4.0 * v * (3 + 12) + 4.0 * 1162128, "flops": 2.0 * macs}
        return {"bytes": 4.0 * v * (3 + 12 + 12) + 4.0 * 5 * 1162128, "flops": 6.0 * macs}
    if kind == "batch":
        parts = [work(dict(case, kind="solve", nodes=8 if q % 2 == 0 else 20, nx=case["nx"] + q % 3,
                           ny=case["ny"] + q % 2)) for q in range(case["count"])]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n, nnz = _unknowns(case)
    ne, o = case["nx"] * case["ny"] * case["nz"], 1 if case["nodes"] == 8 else 2
    npt = (case["nx"] * o + 1) * (case["ny"] * o + 1) * (case["nz"] * o + 1)
    elem = {8: 21768, 20: 376731, 27: 744795}[case["nodes"]] * ne
    # lattice, tensors in; nodal E and H of two polarizations out, per frequency
    nbytes = npt * (8 + 96 + 48) + case["nf"] * npt * 192.0
    if kind == "krylov":
        # one application of the operator per iteration, K, M and the pattern read once each;
        # about 250 iterations (Jacobi COCG, tens of hertz)
        its = 250
        return {"bytes": nbytes + its * (20.0 * nnz + 64.0 * n * case["nf"]),
                "flops": elem + its * 16.0 * nnz * case["nf"]}
    if kind == "boundary":
        nbytes = npt * (8 + 96 + 48) + 24.0 * nnz + 64.0 * n
    # complex symmetric nested-dissection factorization of a 3-D grid, 8 real operations per
    # complex multiply-add; two triangular sweeps are lower order
    return {"bytes": nbytes, "flops": elem + case["nf"] * 34.0 * n * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("train", "predict"):
        # bf16 between the layers: 1e-2 against exact(), less between two orders of summation
        return {"rel": 1e-2, "max": 0.5}
    if kind == "krylov":
        # against a tighter solve: 1e-4 (COCG stops anywhere below a residual of 1e-8)
        return {"rel": 5e-4, "max": 2e-2}
    if kind in ("solve", "batch") and (kind == "batch" or case["nodes"] == 20):
        # a residual of 1e-8 against one of 1e-11: up to 2e-3 at the receivers of 20-node models
        return {"rel": 8e-3, "max": 1e-1}
    # against a residual of 1e-11, and against exact(): below 3e-6
    return {"rel": 1e-5, "max": 1e-3}


# ------------------------------------------------------- the same in 64 bits --
# 8-node elements restated on whole grids in numpy: node reference coordinates and the
# (basis node, direction) of the 12 edges
_R8 = [(1, -1, -1), (1, 1, -1), (-1, 1, -1), (-1, -1, -1), (1, -1, 1), (1, 1, 1), (-1, 1, 1), (-1, -1, 1)]
_E12 = [(3, 2), (3, 1), (7, 1), (2, 2), (3, 0), (7, 0), (2, 0), (6, 0), (0, 2), (0, 1), (4, 1), (1, 2)]
_T6 = [[0, 1, 2], [1, 3, 4], [2, 4, 5]]


def _assemble8(m, f):
    """(ia, ja, K, M, b) of an 8-node Dirichlet model: full symmetric pattern row by row,
    unknowns numbered by first visit in element order (z fastest)."""
    nx, ny, nz = m.nx, m.ny, m.nz
    ne = nx * ny * nz
    ijk = np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"), -1).reshape(ne, 3)
    off = (np.array(_R8) + 1) // 2
    ids = [((ijk[:, 0] + o[0]) * m.nny + ijk[:, 1] + o[1]) * m.nnz + ijk[:, 2] + o[2] for o in off]
    xyz = [np.stack([m.xp[ijk[:, 0] + o[0]], m.yp[ijk[:, 1] + o[1]], m.zp[i]], -1) for o, i in zip(off, ids)]
    # edges by lattice position: key = direction, lower end
    key = np.empty((ne, 12), np.int64)
    keep = np.empty((ne, 12), bool)
    dims = np.array([nx, ny, nz])
    for e, (nd, d) in enumerate(_E12):
        p = ijk + off[nd]
        p[:, d] = ijk[:, d]
        key[:, e] = ((d * (nx + 1) + p[:, 0]) * (ny + 1) + p[:, 1]) * (nz + 1) + p[:, 2]
        keep[:, e] = np.all([(p[:, c] > 0) & (p[:, c] < dims[c]) for c in range(3) if c != d], axis=0)
    flat, kf = key.ravel(), keep.ravel()
    uniq, first, inv = np.unique(flat[kf], return_index=True, return_inverse=True)
    rank = np.empty(len(uniq), np.int64)
    rank[np.argsort(first)] = np.arange(len(uniq))
    dof = np.full(ne * 12, -1, np.int64)
    dof[kf] = rank[inv]
    dof = dof.reshape(ne, 12)
    n = len(uniq)
    # integration, two points per axis; omega and the source constants in float32 as in the program
    om = 2.0 * M.PI * f
    w32 = float(np.float32(om))
    sig = m.sigma.copy()
    for c in (0, 3, 5):
        sig[:, c] = sig[:, c].real + 1j * float(np.float32(M.EPS0 * om))
    dsig = sig.copy()
    for c in (0, 3, 5):
        dsig[:, c] -= 1j * float(np.float32(om * M.EPS0))
    mu = m.mu
    assert np.all(mu[:, [1, 2, 4]] == 0.0) and np.all(mu[:, 0] == mu[0, 0])  # free-space permeability
    imu = 1.0 / mu[0, 0]
    zz = (om * 1.0e-9 * m.zp).astype(np.float32).astype(np.float64)
    K, Mm = np.zeros((ne, 12, 12)), np.zeros((ne, 12, 12))
    b = np.zeros((ne, 12, 2), complex)
    q = float(np.float32(0.5773502691896257645))
    for pt in [(a, bb, c) for a in (-q, q) for bb in (-q, q) for c in (-q, q)]:
        s = [[1 + r[c] * pt[c] for c in range(3)] for r in _R8]
        N = [v[0] * v[1] * v[2] / 8 for v in s]
        # the program's own d/dzeta of the nodal functions, (1 + r0) for (1 + r0 xi)
        dN = [(r[0] * v[1] * v[2] / 8, r[1] * v[0] * v[2] / 8, (1 + r[0]) * v[1] * r[2] / 8) for r, v in zip(_R8, s)]
        J = np.zeros((ne, 3, 3))
        for a in range(3):
            J[:, a, :] = sum(dN[i][a] * xyz[i] for i in range(8))
        det = np.linalg.det(J)
        Ji = np.linalg.inv(J) * np.sign(det)[:, None, None]
        S = sum(N[i] * sig[ids[i]].real for i in range(8))[:, np.array(_T6)]
        curl, val = np.empty((ne, 12, 3)), np.empty((ne, 12, 3))
        for e, (nd, d) in enumerate(_E12):
            r = _R8[nd]
            o = [c for c in range(3) if c != d]
            g = np.zeros(3)
            g[o[0]] = r[o[0]] * s[nd][o[1]] / 4
            g[o[1]] = r[o[1]] * s[nd][o[0]] / 4
            curl[:, e] = np.cross(Ji @ g, Ji[:, :, d])
            val[:, e] = s[nd][o[0]] * s[nd][o[1]] / 4 * Ji[:, :, d]
        K += (det * imu)[:, None, None] * (curl @ curl.transpose(0, 2, 1))
        Mm += det[:, None, None] * (val @ S @ val.transpose(0, 2, 1))
        for p, sg in ((0, -1.0), (1, 1.0)):
            src = sum(N[i] * dsig[ids[i]][:, [_T6[c][p] for c in range(3)]] * (1j * sg * zz[ids[i]])[:, None]
                      for i in range(8)) * (-1j * w32)
            b[:, :, p] += det[:, None] * np.einsum("eac,ec->ea", val, src)
    rows, cols = np.repeat(dof, 12, axis=1).ravel(), np.tile(dof, (1, 12)).ravel()
    ok = (rows >= 0) & (cols >= 0)
    pair, at = np.unique(rows[ok] * n + cols[ok], return_inverse=True)
    Kv = np.bincount(at, weights=K.reshape(-1)[ok], minlength=len(pair))
    Mv = np.bincount(at, weights=Mm.reshape(-1)[ok], minlength=len(pair))
    bv = np.zeros((2, n), complex)
    live = dof.ravel() >= 0
    for p in range(2):
        np.add.at(bv[p], dof.ravel()[live], b[:, :, p].ravel()[live])
    return pair // n, pair % n, Kv, Mv, bv


def _unet64(state, want_grad):
    """The network in float64: 3x3x3 convolutions as sums of 27 shifted products."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = torch.from_numpy(state["net"].params().astype(np.float64)).to(dev)
    ch = [16, 32, 64, 96]
    shapes = []
    for k in range(4):
        shapes += [(3, 16 if k == 0 else ch[k - 1], ch[k]), (3, ch[k], ch[k])]
    for k in range(3):
        shapes += [(3, ch[k + 1] + ch[k], ch[k]), (3, ch[k], ch[k])]
    shapes.append((1, 16, 16))
    ws, o = [], 0
    for ks, ci, co in shapes:
        w = p[o:o + ks ** 3 * ci * co].reshape(ks ** 3, co, ci).clone().requires_grad_(want_grad)
        o += ks ** 3 * ci * co
        bias = p[o:o + co].clone().requires_grad_(want_grad)
        o += co
        ws.append((ks, w, bias))

    def conv(u, i):
        ks, w, bias = ws[i]
        if ks == 1:
            return u @ w[0].T + bias
        _, nx, ny, nz, _ = u.shape
        v = torch.nn.functional.pad(u, (0, 0, 1, 1, 1, 1, 1, 1))
        out = bias
        for t in range(27):
            a, b, c = t // 9, t // 3 % 3, t % 3
            out = out + v[:, a:a + nx, b:b + ny, c:c + nz] @ w[t].T
        return out

    def act(u):
        return torch.where(u > 0, u, state["net"].cfg.leaky * u)

    def pool(u):
        bt, nx, ny, nz, c = u.shape
        return u.reshape(bt, nx // 2, 2, ny // 2, 2, nz // 2, 2, c).mean((2, 4, 6))

    def up(u):
        return u.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)

    h = torch.from_numpy(state["x"].astype(np.float64)).to(dev)
    h = torch.nn.functional.pad(h, (0, 16 - h.shape[-1]))
    skips = []
    for k in range(4):
        h = act(conv(act(conv(h, 2 * k)), 2 * k + 1))
        if k < 3:
            skips.append(h)
            h = pool(h)
    for k in (2, 1, 0):
        h = torch.cat([up(h), skips[k]], -1)
        h = act(conv(act(conv(h, 8 + 2 * k)), 9 + 2 * k))
    return conv(h, 14)[..., :learned.COUT], ws


def exact(case, seed):
    kind = case["kind"]
    if kind == "predict":
        state = prepare(case, seed)
        with torch.no_grad():
            return _unet64(state, False)[0].cpu().numpy()
    if kind == "train":
        state = prepare(case, seed)
        y, ws = _unet64(state, True)
        t, mask = (torch.from_numpy(state[k].astype(np.float64)).to(y.device) for k in ("t", "mask"))
        loss = (mask * (y - t) ** 2).sum() / mask.sum()
        loss.backward()
        g = torch.cat([v.grad.reshape(-1) for _, w, b in ws for v in (w, b)])
        p = torch.cat([v.detach().reshape(-1) for _, w, b in ws for v in (w, b)])
        # first Adam step: m / sqrt(v) with both moments bias-corrected
        return {"loss": float(loss.detach()), "grads": g.cpu().numpy(),
                "params": (p - 1e-4 * g / (g.abs() + state["net"].cfg.eps)).cpu().numpy()}
    if kind == "boundary" and case["nodes"] == 8 and case["nx"] * case["ny"] * case["nz"] <= 4000:
        m = _earth(case, seed)
        f = _freqs(case)[0]
        r, c, K, Mv, b = _assemble8(m, f)
        w32 = float(np.float32(2.0 * M.PI * f))
        upper = c >= r
        # the program hands its solver complex64-rounded values, zero below the diagonal
        a = np.where(upper, K.astype(np.float32) + 1j * (w32 * Mv).astype(np.float32), 0.0).astype(np.complex128)
        n = b.shape[1]
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        A = torch.zeros((n, n), dtype=torch.complex128, device=dev)
        rt, ct, at = (torch.from_numpy(v).to(dev) for v in (r[upper], c[upper], a[upper]))
        A[rt, ct] = at
        A[ct, rt] = at
        x = torch.linalg.solve(A, torch.from_numpy(b.T.copy()).to(dev)).cpu().numpy()
        return {"ia": None, "ja": None, "a": a, "b": b.ravel(), "x": x.T.ravel()}
    # larger grids: a dense or host sparse solution takes minutes
    return None
