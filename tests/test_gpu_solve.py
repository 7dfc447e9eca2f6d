"""GPU Krylov solve vs a direct FP64 solve of the same system.

The reference solves with MUMPS 4.10 (complex LDL^T of the complex64-rounded
upper triangle it assembles, MoVFEM_3DMT.f90:113-115), which is not available
here; SciPy's SuperLU (complex128) on exactly that matrix stands in for it.
Bars: FP64 true relative residual <= 1e-8 per polarization, and the solution
within 1e-6 (relative, 2-norm) of the direct solve."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from movfem_amd import _lib as L
from movfem_amd import model as M
from movfem_amd.vfem import GpuVfem, MvfError

pytestmark = pytest.mark.gpu


def reference_system(g):
    """Matrix and RHS exactly as the reference hands them to MUMPS."""
    ia, ja, a, b = g.global_vfem()
    ia, ja, a = g.remove_zeros(ia, ja, a)
    n = g.nne
    U = sp.coo_matrix((a, (ia - 1, ja - 1)), shape=(n, n)).tocsr()
    A = (U + sp.triu(U, 1).T).tocsc()
    return A, b.reshape(2, n)


def _check(A, b, x, xref, tol_res=1e-8, tol_x=1e-6):
    for d in range(2):
        r = np.linalg.norm(b[d] - A @ x[d]) / np.linalg.norm(b[d])
        assert r <= tol_res * 1.0001, (d, r)
        e = np.linalg.norm(x[d] - xref[d]) / np.linalg.norm(xref[d])
        assert e <= tol_x, (d, e)


@pytest.mark.parametrize("method,precision", [("cocg", "fp64"), ("bicgstab", "fp64"), ("cocg", "mixed")])
def test_solve_small_dirichlet(method, precision, need_gpu):
    m = M.random_small(8, 4, 4, 4, seed=11, nz_air=1, freqs=(1.0,))
    print(f"solve {method}/{precision} nne", flush=True)
    g = GpuVfem(m)
    g.set_frequency(0)
    A, b = reference_system(g)
    lu = spla.splu(A)
    xref = np.stack([lu.solve(b[d]) for d in range(2)])
    x, info = g.solve(b.ravel(), method=method, precision=precision, tol=1e-8)
    assert info["converged"], info
    _check(A, b, x.reshape(2, -1), xref)


def test_solve_gpml_20node(need_gpu):
    m = M.random_small(20, 3, 3, 3, seed=12, dirichlet=False, nextd=1, anisotropic=True, freqs=(10.0,))
    g = GpuVfem(m)
    g.set_frequency(0)
    A, b = reference_system(g)
    lu = spla.splu(A)
    xref = np.stack([lu.solve(b[d]) for d in range(2)])
    x, info = g.solve(b.ravel(), tol=1e-9)
    assert info["converged"], info
    _check(A, b, x.reshape(2, -1), xref, tol_res=1e-9)


def test_batched_frequencies_match_sequential(need_gpu):
    """One batched sweep over 3 frequencies == three single-frequency solves."""
    freqs = (0.1, 1.0, 10.0)
    m = M.random_small(8, 4, 3, 4, seed=13, nz_air=1, freqs=freqs)
    gb = GpuVfem(m)
    info = gb.solve_frequencies(freqs, tol=1e-9)
    assert info["converged"], info
    xb = gb.solution(6)
    gs = GpuVfem(m)
    for i in range(3):
        gs.set_frequency(i)
        A, b = reference_system(gs)
        x, inf2 = gs.solve(b.ravel(), tol=1e-9)
        x = x.reshape(2, -1)
        bb = gb.rhs(6)[2 * i:2 * i + 2]
        assert np.allclose(bb, b, rtol=1e-12, atol=1e-12 * np.abs(b).max())
        for d in range(2):
            assert np.linalg.norm(xb[2 * i + d] - x[d]) <= 1e-6 * np.linalg.norm(x[d])


def test_halfspace_block_solve(need_gpu):
    """The 8-node Dirichlet half-space + block workload (21,660 DOFs, 1 Hz).

    Three air layers above the first hold a gradient null space (see
    tests/gauge.py); the direct solve returns an arbitrary gauge there, so the
    1e-6 bar applies to the gauge-determined DOFs; the residual bar applies to
    every DOF."""
    from tests.gauge import determined_dofs

    m = M.halfspace_block()
    g = GpuVfem(m)
    g.set_frequency(0)
    A, b = reference_system(g)
    lu = spla.splu(A)
    xref = np.stack([lu.solve(b[d]) for d in range(2)])
    x, info = g.solve(b.ravel(), tol=1e-8)
    x = x.reshape(2, -1)
    print("halfspace_block", info["iterations"], info["seconds"], flush=True)
    assert info["converged"], info
    mask = determined_dofs(m, g.gne())
    assert 0.5 < mask.mean() < 1.0
    for d in range(2):
        r = np.linalg.norm(b[d] - A @ x[d]) / np.linalg.norm(b[d])
        assert r <= 1e-8 * 1.0001, (d, r)
        e = np.linalg.norm(x[d][mask] - xref[d][mask]) / np.linalg.norm(xref[d][mask])
        print(f"pol {d}: determined-DOF rel L2 {e:.2e}, full-vector {np.linalg.norm(x[d]-xref[d])/np.linalg.norm(xref[d]):.2e}")
        assert e <= 1e-6, (d, e)


def test_sixteen_frequencies_one_call(need_gpu):
    """The 27-node workload's 16 frequencies (1e-3 to 1e3 Hz) in one
    mvf_solve_frequencies call, which solves them in two batches of 8: every
    frequency to the bar on its own system, and a frequency of the second
    batch equal to its single-frequency solve.  Emulation off, so every
    frequency's system is consistent (the reference's update_sigma range
    leaves the second and later frequencies' air sources the null space
    cannot absorb)."""
    freqs = tuple(np.logspace(-3, 3, 16))
    m = M.random_small(8, 4, 4, 4, seed=14, nz_air=1, freqs=freqs)
    g = GpuVfem(m, emulate=0)
    print("16 frequencies: one call", flush=True)
    info = g.solve_frequencies(list(freqs), method="gmres", precond="direct", tol=1e-8)
    assert info["converged"], info
    assert len(info["true_resid"]) >= 32
    assert max(info["true_resid"][:32]) <= 1e-8 * 1.0001, info["true_resid"][:32]
    xb = g.solution(32)
    i = 12
    gs = GpuVfem(m, emulate=0)
    gs.set_frequency(i)
    A, b = reference_system(gs)
    assert np.allclose(g.rhs(32)[2 * i:2 * i + 2], b, rtol=1e-12, atol=1e-12 * np.abs(b).max())
    x, _ = gs.solve(b.ravel(), method="gmres", precond="direct", tol=1e-8)
    x = x.reshape(2, -1)
    xref = np.stack([spla.splu(A).solve(b[d]) for d in range(2)])
    _check(A, b, xb[2 * i:2 * i + 2], xref)
    _check(A, b, x, xref)


@pytest.mark.parametrize("matrix", ["c64ref", "fp64"])
@pytest.mark.parametrize("nodes,sides,nf", [
    (8, (5, 4, 3), 1),     # two columns, rows shorter than one pass of the lanes
    (8, (11, 9, 7), 2),    # four columns, several workgroups
    (20, (4, 3, 3), 1),    # ~84 entries per row: more than one pass at 4 and 8 lanes per row
    (20, (4, 3, 3), 2),
    (27, (3, 3, 2), 2),
    (8, (5, 4, 3), 3),     # six columns padded to eight, one lane per entry
])
def test_cocg_columns_and_rows(nodes, sides, nf, matrix, need_gpu):
    """The SpMV and the updates for every column count, short and long rows and
    both matrix roundings: the residual of each column, formed on the host from
    the entry list, is the tolerance of 1e-9 (times 1.1: the host's own sums of
    ~100 products round at 1e-14)."""
    freqs = tuple(20.0 * 3.0 ** k for k in range(nf))
    m = M.random_small(nodes, *sides, seed=41, full_tensor=True, freqs=freqs)
    g = GpuVfem(m, emulate=0)
    info = g.solve_frequencies(freqs, method="cocg", matrix=matrix, tol=1e-9, maxit=20000, use_graph=nf == 2)
    assert info["converged"], info
    x, bb = g.solution(2 * nf), g.rhs(2 * nf)
    for i in range(nf):
        g2 = GpuVfem(m, emulate=0)
        g2.set_frequency(i)
        A, _ = reference_system(g2)
        for d in range(2):
            b = bb[2 * i + d]
            r = np.linalg.norm(b - A @ x[2 * i + d]) / np.linalg.norm(b)
            # the unrounded operator differs from the complex64 entry list by its rounding, 2^-24 relative
            assert r <= (1.1e-9 if matrix == "c64ref" else 1e-5), (i, d, r)


@pytest.mark.parametrize("form", [4, 8, 16, 32, -4, -8])  # lanes per row; negative: the grouped form
@pytest.mark.parametrize("nodes,sides,method,nf", [
    (8, (5, 4, 3), "cocg", 1),       # rows shorter than one pass, fewer rows than a workgroup takes
    (8, (11, 9, 7), "cocg", 2),      # several workgroups, the last partly filled
    (8, (11, 9, 7), "bicgstab", 2),  # without the dot product
    (20, (4, 3, 3), "cocg", 2),      # ~84 entries: several passes
    (20, (4, 3, 3), "bicgstab", 1),
    (8, (5, 4, 3), "cocg", 3),       # eight columns: no grouped form, the autotuner's width instead
])
def test_spmv_forms(form, nodes, sides, method, nf, monkeypatch, need_gpu):
    """Every form of the SpMV the autotuner can choose, forced: the residual of each
    column, formed on the host, is at most the tolerance (as in
    test_cocg_columns_and_rows)."""
    monkeypatch.setenv("MVF_SPMV", str(form))
    freqs = tuple(20.0 * 3.0 ** k for k in range(nf))
    m = M.random_small(nodes, *sides, seed=41, full_tensor=True, freqs=freqs)
    g = GpuVfem(m, emulate=0)
    info = g.solve_frequencies(freqs, method=method, tol=1e-9, maxit=20000)
    assert info["converged"], info
    assert nf == 3 or info["spmv_lpr"] == abs(form)
    x, bb = g.solution(2 * nf), g.rhs(2 * nf)
    for i in range(nf):
        g.set_frequency(i)
        A, _ = reference_system(g)
        for d in range(2):
            b = bb[2 * i + d]
            assert np.linalg.norm(b - A @ x[2 * i + d]) <= 1.1e-9 * np.linalg.norm(b)


@pytest.mark.parametrize("form", [8, -8, 0])
def test_spmv_large_grid(form, monkeypatch, need_gpu):
    """249k DOFs, beyond the workgroups of either form (each takes several passes
    over the rows, the last partly filled); form 0: the autotuner's choice."""
    if form:
        monkeypatch.setenv("MVF_SPMV", str(form))
    freqs = (50.0, 80.0)
    m = M.anisotropic_blocks(nx=47, ny=50, nz_earth=35, nz_air=2, h=500.0, nodes=8, freqs=freqs, block=4, seed=5,
                             full_tensor=True, dirichlet=True, nextd=2)
    g = GpuVfem(m, emulate=0)
    info = g.solve_frequencies(freqs, method="cocg", tol=1e-8, maxit=20000)
    assert info["converged"], info
    x, bb = g.solution(4), g.rhs(4)
    for i in range(2):
        g.set_frequency(i)
        A, _ = reference_system(g)
        for d in range(2):
            b = bb[2 * i + d]
            assert np.linalg.norm(b - A @ x[2 * i + d]) <= 1.1e-8 * np.linalg.norm(b)


def test_solution_buffers_out_of_memory(need_gpu):
    """The solution or right-hand-side buffer finds no memory (reported on the
    host) when a call needs more columns: the call says so, nothing is left to
    read out, and a call with the first column count solves again."""
    fail = L.lib().mvf_fail_allocs
    freqs = (20.0, 50.0, 90.0)
    g = GpuVfem(M.random_small(8, 5, 4, 4, seed=51, freqs=freqs), emulate=0)
    opts = dict(method="cocg", tol=1e-10, maxit=20000)
    g.solve_frequencies(freqs[:1], **opts)
    x0 = g.solution(2)
    for skip in (0, 1):
        g.close()
        g = GpuVfem(M.random_small(8, 5, 4, 4, seed=51, freqs=freqs), emulate=0)
        g.solve_frequencies(freqs[:1], **opts)
        fail(skip, 2)
        with pytest.raises(MvfError) as e:
            g.solve_frequencies(freqs, **opts)
        assert (e.value.code, fail(0, 0)) == (L.MVF_E_MEMORY, 0)
        for read in (lambda: g.solution(2), lambda: g.rhs(2), lambda: g.readout(None, f=0)):
            with pytest.raises(MvfError):
                read()
        g.solve_frequencies(freqs[:1], **opts)
        # the relative residual is below 1e-10 in both solves
        assert np.linalg.norm(g.solution(2) - x0) <= 1e-5 * np.linalg.norm(x0)
        g.readout(None, f=0)
    g.close()


def test_assemble_out_of_memory(need_gpu):
    """Re-assembly whose second element buffer finds no memory (reported on the
    host): the call says so each time, loses no device memory (the first buffer
    holds 22 MB) and leaves the operators as they were."""
    import torch

    fail = L.lib().mvf_fail_allocs
    g = GpuVfem(M.random_small(27, 12, 12, 13, seed=51, freqs=(20.0,)), emulate=0)
    ops = g.operators()
    g.assemble()
    before = torch.cuda.mem_get_info()[0]
    for _ in range(20):
        fail(1, 2)
        with pytest.raises(MvfError) as e:
            g.assemble()
        assert (e.value.code, fail(0, 0)) == (L.MVF_E_MEMORY, 0)
    assert torch.cuda.mem_get_info()[0] >= before - (64 << 20)
    for a, b in zip(ops, g.operators()):
        assert np.array_equal(a, b)
    g.close()
