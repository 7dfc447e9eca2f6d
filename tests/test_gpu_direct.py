"""Sparse direct factorization on the device (MVF_PC_DIRECT) against SciPy.

The reference solves every frequency with MUMPS 4.10 (complex LDL^T with
pivoting, MoVFEM_3DMT.f90:113-115), absent here; SciPy's SuperLU (complex128)
on the same matrix stands in for it.  Bars, per polarization:
  * true relative residual ||b - A x|| / ||b|| <= 1e-8 on the matrix the
    reference hands MUMPS (complex64-rounded values, global_assembly.f90:157);
  * relative L2 distance to the SuperLU solution <= 1e-6 on the
    gauge-determined DOFs (tests/gauge.py): all-air elements carry no mass
    (integration.f90:211-238), so any solver leaves the gradient part of the
    field there arbitrary.
The cases include the 20-node GPML system at 1e-3 Hz on which
Jacobi-preconditioned Krylov does not converge."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from movfem_amd import _lib as L
from movfem_amd import model as M
from movfem_amd.vfem import GpuVfem, MvfError
from tests.gauge import determined_dofs, inner_dofs

pytestmark = pytest.mark.gpu


def reference_system(g):
    ia, ja, a, b = g.global_vfem()
    ia, ja, a = g.remove_zeros(ia, ja, a)
    n = g.nne
    U = sp.coo_matrix((a, (ia - 1, ja - 1)), shape=(n, n)).tocsr()
    return (U + sp.triu(U, 1).T).tocsc(), b.reshape(2, n)


CASES = {
    "hex8_dirichlet": lambda: M.random_small(8, 5, 4, 4, seed=21, nz_air=1, freqs=(1.0,)),
    "hex8_gpml_aniso_air3": lambda: M.anisotropic_blocks(nx=6, ny=6, nz_earth=3, nz_air=3, nodes=8, freqs=(100.0,),
                                                         block=2, seed=3, nextd=2),
    "hex20_gpml_aniso_1mHz": lambda: M.anisotropic_blocks(nx=8, ny=8, nz_earth=5, nz_air=3, nodes=20, freqs=(1e-3,),
                                                          block=2, seed=2, nextd=2),
    "hex27_dirichlet_tensor": lambda: M.random_small(27, 3, 3, 3, seed=22, nz_air=1, full_tensor=True, freqs=(3.0,)),
}


@pytest.mark.parametrize("tile", [0, 128])
@pytest.mark.parametrize("name", sorted(CASES))
def test_direct_matches_superlu(name, tile, need_gpu):
    """tile 0 picks the GEMM tile by front size (64 on these small fronts);
    128 forces the large-front kernel onto every level and edge shape."""
    m = CASES[name]()
    print(f"direct {name} tile {tile}: building", flush=True)
    g = GpuVfem(m)
    g.set_frequency(0)
    A, b = reference_system(g)
    lu = spla.splu(A)
    xref = np.stack([lu.solve(b[d]) for d in range(2)])
    print(f"direct {name}: nne={g.nne} solving", flush=True)
    # 1e-9: the solutions are compared to 1e-6, and at 1 mHz under GPML the
    # condition number is ~1e3, so a 1e-8 residual leaves that bar no margin
    x, info = g.solve(b.ravel(), method="gmres", precond="direct", tol=1e-9, direct_tile=tile)
    x = x.reshape(2, -1)
    print(f"direct {name}: its={info['iterations']} applies={info['precond_applies']} "
          f"pert={info['static_pivots']} factor {info['factor_seconds']:.3f}s", flush=True)
    assert info["converged"], info
    # GPML models: outside the stretched zones, whose modes a residual of 1e-8
    # determines only weakly (as in test_direct_frequency_sweep)
    mask = determined_dofs(m, g.gne()) & inner_dofs(m, g.gne())
    for d in range(2):
        r = np.linalg.norm(b[d] - A @ x[d]) / np.linalg.norm(b[d])
        assert r <= 1e-8 * 1.0001, (d, r)
        e = np.linalg.norm(x[d][mask] - xref[d][mask]) / np.linalg.norm(xref[d][mask])
        print(f"direct {name}: pol {d} residual {r:.2e}, solution difference {e:.2e}", flush=True)
        assert e <= 1e-6, (d, e)


def test_direct_frequency_sweep(need_gpu):
    """Device-resident RHS, one factorization per frequency, three frequencies.
    Solutions are compared on gauge-determined DOFs outside the GPML zones
    (tests/gauge.py).  Emulation switches off: the reference's update_sigma leaves earlier
    frequencies' i*omega*eps on most air nodes (geometry.f90:146-152), which
    puts a source into all-air elements that the air gradient null space
    cannot absorb, so no solver reaches 1e-8 there."""
    freqs = (1e-3, 0.3, 30.0)
    m = M.anisotropic_blocks(nx=6, ny=6, nz_earth=4, nz_air=2, nodes=20, freqs=freqs, block=2, seed=5, nextd=2)
    g = GpuVfem(m, emulate=0)
    # 1e-10: the PML modes with mass but no stiffness are weakly determined,
    # so a 1e-8 residual leaves ~1e-5 differences there (observed at 30 Hz);
    # FP64 GMRES bottoms out near 1e-11 on this system
    info = g.solve_frequencies(freqs, method="gmres", precond="direct", tol=1e-10)
    print("sweep", info["iterations"], info["factorizations"], info["factor_seconds"], flush=True)
    assert info["converged"], info
    assert max(info["true_resid"][:6]) <= 1e-10 * 1.0001
    x = g.solution(6)
    bb = g.rhs(6)
    mask = determined_dofs(m, g.gne()) & inner_dofs(m, g.gne())
    assert mask.sum() > 0.2 * len(mask)
    for i in range(3):
        g2 = GpuVfem(m, emulate=0)
        g2.set_frequency(i)
        A, b = reference_system(g2)
        assert np.allclose(b, bb[2 * i:2 * i + 2], rtol=1e-12, atol=1e-14 * np.abs(b).max())
        lu = spla.splu(A)
        for d in range(2):
            xr = lu.solve(b[d])
            rr = np.linalg.norm(b[d] - A @ xr) / np.linalg.norm(b[d])
            e = np.linalg.norm(x[2 * i + d][mask] - xr[mask]) / np.linalg.norm(xr[mask])
            print(f"f={freqs[i]} pol {d}: SuperLU residual {rr:.1e}, determined-DOF difference {e:.1e}")
            # at 30 Hz the 6x6x6 grid is only two cells from its absorbing
            # zones: a 1e-10 residual bounds the difference at ~1e-6 there
            # (observed 0.6-4e-6 depending on the GEMM's rounding), 1e-8 elsewhere
            assert e <= (1e-5 if freqs[i] >= 10 else 1e-6), (i, d, e, rr)


def test_direct_lookahead_fronts(need_gpu):
    """20-node 14 x 14 x 11 GPML model whose largest fronts own 974 DOFs:
    four outer blocks of 256, so the factorization overlaps the trailing
    part of each outer update with the next
    block's panels on its second stream, and the fronts above 512 run the
    128 x 64 three-product tiles.  An error in either split or in the stream
    ordering corrupts the factor that preconditions GMRES: the bar is the
    true residual on the reference's matrix within the few iterations an
    exact factor needs, at both ends of the frequency range."""
    from tests.test_direct_plan import plan_stats
    from oracle.oracle import Oracle
    for f in (1e-3, 100.0):  # one frequency per model, as the reference's first frequency
        m = M.anisotropic_blocks(nx=14, ny=14, nz_earth=8, nz_air=3, nodes=20, freqs=(f,), block=2, seed=5, nextd=2)
        if f == 1e-3:
            o = Oracle(m)
            s = plan_stats(m, o.gne(), o.nne)
            assert s["max_n1"] > 3 * 256, s
        g = GpuVfem(m)
        g.set_frequency(0)
        A, b = reference_system(g)
        print(f"lookahead fronts: f={f} nne={g.nne} solving", flush=True)
        x, info = g.solve(b.ravel(), method="gmres", precond="direct", tol=1e-8)
        x = x.reshape(2, -1)
        print(f"lookahead fronts: f={f} its={info['iterations']} pert={info['static_pivots']}", flush=True)
        assert info["converged"] and info["iterations"] <= 10, info
        for d in range(2):
            r = np.linalg.norm(b[d] - A @ x[d]) / np.linalg.norm(b[d])
            assert r <= 1e-8 * 1.0001, (f, d, r)


@pytest.mark.parametrize("nodes,sides", [
    (8, (5, 3, 2)),    # a root of one partial panel with nothing right of it
    (8, (9, 7, 6)),    # last panels of every width the small fronts have
    (20, (5, 5, 3)),
    (20, (9, 3, 3)),   # narrow separators: fronts with one partial panel
    (27, (4, 3, 5)),
])
@pytest.mark.parametrize("tile", [0, 128])
def test_direct_block_rows(nodes, sides, tile, need_gpu):
    """Symmetric block factorization on fronts with partial panels, partial
    column tiles and no update columns.  With every pivot block nonsingular the
    factor is that of the matrix itself up to the air shift, so GMRES needs at
    most four iterations, and the solution is SuperLU's to 1e-6 where it is
    determined (a residual of 1e-10 at condition numbers below 1e4)."""
    m = M.random_small(nodes, *sides, seed=31, nz_air=1, full_tensor=True, freqs=(10.0,))
    g = GpuVfem(m)
    g.set_frequency(0)
    A, b = reference_system(g)
    lu = spla.splu(A)
    x, info = g.solve(b.ravel(), method="gmres", precond="direct", tol=1e-10, direct_tile=tile)
    x = x.reshape(2, -1)
    print(f"block rows {nodes} {sides}: nne={g.nne} its={info['iterations']}", flush=True)
    assert info["converged"] and info["iterations"] <= 4, info
    mask = determined_dofs(m, g.gne())
    for d in range(2):
        xr = lu.solve(b[d])
        assert np.linalg.norm(x[d][mask] - xr[mask]) <= 1e-6 * np.linalg.norm(xr[mask])


def test_direct_out_of_memory(need_gpu):
    """Every device allocation of a first direct solve fails in turn (reported on
    the host; both tries).  The call returns MVF_E_MEMORY, and the next call on
    the same handle solves: no half-built plan is left to run on."""
    fail = L.lib().mvf_fail_allocs
    m = M.random_small(8, 5, 4, 4, seed=33, nz_air=1, freqs=(10.0,))
    opts = dict(method="gmres", precond="direct", tol=1e-10)
    g = GpuVfem(m)
    g.set_frequency(0)
    mask = determined_dofs(m, g.gne())
    _, _, _, b = g.global_vfem()
    xr = g.solve(b, **opts)[0].reshape(2, -1)[:, mask]
    g.close()
    for skip in range(100):
        g = GpuVfem(m)
        g.set_frequency(0)
        fail(skip, 2)
        try:
            g.solve(b, **opts)
            code = 0
        except MvfError as e:
            code = e.code
        unused = fail(0, 0)
        assert (code, unused) in ((L.MVF_E_MEMORY, 0), (0, 2)), (skip, code, unused)
        x, info = g.solve(b, **opts)
        assert info["converged"], info
        assert np.linalg.norm(x.reshape(2, -1)[:, mask] - xr) <= 1e-6 * np.linalg.norm(xr)
        g.close()
        if not code:
            break
    print(f"allocations failed in turn: {skip}", flush=True)
    assert 20 <= skip < 99
