"""Kernels of one lane per cell or face at the sizes where their index maps can
go wrong: blocks of 4 to 64 cells (odd numbers of 4-cell rows, pencils that do
not fill a workgroup, workgroups over several blocks), launches on both sides
of the small-grid rule, adjoint faces over several tiles, fine faces of small
blocks, a handful of states, and transfers on both sides of the rules that
convert them on the host, in one piece or through staged ones."""
import ctypes

import numpy as np
import pytest
import torch   # before the library: one HIP runtime in the process

from amun_amd import mesh, solver
from amun_amd.config import Params
from amun_amd.problems import prim_to_cons
from amun_amd.solver import AmrSolver, Solver
import oracle_lib as ol
import test_gpu_amr as amr
from test_gpu_parity import _mhd_state, relerr

pytestmark = pytest.mark.gpu


def _params(nd, eq, rec, n, blocks, precision="fp64", **kw):
    ext = np.array(blocks + (1,) * (3 - len(blocks)), dtype=float)
    ext /= ext.max()
    return Params(ndims=nd, equation_system=eq, reconstruction=rec, limiter="mc",
                  riemann_solver="hlld" if eq == "mhd" else "hllc", time_advance="rk2",
                  gamma=5.0 / 3.0 if eq == "mhd" else 1.4, cfl=0.3, ncells=n,
                  nghosts=4 if rec == "weno5z" else 2, xblocks=blocks[0], yblocks=blocks[1],
                  zblocks=blocks[2] if nd == 3 else 1, xmin=0.0, xmax=ext[0], ymin=0.0,
                  ymax=ext[1], zmin=0.0, zmax=ext[2], precision=precision, **kw)


def _state(p):
    """smooth rows with noise; HD takes the first four and the pressure"""
    u = _mhd_state(p, noise=0.01)
    if p.equation_system == "mhd":
        return u
    q = np.stack([u[0], u[1] / u[0], u[2] / u[0], u[3] / u[0], 0.5 + 0.1 * u[0]])
    return prim_to_cons(p, q)


SWEEPS = [(2, "hd", "tvd", 4, (5, 3)), (2, "mhd", "weno5z", 12, (3, 2)),
          (2, "mhd", "tvd", 20, (2, 3)), (2, "hd", "weno5z", 64, (1, 2)),
          (2, "hd", "tvd", 16, (15, 14)), (2, "hd", "tvd", 16, (16, 15)),
          (3, "hd", "tvd", 4, (3, 2, 5)), (3, "mhd", "weno5z", 12, (2, 1, 3)),
          (3, "hd", "weno5z", 20, (1, 2, 1)), (3, "mhd", "tvd", 28, (1, 2, 1)),
          (3, "mhd", "tvd", 16, (3, 2, 3))]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("case", SWEEPS)
def test_sweep_sizes_vs_oracle(case, precision):
    """One RK2 step.  FP64 within 1e-12, as every step against the oracle.
    Mixed: a step moves the state by at most cfl of the neighbours' states in
    each of two stages, with face fluxes of FP32 arithmetic; 16 roundings of
    2^-24 on fluxes whose momentum part (the pressure) is up to 8 times the
    momentum's own gives 2 x 0.3 x 16 x 8 x 2^-24 = 4.6e-6 of the largest
    value; psi, made by cancellations in div B, on the scale of B."""
    p = _params(*case, precision=precision)
    print(f"[case] {case} {precision}", flush=True)
    u0 = _state(p)
    o = ol.OracleRun(_params(*case))
    o.set_state(u0)
    tr = o.run(1)
    uo = o.get_state()
    with Solver(p) as s:
        s.upload(u0)
        dt, _ = s.advance()
        ug = s.download()
    assert dt == pytest.approx(tr[0, 0], rel=1e-13)
    assert relerr(ug, uo).max() <= (1e-12 if precision == "fp64" else 4.6e-6)


@pytest.mark.parametrize("nd,n,blocks", [(2, 4, (3, 5)), (2, 64, (2, 1)), (2, 16, (17, 16)),
                                         (3, 4, (3, 2, 2)), (3, 12, (2, 1, 2)),
                                         (3, 20, (1, 2, 1))])
def test_adjoint_sizes(nd, n, blocks):
    """<lam, T(du0, dg)> = <A(lam), du0> + A_gamma(lam) dg to round-off, at
    block sizes with fewer and more faces than a tile of the adjoint holds, and
    on both sides of its rules for few tiles"""
    p = _params(nd, "mhd", "tvd", n, blocks)
    print(f"[case] adjoint {nd}D n={n} blocks={blocks}", flush=True)
    u0 = _mhd_state(p, noise=0.01)
    rng = np.random.default_rng(5)
    lam = rng.normal(size=u0.shape)
    du0 = rng.normal(size=u0.shape) * 1e-3
    with Solver(p) as s:
        s.upload(u0)
        s.tape_forward(3, 2)
        du = s.tape_tangent(du0, 0.01)
        lam0, gg = s.tape_backward(lam)
    lhs, rhs = float((lam * du).sum()), float((lam0 * du0).sum()) + gg * 0.01
    assert abs(lhs - rhs) <= 1e-11 * (abs(lhs) + abs(rhs))


@pytest.mark.parametrize("nd,n", [(2, 4), (2, 20), (3, 4), (3, 12)])
def test_fine_faces_vs_oracle(nd, n):
    """One step of a 3-level mesh of small and odd blocks: the fluxes of the
    fine faces against the oracle (and the transfer of block interiors)."""
    p, _, _ = amr._case(nd)
    p.ncells = n
    meta = mesh.refine(p, mesh.near_sphere(p, 0.15, 0.05), 3)
    u0 = mesh.block_state(p, meta, mesh.blast_prim(p))
    print(f"[case] fine faces {nd}D n={n} blocks={len(meta)}", flush=True)
    o = ol.OracleAmr(p, meta)
    o.set_blocks(u0)
    o.run(1)
    uo = o.get_blocks()
    with AmrSolver(p, meta) as s:
        assert s.info()["corrected_faces"] > 0
        s.upload(u0)
        np.testing.assert_array_equal(s.download().reshape(u0.shape), u0)
        s.run(1)
        ug = s.download()
    assert amr.relerr(ug.reshape(-1, p.nv), uo.reshape(-1, p.nv)).max() <= 1e-12


@pytest.mark.parametrize("eq", ["hd", "srmhd"])
@pytest.mark.parametrize("n", [1, 63, 64, 65])
def test_cons2prim_noalloc_sizes(eq, n):
    """Counts and states of the allocation-free cons2prim at the edges of a
    wave, two calls on the same counters, against the unit entry point."""
    p = Params(ndims=3, equation_system=eq, reconstruction="tvd", gamma=5.0 / 3.0,
               riemann_solver="hll")
    rng = np.random.default_rng(n)
    q = np.zeros((n, p.nv))
    q[:, 0], q[:, p.nv - 1] = rng.uniform(0.5, 2, n), rng.uniform(0.1, 1, n)
    q[:, 1:4] = 0.3 * rng.uniform(-1, 1, (n, 3))
    u = np.ascontiguousarray(prim_to_cons(p, q.T).T)
    u[n // 2, p.nv - 1] *= 1e-3                       # one recovery that fails
    ref, ev = solver.unit_cons2prim(p, u, q, events=True)
    lib, cfg = solver.load_library(), p.to_cfg()
    du, dev = torch.from_numpy(u).cuda(), torch.full((3,), -1, dtype=torch.int64, device="cuda")
    for _ in range(2):
        dq = torch.from_numpy(q).cuda()
        assert lib.amun_dev_cons2prim_noalloc(
            ctypes.byref(cfg), n, du.data_ptr(), dq.data_ptr(), dev.data_ptr(),
            torch.cuda.current_stream().cuda_stream) == 0
        np.testing.assert_array_equal(dq.cpu().numpy(), ref)
        assert dev.cpu().tolist() == list(ev)


@pytest.mark.parametrize("blocks", [(128, 63), (128, 64), (128, 65)])
def test_download_sizes(blocks):
    """Four variables of 2048 x 1008, 1024 and 1040 cells: just below, at and
    beyond (with an incomplete last piece) the 64 MiB of the staged copy.  The
    state comes back as it went, twice, and after a step as its blocks hold it."""
    p = _params(2, "hd", "tvd", 16, blocks, equation_of_state="iso", csnd=0.8)
    p.riemann_solver = "hll"
    u0 = np.random.default_rng(1).uniform(0.9, 1.1, (4,) + p.shape)
    with Solver(p) as s:
        s.upload(u0)
        for _ in range(2):
            np.testing.assert_array_equal(s.download(), u0)
        s.run(1)
        u, b = s.download(), s.download_blocks()
    g, n = p.nghosts, p.ncells
    b = np.asarray(b).reshape(blocks[1], blocks[0], n + 2 * g, n + 2 * g, 4)
    b = b[:, :, g:g + n, g:g + n].transpose(4, 0, 2, 1, 3).reshape(u.shape)
    np.testing.assert_array_equal(u, b)


def test_contexts_share_a_kernel():
    """A context of 4-cell blocks (83 KB of LDS a workgroup) steps on after
    one of 16-cell blocks (39 KB) has taken the same kernels into use."""
    small, large = (_params(3, "mhd", "weno5z", n, (2, 1, 2)) for n in (4, 16))
    u0 = _state(small)
    print("[case] contexts of 4- and 16-cell blocks", flush=True)
    with Solver(small) as a:
        a.upload(u0)
        want = a.run(3), a.download()
        a.upload(u0)
        with Solver(large) as b:
            b.upload(_state(large))
            b.run(1)
            np.testing.assert_array_equal(a.run(3), want[0])
        np.testing.assert_array_equal(a.download(), want[1])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nd,eq,n,blocks", [(2, "hd", 4, (1, 1)), (2, "mhd", 16, (3, 1)),
                                            (2, "hd", 4, (12, 25)), (2, "hd", 4, (7, 43)),
                                            (3, "mhd", 4, (3, 2, 5)), (3, "hd", 16, (1, 1, 1)),
                                            (3, "mhd", 12, (2, 1, 1)), (3, "mhd", 4, (43, 1, 1))])
def test_small_download_sizes(nd, eq, n, blocks, precision):
    """States below, next to (187.5 and 188.1 of 192 KiB; 193.5) and above the
    size that is converted on the host, with their primitives: the values that
    the block arrays hold."""
    p = _params(nd, eq, "tvd", n, blocks, precision)
    print(f"[case] small download {nd}D {eq} n={n} blocks={blocks} {precision}", flush=True)
    with Solver(p) as s:
        s.upload(_state(p))
        s.run(1)
        got = s.download(with_q=True)
        blk = s.download_blocks(with_q=True)
    bx, by, bz = (blocks + (1,))[:3]
    g, kn = p.nghosts, n if nd == 3 else 1
    for a, b in zip(got, blk):
        b = b.reshape((bz, by, bx) + b.shape[1:])[:, :, :, g if nd == 3 else 0:][:, :, :, :kn]
        b = b[:, :, :, :, g:g + n, g:g + n].transpose(6, 0, 3, 1, 4, 2, 5)
        np.testing.assert_array_equal(a, b.reshape(a.shape))


@pytest.mark.parametrize("nd,eq,n,blocks", [(2, "hd", 4, (1, 1)), (2, "mhd", 32, (1, 1)),
                                            (2, "mhd", 16, (12, 11)), (2, "mhd", 32, (8, 8)),
                                            (3, "hd", 8, (5, 5, 5)), (3, "hd", 4, (24, 24, 12)),
                                            (2, "mhd", 16, (32, 32)), (3, "mhd", 8, (10, 9, 10))])
def test_block_upload_sizes(nd, eq, n, blocks):
    """Block arrays with ghost layers on both sides of the rule that gathers
    their interiors on the host (0.6 KB to 33 MB; ghost layers of 0.3 to 7
    times the interiors): the state of the interiors, whatever the ghost cells
    hold."""
    p = _params(nd, eq, "tvd", n, blocks)
    print(f"[case] block upload {nd}D {eq} n={n} blocks={blocks}", flush=True)
    u0 = _state(p)
    g = p.nghosts
    bx, by, bz = (blocks + (1,))[:3]
    gk, kn = (g, n) if nd == 3 else (0, 1)
    inner = u0.reshape(p.nv, bz, kn, by, n, bx, n).transpose(1, 3, 5, 2, 4, 6, 0)
    with Solver(p) as s:
        ub = np.full(s._block_shape(), np.nan)
        ub[:, gk:gk + kn, g:g + n, g:g + n] = inner.reshape(-1, kn, n, n, p.nv)
        for _ in range(2):
            s.upload_blocks(ub)
            np.testing.assert_array_equal(s.download(), u0)
            s.run(1)
        got = s.download()
        s.upload(u0)
        s.run(1)
        np.testing.assert_array_equal(got, s.download())


@pytest.mark.parametrize("blocks", [(3, 3), (12, 11), (40, 38)])
def test_ghosted_download_sizes(blocks):
    """Block arrays of an open domain in one copy (u and q of 141 KB each), in
    one piece (2.1 MB) and in several (24 MB): u alone and with q, interiors
    as the global arrays hold them, ghost layers as the neighbours do."""
    p = _params(2, "hd", "tvd", 16, blocks)
    p.xlbndry = p.xubndry = p.ylbndry = p.yubndry = "open"
    print(f"[case] ghosted download blocks={blocks}", flush=True)
    with Solver(p) as s:
        s.upload(_state(p))
        s.run(1)
        glob = s.download(with_q=True)
        u = s.download_blocks()
        blk = s.download_blocks(with_q=True)
    np.testing.assert_array_equal(u, blk[0])
    g, n, (bx, by) = p.nghosts, p.ncells, blocks
    u, q = (b.reshape(by, bx, n + 2 * g, n + 2 * g, p.nv) for b in blk)
    for b, a in zip((u, q), glob):
        b = b[:, :, g:g + n, g:g + n].transpose(4, 0, 2, 1, 3)
        np.testing.assert_array_equal(b.reshape(a.shape), a)
    np.testing.assert_array_equal(q[:, 1:, g:-g, :g], q[:, :-1, g:-g, n:n + g])
    np.testing.assert_array_equal(q[:-1, :, n + g:, g:-g], q[1:, :, g:2 * g, g:-g])
    np.testing.assert_array_equal(q[:, 0, g:-g, 0], q[:, 0, g:-g, g])      # open side
    np.testing.assert_allclose(u[:, 1:, g:-g, :g], u[:, :-1, g:-g, n:n + g], rtol=1e-14, atol=1e-15)
