"""Launch shapes and the stage switch (amun_dev_set_stage_fusion).

The configurations of CASES (2D and 3D, HD and MHD, adiabatic and isothermal,
TVD and WENO5-Z, Roe, blocks of 4 to 16 cells, viscous, resistive and gravity
sources) take one step against the oracle, and several with every workgroup
size and order of amun_dev_set_launch, which must give the same bits: the
workgroups, and so the pencils and tiles of a lane, differ, the arithmetic of
a cell does not.  The stage switch changes the times that amun_dev_timed_run
reports and nothing else; on, off and toggled, the results are the same."""
import os
import sys

import numpy as np
import pytest

from amun_amd.config import Params, c1_params, c2_params
from amun_amd.problems import cell_centres, initial_state, prim_to_cons
from amun_amd.solver import AmunError, Solver

GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
sys.path.insert(0, GOLD)
from make_golden import grav_params, grav_state  # noqa: E402
import oracle_lib as ol  # noqa: E402
from test_gpu_parity import relerr  # noqa: E402

pytestmark = pytest.mark.gpu


def noisy(p, seed):
    """rho ~ 1, small velocities, B ~ 0.3, p ~ 1, each with 10% noise"""
    rng = np.random.default_rng(seed)
    z, y, x = cell_centres(p)
    shape = (len(z) if p.ndims == 3 else 1, len(y), len(x))
    q = rng.uniform(-0.1, 0.1, (p.nv,) + shape)
    q[0] += 1.0
    if p.equation_system == "mhd":
        q[4:7] += 0.3
        q[7] *= 0.1
    if p.equation_of_state not in ("iso", "isothermal"):
        q[p.nv - 1] += 1.0
    return prim_to_cons(p, q)


def _cfg(nd, eq, rec, rs, ta="rk3", n=8, **kw):
    p = Params(ndims=nd, equation_system=eq, reconstruction=rec, limiter="mc",
               riemann_solver=rs, time_advance=ta, gamma=5.0 / 3.0 if eq == "mhd" else 1.4,
               cfl=0.3, ncells=n, nghosts=4 if rec == "weno5z" else 2, xblocks=2, yblocks=2,
               zblocks=2 if nd == 3 else 1, **kw)
    return p


CASES = {
    "c1_hd2d_tvd_hllc": lambda: c1_params(),
    "c2_mhd3d_weno5z_hlld_32": lambda: c2_params(32),
    "c2_mhd3d_weno5z_hlld_32_mixed": lambda: c2_params(32, precision="mixed"),
    "hd3d_tvd_hllc_8": lambda: _cfg(3, "hd", "tvd", "hllc"),
    "mhd2d_weno5z_hlld_16_rk2": lambda: _cfg(2, "mhd", "weno5z", "hlld", ta="rk2", n=16),
    "mhd3d_tvd_roe_4_ssprk4": lambda: _cfg(3, "mhd", "tvd", "roe", ta="ssprk(4,3)", n=4),
    "hd2d_iso_weno5z_hllc_16": lambda: _cfg(2, "hd", "weno5z", "hllc", n=16,
                                            equation_of_state="iso", csnd=0.8),
    "mhd3d_iso_tvd_hlld_8": lambda: _cfg(3, "mhd", "tvd", "hlld", equation_of_state="iso",
                                         csnd=1.0),
    "hd2d_visc_tvd_hllc_16": lambda: _cfg(2, "hd", "tvd", "hllc", n=16, viscosity=2e-3),
    "mhd3d_resist_weno5z_hlld_8": lambda: _cfg(3, "mhd", "weno5z", "hlld", viscosity=1e-3,
                                               resistivity=2e-3),
    "grav_mhd2d_tvd_hlld_16": lambda: grav_params(2, "mhd", "tvd"),
    "grav_hd3d_weno5z_hllc_8": lambda: grav_params(3, "hd", "weno5z"),
}


def _case(name):
    p = CASES[name]()
    if name.startswith("grav"):
        return p, grav_state(p)
    return p, initial_state(p) if name.startswith("c") else noisy(p, 17)


@pytest.mark.parametrize("name", [n for n in CASES if CASES[n]().precision == "fp64"])
def test_one_step_vs_oracle(name):
    p, u0 = _case(name)
    print(f"[case] one step {name}", flush=True)
    o = ol.OracleRun(p)
    o.set_state(u0)
    tr = o.run(1)
    with Solver(p) as s:
        s.upload(u0)
        dt, _ = s.advance()
        ug = s.download()
    assert dt == pytest.approx(tr[0, 0], rel=1e-13)
    assert relerr(ug, o.get_state()).max() <= 1e-12


def _shapes(nd):
    sizes = (64, 128, 256) if nd == 3 else (256,)
    return [[(256, z)] * 2 + [(wg, z)] * (nd - 2) for wg in sizes for z in (0, 1)]


@pytest.mark.parametrize("name", list(CASES))
def test_launch_shapes_agree(name):
    """Five steps in every launch shape: states, time steps and statistics
    bit for bit those of the default."""
    p, u0 = _case(name)
    print(f"[case] shapes {name}", flush=True)
    with Solver(p) as s:
        want = None
        for shape in [None] + _shapes(p.ndims):
            if shape:
                s.set_launch(shape)
            s.upload(u0)
            got = s.run(5), s.download(), s.statistics()
            want = want or got
            for a, b in zip(got, want):
                np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("graph", [False, True])
def test_stage_switch_changes_no_result(graph):
    """On, off and toggled between the steps, launched and replayed."""
    p = c2_params(32)
    u0 = initial_state(p)
    print(f"[case] stage switch graph={graph}", flush=True)
    with Solver(p) as s:
        s.upload(u0)
        want = s.run(6), s.download()
    for on in (lambda k: True, lambda k: k % 2 == 0):
        with Solver(p) as s:
            s.set_graph(graph)
            s.upload(u0)
            dts = []
            for k in range(6):
                s.set_stage_fusion(on(k))
                dts.append(s.run(1)[0])
            np.testing.assert_array_equal(dts, want[0])
            np.testing.assert_array_equal(s.download(), want[1])


def test_times_per_stage():
    """Three stages and the end of the step with the switch on, nine sweeps
    and the end with it off; the tuner needs the sweeps' own times."""
    with Solver(c2_params(32)) as s:
        s.upload(initial_state(c2_params(32)))
        s.set_stage_fusion(True)
        ms, kms = s.timed_run(2, per_kernel=True)
        print(f"[case] stage times {ms:.3f} ms, {kms}", flush=True)
        assert len(kms) == 4 and all(k > 0 for k in kms)
        with pytest.raises(AmunError, match="fused stage off"):
            s.autotune(1)
        s.set_stage_fusion(False)
        ms, kms = s.timed_run(2, per_kernel=True)
        assert len(kms) == 10 and all(k > 0 for k in kms)


@pytest.mark.parametrize("cfg", ["crmp5", "srmhd", "ncells12"])
def test_stage_switch_refused(cfg):
    if cfg == "crmp5":
        p = _cfg(2, "hd", "crmp5", "hllc", n=16)
        p.nghosts = 4
    elif cfg == "srmhd":
        p = _cfg(2, "srmhd", "tvd", "hll", n=16)
    else:
        p = _cfg(2, "hd", "tvd", "hllc", n=12)
    with Solver(p) as s:
        with pytest.raises(AmunError) as e:
            s.set_stage_fusion(True)
        assert e.value.code == 600
        s.set_stage_fusion(False)
