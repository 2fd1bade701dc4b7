"""GPU parity of the step on mixed-phase states: every species of WSM6,
Thompson, Morrison, NSSL and aerosol-aware Thompson transported with the
substep-averaged fluxes (positive definite on the final stage), the ice
and hail masses loading the buoyancy, and the retained microphysics
heating h_diabatic added to every stage's theta tendency and removed by
the final stage.  Bit-identical to the float32 oracle after whole steps;
the FP64 build agrees with the float64 oracle to a stated tolerance."""
import numpy as np
import pytest
import torch

from arwen_amd import cases
from arwen_amd.config import EXTRA_SPECIES
from oracle import dycore_np as O
from tests.helpers import compare, oracle_and_gpu

pytestmark = pytest.mark.gpu

BASE = ("u", "v", "w", "thp", "php", "mup", "p", "al", "alt", "qv", "qc",
        "qr")

#: relative (normwise, per field) FP64 agreement after two steps
FP64_TOL = 1e-9


@pytest.mark.parametrize("mp", [6, 8, 10, 18, 28])
def test_mixed_phase_step_matches_oracle_bitwise(mp):
    from arwen_amd import dycore
    case = cases.mixed_phase(mp, nx=24, ny=16, nz=20)
    o, g = oracle_and_gpu(case)
    assert g.extra_species == EXTRA_SPECIES[mp]
    print(f"mixed-phase step parity mp={mp}", flush=True)
    for _ in range(2):
        O.step(o, case.cfg)
        dycore.step(g, case.cfg)
    res = compare(o, g, BASE + EXTRA_SPECIES[mp])
    bad = {k: v for k, v in res.items() if v[1] < 1.0}
    assert not bad, bad
    for q in EXTRA_SPECIES[mp]:
        assert float(getattr(g, q).min()) >= 0.0, q


def test_heating_enters_the_device_step():
    """The same state with and without h_diabatic differs on the device
    exactly as in the oracle (both bitwise), so the heating path is live."""
    from arwen_amd import dycore
    case = cases.mixed_phase(6, nx=24, ny=16, nz=20)
    cold = cases.mixed_phase(6, nx=24, ny=16, nz=20)
    cold.fields["h_diabatic"][...] = 0.0
    o1, g1 = oracle_and_gpu(case)
    o0, g0 = oracle_and_gpu(cold)
    print("heated vs unheated step on the device", flush=True)
    for o, g in ((o1, g1), (o0, g0)):
        O.step(o, case.cfg)
        dycore.step(g, case.cfg)
    d_dev = (g1.thp - g0.thp).cpu().numpy()
    d_ora = o1.thp - o0.thp
    assert np.abs(d_ora).max() > 0.0
    np.testing.assert_array_equal(d_dev, d_ora)


def test_fp64_mixed_phase_step_matches_fp64_oracle():
    from arwen_amd import dycore
    from arwen_amd.state import DomainState
    case = cases.mixed_phase(18, nx=24, ny=16, nz=20)
    o = O.from_case(case, np.float64)
    g = DomainState.from_host(case, dtype=torch.float64)
    print("fp64 mixed-phase parity mp=18", flush=True)
    for _ in range(2):
        O.step(o, case.cfg)
        dycore.step(g, case.cfg)
    rel = {}
    for n in BASE + EXTRA_SPECIES[18]:
        a = getattr(g, n).detach().cpu().numpy()
        b = getattr(o, n)
        rel[n] = float(np.max(np.abs(a - b))
                       / max(np.max(np.abs(b)), 1e-300))
    assert max(rel.values()) < FP64_TOL, rel


def test_microphysics_slot_runs_after_the_dynamics():
    """The reference's post-RK3 microphysics slot (dycore.py:2491-2502):
    a supplied scheme runs once with cfg.dt after the dynamics, then the
    EOS is refreshed from its output."""
    from arwen_amd import dycore
    from arwen_amd.state import DomainState
    case = cases.mixed_phase(10, nx=24, ny=16, nz=20)
    calls = []

    def scheme(state, cfg, dt, refl_10cm_due=False):
        calls.append((dt, refl_10cm_due))
        state.thp.add_(0.25)
        state.h_diabatic.zero_()

    plain = DomainState.from_host(case)
    dycore.step(plain, case.cfg)
    g = DomainState.from_host(case)
    print("microphysics slot", flush=True)
    dycore.step(g, case.cfg, microphysics=scheme)
    assert calls == [(case.cfg.dt, False)]
    assert torch.equal(g.thp, plain.thp + 0.25)
    assert float(g.h_diabatic.abs().max()) == 0.0
    p = g.p.clone()
    dycore.update_diagnostics(g)
    assert torch.equal(p, g.p)
    assert not torch.equal(g.p, plain.p)


@pytest.mark.parametrize("opt", [1, 0])
def test_column_march_scalars_match_oracle_bitwise(opt):
    """The step's unlimited scalar transport is a column march
    (k_scalar_cols); from 128 x 128 columns on so is the final stage's limiter
    (k_pd_scale_cols / k_pd_apply_cols), below it one thread per point.  One
    WSM6 step at 512 x 512 columns against the oracle, with and without the PD
    limiter."""
    from arwen_amd import dycore
    case = cases.mixed_phase(6, nx=512, ny=512, nz=6, dx=3000.0,
                             moist_adv_opt=opt)
    o, g = oracle_and_gpu(case)
    print(f"column-march scalars 512x512x6 moist_adv_opt={opt}", flush=True)
    O.step(o, case.cfg)
    dycore.step(g, case.cfg)
    res = compare(o, g, BASE + EXTRA_SPECIES[6])
    bad = {k: v for k, v in res.items() if v[1] < 1.0}
    assert not bad, bad
