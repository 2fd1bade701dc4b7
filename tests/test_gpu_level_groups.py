"""The step's kernels where their launches change shape: one-column and
ragged domains, the fewest levels, remainders of the level groups and of
the 16- and 64-column tiles, more levels than a tile's LDS holds, and
duplicate faces that differ from face 0.  One step, bit-identical to the
float32 oracle; the FP64 build to the float64 oracle but for its pow, whose
last bit may differ."""
import numpy as np
import pytest

from helpers import DIAG, PROG, compare, oracle_and_gpu
from oracle import dycore_np as O

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 3), (5, 3, 3), (64, 4, 4), (65, 5, 7), (20, 3, 5), (17, 2, 9),
         (33, 3, 36), (130, 1, 33),
         (63, 9, 50), (200, 67, 17), (257, 60, 65), (3, 70, 130),
         (17, 9, 128), (131, 127, 9), (2, 3, 1030)]


def _noisy(case, seed=5):
    """w noise, and duplicate faces of their own (the step carries them
    separately)."""
    rng = np.random.default_rng(seed)
    f = case.fields
    f["w"][1:-1] = 0.2 * rng.standard_normal(f["w"][1:-1].shape)
    f["u"][..., -1] += 0.05
    f["v"][:, -1] -= 0.05
    return case


def _case(kind, nx, ny, nz):
    from arwen_amd import cases as C
    if kind in ("flat", "precision", "fp64"):
        return _noisy(C.ensemble_member(nx, ny, nz, seed=3))
    if kind == "terrain":
        return _noisy(C.stratified_hill(nx=nx, ny=ny, nz=nz, dx=3000.0,
                                        dt=12.0, radius=20000.0,
                                        hill=300.0))
    if kind == "moist":
        return _noisy(C.mixed_phase(10, nx=nx, ny=ny, nz=nz))
    case = _noisy(C.ensemble_member(nx, ny, nz, seed=3))
    case.cfg = case.cfg.with_(khdif=75.0, kvdif=75.0, time_step_sound=6)
    return case


@pytest.mark.parametrize("kind", ["flat", "terrain", "diffusion", "moist"])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_step_is_bit_identical_at_the_edges_of_the_launch_shapes(kind, size):
    from arwen_amd import dycore
    case = _case(kind, *size)
    o, g = oracle_and_gpu(case)
    names = PROG + DIAG
    if kind == "moist":
        import torch
        q = ("qv", "qc", "qr") + o.extra
        names = names + q
        for n in q + ("h_diabatic",):
            getattr(g, n).copy_(torch.as_tensor(getattr(o, n)))
    O.step(o, case.cfg)
    dycore.step(g, case.cfg)
    for n, (err, same) in compare(o, g, names).items():
        assert np.all(np.isfinite(getattr(o, n))), n
        assert same == 1.0, f"{n}: rel {err:.3e}, {same:.6f} identical"


# 768 workgroups of 64 x 4 columns and 975, 1046: the duplicate faces in a
# launch of their own, the levels in one group and in several
@pytest.mark.parametrize("kind", ["flat", "terrain", "diffusion"])
@pytest.mark.parametrize("size", [(3, 3070, 5), (2, 3900, 5), (65, 2091, 4)],
                         ids=lambda s: "x".join(map(str, s)))
def test_duplicate_faces_launched_apart(kind, size):
    from arwen_amd import dycore
    case = _case(kind, *size)
    o, g = oracle_and_gpu(case)
    O.step(o, case.cfg)
    dycore.step(g, case.cfg)
    for n, (err, same) in compare(o, g, PROG + DIAG).items():
        assert np.all(np.isfinite(getattr(o, n))), n
        assert same == 1.0, f"{n}: rel {err:.3e}, {same:.6f} identical"


@pytest.mark.parametrize("size", [(5, 3, 3), (17, 9, 128), (131, 127, 9)],
                         ids=lambda s: "x".join(map(str, s)))
def test_precision_form_is_bit_identical_there(size):
    from arwen_amd import dycore
    case = _case("precision", *size)
    case.cfg = case.cfg.with_(precision_form=True)
    o, g = oracle_and_gpu(case)
    O.step(o, case.cfg)
    dycore.step(g, case.cfg)
    for n, (err, same) in compare(o, g, PROG + DIAG).items():
        assert same == 1.0, f"{n}: rel {err:.3e}, {same:.6f} identical"


@pytest.mark.parametrize("size", [(5, 3, 3), (17, 9, 128), (131, 127, 9)],
                         ids=lambda s: "x".join(map(str, s)))
def test_fp64_build_agrees_there(size):
    import torch
    from arwen_amd import dycore
    from arwen_amd.state import DomainState
    case = _case("fp64", *size)
    o = O.from_case(case, np.float64)
    g = DomainState.from_host(case, dtype=torch.float64)
    O.step(o, case.cfg)
    dycore.step(g, case.cfg)
    # pow's last bit, 2e-16 of a pressure whose differences the step takes
    for n, (err, _) in compare(o, g, PROG + DIAG).items():
        assert err < 1e-9, f"{n}: rel {err:.3e}"


# more levels than a column tile takes: k_column, whose forms these few columns
# would otherwise not reach
@pytest.mark.parametrize("kind", ["terrain", "moist_cq"])
def test_column_march_options_are_bit_identical(kind):
    """The precision form over terrain, and moist_cq."""
    from arwen_amd import dycore
    if kind == "terrain":
        case = _case(kind, 3, 70, 130)
        case.cfg = case.cfg.with_(precision_form=True)
    else:
        case = _case("moist", 3, 70, 130)
        case.cfg = case.cfg.with_(moist_cq=True)
    o, g = oracle_and_gpu(case)
    names = PROG + DIAG
    if kind == "moist_cq":
        import torch
        q = ("qv", "qc", "qr") + o.extra
        names = names + q
        for n in q + ("h_diabatic",):
            getattr(g, n).copy_(torch.as_tensor(getattr(o, n)))
    O.step(o, case.cfg)
    dycore.step(g, case.cfg)
    for n, (err, same) in compare(o, g, names).items():
        assert np.all(np.isfinite(getattr(o, n))), n
        assert same == 1.0, f"{n}: rel {err:.3e}, {same:.6f} identical"


def test_column_march_precision_form_is_bit_identical():
    test_precision_form_is_bit_identical_there((3, 70, 130))


@pytest.mark.parametrize("kind", ["fp64", "terrain"])
def test_column_march_fp64_agrees(kind):
    import torch
    from arwen_amd import dycore
    from arwen_amd.state import DomainState
    case = _case(kind, 3, 70, 130)
    o = O.from_case(case, np.float64)
    g = DomainState.from_host(case, dtype=torch.float64)
    O.step(o, case.cfg)
    dycore.step(g, case.cfg)
    # as above: pow's last bit
    for n, (err, _) in compare(o, g, PROG + DIAG).items():
        assert err < 1e-9, f"{n}: rel {err:.3e}"


def test_omega_in_wide_tiles_parks_more_levels_than_its_lds_holds():
    """Above 16384 columns Omega's tile is 64 columns wide; its LDS holds 256
    levels of them."""
    from arwen_amd import dycore
    case = _case("flat", 129, 128, 257)
    o, g = oracle_and_gpu(case)
    O.step(o, case.cfg)
    dycore.step(g, case.cfg)
    for n, (err, same) in compare(o, g, PROG + DIAG).items():
        assert same == 1.0, f"{n}: rel {err:.3e}, {same:.6f} identical"
