"""The EOS's power x**GAMMA over and beyond the range of its short form,
bit-identical to the float64 power rounded once: arguments from 2^-18 to 2^5
(the short form takes 2^-16 .. 2^4), zero and negative theta."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_pressure_is_the_rounded_power():
    import torch
    from arwen_amd import cases as C
    from arwen_amd import dycore
    from arwen_amd.state import DomainState
    f32 = np.float32
    case = C.ensemble_member(200, 120, 40, seed=3)
    g = DomainState.from_host(case)
    rng = np.random.default_rng(11)
    thb = g.thb.cpu().numpy().astype(f32)[:, None, None]
    th = np.exp2(rng.uniform(-10.0, 13.2, tuple(g.thp.shape)))
    th[0, 0, :2] = (0.0, -1.0)
    g.thp.copy_(torch.as_tensor((th - thb).astype(f32)))
    thp = g.thp.cpu().numpy()
    dycore.update_diagnostics(g)
    alt, p = g.alt.cpu().numpy(), g.p.cpu().numpy()
    x = (f32(287.0) * (thb + thp)) / (f32(1.0e5) * alt)
    with np.errstate(invalid="ignore"):
        want = f32(1.0e5) * np.power(x.astype(np.float64),
                                     np.float64(f32(1.4))).astype(f32)
    assert x.min() < 0.0 and x[x > 0.0].min() < 2.0 ** -16 and x.max() > 16.0
    assert np.array_equal(p, want, equal_nan=True), \
        np.flatnonzero(~((p == want) | (np.isnan(p) & np.isnan(want))))[:8]


def test_pressure_over_whole_binades():
    """2^23 arguments in each binade the short form takes, near every float
    in it (no base theta, so theta' sets the argument to a rounding or two)."""
    import torch
    from arwen_amd import cases as C
    from arwen_amd import dycore
    from arwen_amd.state import DomainState
    g = DomainState.from_host(C.ensemble_member(1024, 1024, 8, seed=3))
    g.thb.zero_()
    dycore.update_diagnostics(g)
    p0alt = (g.alt.double() * 1.0e5).float().double()
    m = torch.arange(1 << 23, device=g.alt.device).reshape(g.alt.shape)
    gamma = float(np.float32(1.4))
    for e in range(-16, 5):
        target = (1.0 + m.double() * 2.0 ** -23) * 2.0 ** e
        th = (target * p0alt / 287.0).float()
        g.thp.copy_(th)
        dycore.update_diagnostics(g)
        # a double quotient of floats, rounded, is the float quotient
        x = ((th.double() * 287.0).float().double() / p0alt).float()
        want = (torch.pow(x.double(), gamma).float().double() * 1.0e5).float()
        assert torch.equal(g.p, want), (e, int((g.p != want).sum()))
        d = torch.unique(x).numel()
        print(f"2^{e}: {d} arguments", flush=True)
        assert d > 1 << 22
