"""GPU checks of the batched ensemble (arw_ensemble_*): members of uneven
extents advanced by one launch per pass agree bit for bit with stepping
each member alone through arw_step -- eagerly, through a replayed HIP
graph (with eager work between replays), with several member groups and
reordered work tables, on flat and terrain bases, in FP32 and FP64."""
import numpy as np
import pytest
import torch

from arwen_amd import cases
from arwen_amd.ensemble import STATE_ARRAYS

pytestmark = pytest.mark.gpu

SHAPES = [(24, 20, 12), (37, 16, 10), (16, 33, 14), (50, 9, 11), (8, 8, 16)]


def _members(dtype=torch.float32, terrain=False):
    from arwen_amd.state import DomainState
    out = []
    for i, (nx, ny, nz) in enumerate(SHAPES):
        if terrain:
            case = cases.stratified_hill(nx=nx, ny=ny, nz=nz, seed=100 + i,
                                         radius=20000.0)
        else:
            case = cases.ensemble_member(nx, ny, nz, seed=100 + i)
        out.append((case, DomainState.from_host(case, dtype=dtype)))
    return out


def _pair(dtype=torch.float32, terrain=False):
    a = _members(dtype, terrain)
    b = _members(dtype, terrain)
    return a[0][0].cfg, [s for _, s in a], [s for _, s in b]


def _assert_same(sa, sb):
    for i, (x, y) in enumerate(zip(sa, sb)):
        for n in STATE_ARRAYS:
            assert torch.equal(getattr(x, n), getattr(y, n)), (i, n)


@pytest.mark.parametrize("terrain", [False, True])
def test_eager_ensemble_matches_member_steps_bitwise(terrain):
    from arwen_amd import dycore
    from arwen_amd.ensemble import Ensemble
    cfg, seq, ens_states = _pair(terrain=terrain)
    print(f"ensemble eager terrain={terrain}", flush=True)
    for st in seq:
        dycore.run_steps(st, st.cfg, 3)
    with Ensemble(ens_states, cfg) as ens:
        ens.step(3)
    torch.cuda.synchronize()
    _assert_same(seq, ens_states)


# (these few columns are solved in tiles of 16 whatever col_tile says;
# test_column_march_ensemble_matches_member_steps_bitwise reaches 64 and 128)
@pytest.mark.parametrize("groups,order,join,tile", [
    (1, None, 0, 256), (2, "largest_first", 0, 128),
    (3, "smallest_first", 1, 64)])
def test_graph_replays_match_member_steps_bitwise(groups, order, join, tile):
    from arwen_amd import dycore
    from arwen_amd.ensemble import Ensemble, member_orders
    cfg, seq, ens_states = _pair()
    print(f"ensemble graph groups={groups} order={order} join={join} "
          f"col_tile={tile}", flush=True)
    ordl = member_orders(ens_states)[order] if order else None
    with Ensemble(ens_states, cfg, order=ordl, groups=groups,
                  join_every=join, col_tile=tile) as ens:
        ens.capture(2)
        for rep in range(3):
            ens.launch()
            for st in seq:
                dycore.run_steps(st, st.cfg, 2)
            # eager work of the program's own between replays
            _ = [float(st.u.abs().max()) for st in seq]
            torch.cuda.synchronize()
            _assert_same(seq, ens_states)


def test_fp64_ensemble_matches_member_steps_bitwise():
    from arwen_amd import dycore
    from arwen_amd.ensemble import Ensemble
    cfg, seq, ens_states = _pair(dtype=torch.float64)
    print("ensemble fp64", flush=True)
    for st in seq:
        dycore.run_steps(st, st.cfg, 2)
    with Ensemble(ens_states, cfg, groups=2) as ens:
        ens.capture(2)
        ens.launch()
    torch.cuda.synchronize()
    _assert_same(seq, ens_states)


def test_autotune_leaves_state_and_picks_a_layout():
    from arwen_amd import ensemble as E
    cfg, _, states = _pair()
    print("ensemble autotune", flush=True)
    before = E.save_state(states)
    res = E.autotune(states, cfg, steps=1, reps=1, groups=(1, 2))
    torch.cuda.synchronize()
    for st, (sv, el) in zip(states, before):
        assert st.elapsed_seconds == el
        for n, t in sv.items():
            assert torch.equal(getattr(st, n), t), n
    assert res["groups"] in (1, 2) and sorted(res["order"]) == list(range(5))
    assert res["join_every"] in (1, 5)      # 0 measured as every `steps`
    assert res["col_tile"] in (64, 128, 256)
    # 3 orders, then 3 joins x 2 groups, then 2 more column tiles
    assert len(res["trials"]) == 8


def test_ensemble_rejects_bad_members():
    from arwen_amd.ensemble import Ensemble
    from arwen_amd.state import DomainState
    cfg, _, states = _pair()
    print("ensemble argument checks", flush=True)
    other = cases.ensemble_member(12, 12, 8, seed=1, dt=9.0)
    with pytest.raises(ValueError):
        Ensemble(states + [DomainState.from_host(other)], cfg)
    with pytest.raises(ValueError):
        Ensemble(states, cfg, order=[0, 0, 1, 2, 3])
    from arwen_amd import _lib
    with pytest.raises(_lib.ArwenError):
        Ensemble(states, cfg, groups=9)
    with pytest.raises(_lib.ArwenError, match="col_tile"):
        Ensemble(states, cfg, col_tile=96)


@pytest.mark.parametrize("terrain", [False, True])
def test_precision_form_ensemble_matches_member_steps_bitwise(terrain):
    """The precision form (perturbation EOS, p' array, FP64 tridiagonal)
    through the batched launches equals each member's own precision-form
    step."""
    from arwen_amd import dycore
    from arwen_amd.ensemble import Ensemble
    cfg, seq, ens_states = _pair(terrain=terrain)
    cfg = cfg.with_(precision_form=True)
    for st in seq + ens_states:
        st.cfg = st.cfg.with_(precision_form=True)
    print(f"ensemble precision form terrain={terrain}", flush=True)
    for st in seq:
        dycore.run_steps(st, st.cfg, 2)
    with Ensemble(ens_states, cfg, groups=2) as ens:
        ens.step(2)
    torch.cuda.synchronize()
    _assert_same(seq, ens_states)


@pytest.mark.parametrize("tile", [64, 128, 256])
@pytest.mark.parametrize("form", ["flat", "terrain", "precision",
                                  "precision terrain", "fp64", "fp64 terrain"])
def test_column_march_ensemble_matches_member_steps_bitwise(form, tile):
    """A member of 130 levels (flat: and one of 260, more than the batched
    Omega's LDS holds) is more than a column tile takes, so the ensemble's
    column solve is k_column with col_tile columns a workgroup; the members
    stepped alone take the column tile but for the tall ones."""
    from arwen_amd import dycore
    from arwen_amd.ensemble import Ensemble
    from arwen_amd.state import DomainState
    shapes = SHAPES[:3] + [(21, 13, 130)] + [(9, 7, 260)] * (form == "flat")
    dtype = torch.float64 if "fp64" in form else torch.float32
    print(f"ensemble column march {form} col_tile={tile}", flush=True)

    def states():
        out = []
        for i, (nx, ny, nz) in enumerate(shapes):
            case = (cases.stratified_hill(nx=nx, ny=ny, nz=nz, seed=100 + i,
                                          radius=20000.0)
                    if "terrain" in form
                    else cases.ensemble_member(nx, ny, nz, seed=100 + i))
            st = DomainState.from_host(case, dtype=dtype)
            st.cfg = st.cfg.with_(precision_form="precision" in form)
            out.append(st)
        return out

    seq, ens_states = states(), states()
    for st in seq:
        dycore.run_steps(st, st.cfg, 2)
    with Ensemble(ens_states, seq[0].cfg, col_tile=tile) as ens:
        ens.step(2)
    torch.cuda.synchronize()
    _assert_same(seq, ens_states)
    assert all(bool(torch.isfinite(st.p).all()) for st in seq)


@pytest.mark.parametrize("members,groups,tile", [(2, 1, 16), (2, 2, 16),
                                                 (4, 1, 128), (4, 2, 128)])
def test_column_tile_counts_all_groups_columns(members, groups, tile):
    """A captured graph's groups run side by side, so the column solve is
    chosen by the columns of all of them: 39 000 take 16-column tiles, 78 000
    in two groups take k_column like 78 000 in one."""
    from arwen_amd import dycore
    from arwen_amd.ensemble import Ensemble
    from arwen_amd.state import DomainState
    states = [[DomainState.from_host(cases.ensemble_member(150, 130, 8,
                                                           seed=7 + i))
               for i in range(members)] for _ in range(2)]
    print(f"ensemble column tile members={members} groups={groups}",
          flush=True)
    for st in states[0]:
        dycore.run_steps(st, st.cfg, 1)
    with Ensemble(states[1], states[1][0].cfg, groups=groups,
                  col_tile=128) as ens:
        assert ens.column_tile == tile
        ens.capture(1)
        ens.launch()
    torch.cuda.synchronize()
    _assert_same(*states)


def test_short_members_in_a_tall_batch():
    """Members of the fewest levels beside one of 64: level groups without
    levels in their workgroups."""
    from arwen_amd import dycore
    from arwen_amd.ensemble import Ensemble
    from arwen_amd.state import DomainState
    states = [[DomainState.from_host(cases.ensemble_member(*sh, seed=3))
               for sh in ((5, 3, 3), (64, 4, 4), (20, 9, 5), (33, 7, 64))]
              for _ in range(2)]
    print("ensemble short members", flush=True)
    for st in states[0]:
        dycore.run_steps(st, st.cfg, 2)
    with Ensemble(states[1], states[1][0].cfg) as ens:
        assert ens.column_tile == 16
        ens.step(2)
    torch.cuda.synchronize()
    _assert_same(*states)


@pytest.mark.parametrize("tall", [False, True])
def test_autotune_times_column_tiles_only_where_they_differ(tall, monkeypatch):
    """Few columns take 16-column tiles whatever col_tile says: the tuner
    neither times those layouts again nor picks one of them by noise."""
    from arwen_amd import ensemble as E
    from arwen_amd.state import DomainState
    shapes = SHAPES[:2] + [(11, 10, 130 if tall else 13)]
    states = [DomainState.from_host(cases.ensemble_member(*sh, seed=100))
              for sh in shapes]
    timed, time_layout = [], E._time_layout
    monkeypatch.setattr(E, "_time_layout", lambda *a: (
        timed.append(a[-1]), time_layout(*a))[1])
    print(f"ensemble autotune tall={tall}", flush=True)
    res = E.autotune(states, states[0].cfg, steps=1, reps=1, groups=(1,))
    assert [t for t in timed if t != 256] == ([128, 64] if tall else [])
    assert [t["col_tile"] for t in res["trials"]][-2:] == [128, 64]
    if not tall:
        assert res["col_tile"] == 256
