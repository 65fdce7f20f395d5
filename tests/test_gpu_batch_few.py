"""A few proposals are evaluated, and accepted, in one launch for all template
lengths; more of them, and a caller's own launch shapes, in one launch per
length.  Both have the same results: the same per-bin values (1e-12 of the
sums, whose terms may be added in another order), so the same state after an
accept to the rounding of r + h_old - h_new."""
import numpy as np
import pytest

from test_gpu_batch import make_cfg, new_plan

pytestmark = pytest.mark.gpu


def _plans(gl, cfg):
    E = len(cfg["p_chain"])
    few, own = new_plan(gl, cfg, E), new_plan(gl, cfg, E)
    tiles = own.tiles()
    own.set_tiles([(t[0], 1, t[2]) for t in tiles])  # not the default: one launch per length
    return few, own


def _rel(a, b):
    return float(((a - b).abs() / b.abs().clamp_min(1e-300)).max())


# the last windows hold templates of at most 512, 1024 and 4096 bins: both
# workgroup sizes, at the edges of the sizes they take
@pytest.mark.parametrize("windows,f_lo,f_hi", [((64, 600), 0.5e-3, 2e-3), ((1024, 1500), 3e-3, 9e-3),
                                               ((2048, 4096, 5001), 4e-3, 20e-3)])
def test_one_launch_equals_class_launches(gl, orc, windows, f_lo, f_hi):
    cfg = make_cfg(orc, seed=23, ngroup=5, ntemp=2, nprop=3, windows=windows, f_lo=f_lo, f_hi=f_hi)
    src = cfg["p_src"].copy()
    src[1] = -1  # left out
    few, own = _plans(gl, cfg)
    n, C = len(src), len(cfg["chain_group"])
    out = []
    for plan in (few, own):
        plan.set_proposals(cfg["p_chain"], src, cfg["p_params"])
        plan.logL.fill_(7.0)
        plan.snr.fill_(7.0)
        l, s = plan.eval(n)
        l, s = l.clone(), s.clone()
        assert float(l[1]) == 7.0 and float(s[1]) == 7.0
        idx = [int(np.flatnonzero((cfg["p_chain"] == c) & (src >= 0))[0]) for c in range(C)]
        plan.accept(idx)
        st = plan.state()
        l2, s2 = plan.eval(n)
        out.append((l, s, st, l2.clone(), s2.clone()))
        plan.refresh()
        st2 = plan.state()
        # the kept residual against one summed afresh
        assert np.max(np.abs(st2[0] - st[0]) / np.abs(st[0])) < 1e-9
    (l, s, st, l2, s2), (m, t, su, m2, t2) = out
    assert _rel(l, m) < 1e-12 and _rel(s, t) < 1e-12
    assert _rel(l2, m2) < 1e-12 and _rel(s2, t2) < 1e-12
    assert np.max(np.abs(st[0] - su[0]) / np.abs(su[0])) < 1e-12 and np.array_equal(st[1], su[1])
    few.close()
    own.close()


@pytest.mark.parametrize("concurrent", [True, False])
def test_line_between_them(gl, orc, concurrent):
    """1024 proposals go in one launch, 1025 in eight: 1020 and 1030 of the
    same plan agree on what they share, eager and captured."""
    cfg = make_cfg(orc, seed=29, ngroup=5, ntemp=2, nprop=103, windows=(512, 1024, 2048), f_lo=0.5e-3, f_hi=9e-3)
    E = len(cfg["p_chain"])
    assert E == 1030
    plan = new_plan(gl, cfg, E)
    plan.set_concurrent(concurrent)
    plan.set_proposals(cfg["p_chain"], cfg["p_src"], cfg["p_params"])
    a = [x[:1020].clone() for x in plan.eval(1020)]
    for graph in (False, True, True):
        b = [x.clone() for x in plan.eval(E, graph=graph)]
        c = [x[:1020].clone() for x in plan.eval(1020, graph=graph)]
        for i in range(2):
            assert _rel(a[i], b[i][:1020]) < 1e-12 and bool((a[i] == c[i]).all())
    plan.close()


def test_tuned_tiles_leave_a_few_proposals_in_one_launch(gl, orc, tmp_path):
    """An autotuner's tiles are for the class kernels of many proposals; with a
    caller's own every evaluation and accept runs those."""
    from glass_amd import autotune
    from glass_amd.batch import NCLASS, tile_candidates
    cfg = make_cfg(orc, seed=31, ngroup=5, ntemp=2, nprop=103, windows=(512, 1024, 2048), f_lo=0.5e-3, f_hi=9e-3)
    plan = new_plan(gl, cfg, 1030)
    plan.set_proposals(cfg["p_chain"], cfg["p_src"], cfg["p_params"])
    assert plan.one_launch(1) and plan.one_launch(1024) and not plan.one_launch(1025)
    ref = [x.clone() for x in plan.eval(500)]
    other = [tile_candidates(k)[1] for k in range(NCLASS)]
    assert other != plan.tiles()
    plan.set_tiles(other)
    assert not plan.one_launch(1) and plan.tiles() == other
    plan.set_tiles(other, tuned=True)
    assert plan.one_launch(1024) and plan.tiles() == other
    for got in (plan.eval(500), plan.eval(500, graph=True)):
        assert all(bool((a == b).all()) for a, b in zip(got, ref))
    cache = str(tmp_path / "tiles.json")
    for _ in range(2):  # measured, then from the cache
        plan.set_tiles(other)
        tiles, _, cached = autotune.tune(plan, 1030, cache=cache, reps=1)
        assert plan.tiles() == tiles and plan.one_launch(1024) and not plan.one_launch(1025)
    assert cached
    plan.profile(True)
    assert not plan.one_launch(1)
    plan.profile(False)
    plan.close()


@pytest.mark.parametrize("k", [0, 1, 6, 7])
def test_autotuner_times_a_launch_once(gl, orc, k):
    """Where the default grid strides, gmul 0 and 4 are the same launch: the
    tuner keeps gmul 0 for it."""
    cfg = make_cfg(orc, seed=37, ngroup=6, ntemp=2, nprop=4, windows=(64, 4096, 6000), f_lo=0.5e-3, f_hi=20e-3)
    plan = new_plan(gl, cfg, len(cfg["p_chain"]))
    plan.set_proposals(cfg["p_chain"], cfg["p_src"], cfg["p_params"])
    for _ in range(4):
        tiles, _ = plan.autotune(len(cfg["p_chain"]), reps=1)
        assert tiles[k][1] != 4
    plan.close()


def test_accepting_a_left_out_item_changes_nothing(gl, orc):
    """An accepted item without a source (negative index) is left out: in one
    launch, and in the launches per length of more than 1024."""
    cfg = make_cfg(orc, seed=41, ngroup=103, ntemp=10, nprop=1, windows=(64, 100, 256), f_lo=0.5e-3, f_hi=2e-3)
    n = len(cfg["p_chain"])
    assert n == 1030 and len(set(cfg["p_chain"])) == n
    src = cfg["p_src"].copy()
    src[[0, 511, 1029]] = -1
    out = []
    for parts in ([n], [515, n - 515]):
        plan = new_plan(gl, cfg, n)
        plan.set_proposals(cfg["p_chain"], src, cfg["p_params"])
        before = plan.state()
        plan.eval(n)
        a = 0
        for m in parts:
            plan.accept(np.arange(a, a + m))
            a += m
        after = plan.state()
        same = np.all(before[1] == after[1], axis=(1, 2)) & (before[0] == after[0])
        assert sorted(np.flatnonzero(same)) == sorted(cfg["p_chain"][[0, 511, 1029]])
        plan.refresh()
        fresh = plan.state()
        assert np.max(np.abs(fresh[0] / after[0] - 1)) < 1e-9
        out.append(after)
        plan.close()
    assert np.max(np.abs(out[0][0] / out[1][0] - 1)) < 1e-12 and np.array_equal(out[0][1], out[1][1])
