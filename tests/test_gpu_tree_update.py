"""The dynamic tree update on the device (tree kicks inside
tdv_kick_halfstep, tdv_tree_update_drift) against oracle/tree_update.py,
Tandav's tree_update.c restated: every node's Dp, UPDATED bit and CoM and
every top node's float Dp, Level sign and CoM bit for bit, for an active
subset spread over time bins; and the identity Dp Mass = sum of the
node's kicked particles' m dt a."""
import numpy as np
import pytest

from oracle import tree_update as U
from tandav_amd import Engine, engine, ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic", [True, False])
def test_tree_kicks_and_drift_match_oracle(periodic):
    if periodic:
        pos, vel, m = ics.zeldovich_box(24, seed=7)
        soft = 1 / 960.
    else:
        pos, vel, m = ics.hernquist_sphere(20000, seed=2)
        soft = 0.01
    n = len(m)
    e = Engine(periodic=periodic, softening=soft, alpha_rel=0.005)
    e.set_particles(pos, m, vel=vel)
    e.setup_domain()
    e.domain_decomposition()
    e.compute_acceleration(True)
    g = np.random.Generator(np.random.Philox(17))
    bins = g.integers(1, 9, n).astype(np.int32)
    e.make_active_list(31, time_bin=bins)
    e.set_timeline(engine.timeline(False, 0.0, 1.0))
    it = (g.integers(0, 1 << 14, n) << 9).astype(np.uint32)
    e.set_integer_times(it, it)
    act = np.sort(g.choice(n, n // 4, replace=False)).astype(np.int32)
    e.set_active(act)
    tree0, top0 = e.tree(), e.top_nodes()
    st = e.get("mass", "acc", "tree_parent", "time_bin")
    e.kick_halfstep(update_tree=True)
    _, itk = e.integer_times()
    step = (np.left_shift(np.uint32(1), st["time_bin"].astype(np.uint32))
            >> np.uint32(1)).astype(np.uint32)
    t0 = it.astype(np.float64) / 2.0 ** 31
    t1 = (it + step).astype(np.float64) / 2.0 ** 31
    dt = t1 - t0                                   # Particle_Kick_Step
    want_tree, want_top = U.kicks(tree0, top0, st["mass"], st["acc"], dt,
                                  st["tree_parent"], act)
    tree1, top1 = e.tree(), e.top_nodes()
    for f in ("Bitfield", "Dp", "CoM"):
        np.testing.assert_array_equal(tree1[f], want_tree[f], err_msg=f)
    for f in ("Level", "Dp", "CoM"):
        np.testing.assert_array_equal(top1[f], want_top[f], err_msg=f)
    upd = (tree1["Bitfield"] >> 11) & 1 == 1
    assert upd.sum() > 10
    # Dp Mass = the momentum the node's kicked particles took
    mdt_a = (st["mass"] * dt)[:, None] * st["acc"]
    on = np.zeros(n, bool)
    on[act] = True
    for j in np.flatnonzero(upd)[:200]:
        first = _first_particle(tree1, j)
        sel = np.arange(first, first + tree1["Npart"][j])
        want = (mdt_a[sel] * on[sel, None]).sum(0)
        np.testing.assert_allclose(tree1["Dp"][j] * tree1["Mass"][j], want,
                                   rtol=1e-11, atol=1e-13 * np.abs(want).max())
    e.tree_update_drift(0.01)
    want_tree, want_top = U.drift(want_tree, want_top, 0.01)
    tree2, top2 = e.tree(), e.top_nodes()
    for f in ("Bitfield", "Dp", "CoM"):
        np.testing.assert_array_equal(tree2[f], want_tree[f], err_msg=f)
    for f in ("Level", "Dp", "CoM"):
        np.testing.assert_array_equal(top2[f], want_top[f], err_msg=f)
    assert not ((tree2["Bitfield"] >> 11) & 1).any()


def _first_particle(tree, j):
    """A node's first particle: the first bundle at or below it in the
    depth-first array."""
    k = j
    while tree["DNext"][k] >= 0:
        k += 1
    return -int(tree["DNext"][k]) - 1


@pytest.mark.parametrize("n", [200, 4096 + 63, 30001])
def test_tree_kicks_of_long_runs_match_oracle(n):
    """Every particle active: runs of the active list below, at and far
    beyond a wavefront, with a remainder."""
    pos, vel, m = ics.hernquist_sphere(n, seed=5)
    e = Engine(periodic=False, softening=0.01, alpha_rel=0.005)
    e.set_particles(pos, m, vel=vel)
    e.setup_domain()
    e.domain_decomposition()
    e.compute_acceleration(True)
    e.make_active_list(31, time_bin=np.full(n, 9, np.int32))
    e.set_timeline(engine.timeline(False, 0.0, 1.0))
    st = e.get("mass", "acc", "tree_parent")
    dt = np.full(n, 2.0 ** 8 / 2.0 ** 31)
    tree, top = e.tree(), e.top_nodes()
    for _ in range(2):                   # the second on top of the first
        e.kick_halfstep(update_tree=True)
        tree, top = U.kicks(tree, top, st["mass"], st["acc"], dt,
                            st["tree_parent"], np.arange(n, dtype=np.int32))
        got, gtop = e.tree(), e.top_nodes()
        for f in ("Bitfield", "Dp", "CoM"):
            np.testing.assert_array_equal(got[f], tree[f], err_msg=f)
        for f in ("Level", "Dp", "CoM"):
            np.testing.assert_array_equal(gtop[f], top[f], err_msg=f)


def _quotients(g, n):
    """Runs of the kicks' addends that the sums in whole units have to stop
    at: ties of a float and of a double sum, sums about zero whose binade
    changes with every term, terms from 2^-1060 to 2^60 of both signs."""
    half = g.integers(-9, 10, n) * 1.0
    about = g.normal(0.0, 1.0, n)
    about[1::2] = -about[::2][:n // 2] * (1 + g.integers(-3, 4, n // 2)
                                          * 2.0 ** -52)
    wide = g.choice([-1.0, 1.0], n) * 2.0 ** g.uniform(-60, 60, n)
    wide[g.integers(0, n, n // 16)] = 2.0 ** -1060
    wide[g.integers(0, n, n // 16)] = 0.0
    ties32, ties64 = half * 2.0 ** -24, half * 2.0 ** -53
    for t in (ties32, ties64):
        t[0] = 1.5                       # the sums' binade is [1, 2) then
        t[n // 2] = -1.5
        t[n // 2 + 1] = -0.75
    return [ties32, ties64, about, wide]


def test_tree_kicks_at_ties_and_sign_changes_match_oracle():
    """Nodes of 4096 and 2048 particles of mass 1 in steps of powers of two:
    the addends are the chosen ones exactly, in the top nodes' float sums and
    in the nodes' double sums; three kicks on top of one another."""
    g = np.random.Generator(np.random.Philox(23))
    pos = np.concatenate([
        g.uniform(0.0998, 0.1012, (4096, 3)),        # one cell of level 9
        g.uniform(0.6, 0.62, (2048, 3)),
        g.uniform(0.0, 1.0, (300, 3)) * (0.2, 0.2, 0.2) + (0.0, 0.0, 0.78),
        g.uniform(0.3, 0.45, (40, 3))])              # no subtree
    n = len(pos)
    e = Engine(periodic=True, softening=1e-4)
    e.set_particles(pos, np.ones(n))
    e.setup_domain()
    e.domain_decomposition()
    e.tree_build()
    tree, top = e.tree(), e.top_nodes()
    assert {4096, 2048, 40} <= set(top["Npart"].tolist())
    assert (tree["Npart"] == 4096).sum() >= 6
    e.make_active_list(31, time_bin=np.full(n, 9, np.int32))
    e.set_timeline(engine.timeline(False, 0.0, 1.0))
    dt = np.full(n, 2.0 ** 8 / 2.0 ** 31)
    st = e.get("mass", "tree_parent", "pos")
    for kick in range(3):
        acc = np.empty((n, 3))
        for t in top:
            f, c = int(t["First_Part"]), int(t["Npart"])
            q = _quotients(g, c)
            for d in range(3):
                acc[f:f + c, d] = q[(kick + d) % 4] * (2.0 ** 23 * c)
        e.update_particles(st["pos"], acc=acc)
        e.kick_halfstep(update_tree=True)
        tree, top = U.kicks(tree, top, st["mass"], acc, dt,
                            st["tree_parent"], np.arange(n, dtype=np.int32))
        got, gtop = e.tree(), e.top_nodes()
        for f in ("Bitfield", "Dp"):
            np.testing.assert_array_equal(got[f], tree[f], err_msg=f)
        for f in ("Level", "Dp"):
            np.testing.assert_array_equal(gtop[f], top[f], err_msg=f)
