"""Domain_Decomposition with NTarget > 1 (domain.c:67-145) through the C
ABI against the oracle on the same particles and P.Cost: the same bunches
as top nodes (keys, levels, particle ranges, float centres), the same
target for each and the same number of passes; then the tree on those top
nodes and the FP64 walk, bit for bit as in the other parity tests."""
import numpy as np
import pytest

import oracle
from tandav_amd import Engine, TDVError, ics
from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ewald():
    return oracle.cached_ewald_table()


@pytest.mark.parametrize("case,ntarget", [("clustered", 2), ("clustered", 8),
                                          ("clustered", 16),
                                          ("periodic", 8), ("periodic", 64)])
def test_domain_targets_match_oracle(case, ntarget, ewald):
    from test_oracle_tree import clustered
    if case == "periodic":
        pos, _, m = ics.zeldovich_box(32, seed=7)
        kw = dict(periodic=True, softening=1 / 1280.)
    else:
        pos, m = clustered(30000, 5)
        kw = dict(periodic=False, softening=1e-3)
    table = ewald if kw["periodic"] else None
    print("case", case, "ntarget", ntarget, flush=True)
    s = oracle.Sim(pos, m, alpha_rel=0.005, nthreads=16, ewald_table=table,
                   **kw)
    s.setup_domain()
    s.domain_decomposition()
    s.compute_acceleration(True)            # P.Cost for the decomposition
    tasks_s, it_s = s.domain_decomposition_targets(ntarget)
    s.compute_acceleration(False)
    e = Engine(alpha_rel=0.005, compat=True, **kw)
    if kw["periodic"]:
        e.set_ewald_table(ewald)
    e.set_particles(pos, m)
    e.setup_domain()
    e.domain_decomposition()
    e.compute_acceleration(True)
    tasks_e, it_e = e.domain_decomposition_targets(ntarget)
    assert it_e == it_s
    np.testing.assert_array_equal(tasks_e, tasks_s)
    assert len(tasks_e) == len(s.top)
    e.compute_acceleration(False)
    _compare(s, e)


def test_domain_targets_rejects_too_few_bunches():
    """Every particle in one level-2 cell: one bunch for two targets (the
    reference would index past its bunch list) is an error."""
    g = np.random.Generator(np.random.Philox(4))
    pos = 0.01 * g.random((5000, 3))        # one cell of the unit box
    m = np.full(5000, 1.0 / 5000)
    e = Engine(periodic=True, boxsize=1.0, softening=1e-3)
    e.set_particles(pos, m)
    with pytest.raises(TDVError):
        e.domain_decomposition_targets(2)


@pytest.mark.parametrize("n,ntarget", [(1000, 2), (65537, 3), (400000, 16)])
def test_domain_targets_of_long_cost_sums_match_oracle(n, ntarget):
    """Bunches of up to a few hundred thousand particles: their float costs
    in particle order, from the walk's own Cost, bit for bit the serial
    sums (the refinement depends on every one of them)."""
    pos, _, m = ics.clustered_box(n, nhalo=3, seed=9)
    e = Engine(periodic=True, softening=1e-4, alpha_rel=0.005, compat=False,
               precision="fp32", fp32_criterion=3, ewald_accuracy=1.0)
    e.set_particles(pos, m)
    e.setup_domain()
    e.domain_decomposition()
    e.compute_acceleration(True)
    cost = e.get("cost")["cost"]
    short = e.keys(reversed_=False)[:, 1].copy()
    rec, it = oracle.domain_targets(short, cost, ntarget)
    tasks, passes = e.domain_decomposition_targets(ntarget)
    top = e.top_nodes()
    assert passes == it
    assert len(top) == len(rec)
    for f in ("Key", "Level", "First_Part", "Npart"):
        np.testing.assert_array_equal(top[f], rec[f], err_msg=f)
    np.testing.assert_array_equal(tasks, -rec["Target"] - 1)


def test_reports_after_the_top_node_table_grew():
    """More than 64 top nodes move the table; the counts that every call's
    report reads stay, and so does what comes after."""
    pos, _, m = ics.clustered_box(20000, nhalo=8, seed=4)
    e = Engine(periodic=True, softening=1e-3, alpha_rel=0.005)
    e.set_particles(pos, m)
    e.setup_domain()
    e.domain_decomposition()
    e.compute_acceleration(True)
    few = e.top_nodes()
    for _ in range(2):
        e.domain_decomposition_targets(60)
        assert len(e.top_nodes()) > 64
        e.tree_build()
        assert int(e.top_nodes()["Npart"].sum()) == len(m)
        keys = np.arange(2 * 5000, dtype=np.uint64).reshape(5000, 2)[::-1]
        np.testing.assert_array_equal(e.sort_keys(np.ascontiguousarray(keys)),
                                      np.arange(5000)[::-1])
        e.set_particles(pos, m)
        e.setup_domain()
        e.domain_decomposition()
        e.compute_acceleration(True)
        np.testing.assert_array_equal(e.top_nodes(), few)
