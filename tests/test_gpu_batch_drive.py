"""A batch member that fits on chip is its own resident solve loop: its result does
not depend on the calls that drive the batch, to the bit."""
import warnings

import numpy as np
import pytest

from tests.cases import all_fields, batch_case, build_sim, rel_l2
from tests.test_gpu_batch import SMALL
from tests.test_gpu_resident import TOL, _boxes

pytestmark = pytest.mark.gpu

LIMITS = [dict(), dict(fixed_n0=300), dict(fixed_n0=0), dict(Nmax=170.5)]


def _sim(case, limits, resident=(1, 0)):
    sim = build_sim(case)
    for key, value in limits.items():
        setattr(sim, key, value)
    sim._lib.emf_set_resident(sim._h, *resident)
    return sim


def _result(sim, case):
    return ({k: sim.last_solve[k] for k in ("n0", "Tn", "steps", "status", "nchecks")},
            list(sim.convergence_history), all_fields(sim, case, case["adjoint"]))


def _same(a, b):
    assert a[0] == b[0]
    assert np.array_equal(a[1], b[1])
    assert all(np.array_equal(x, y) for x, y in zip(a[2], b[2]))


def _driven(cases, limits, graphs, spg=8, resident=(1, 0)):
    """Results of `cases` stepped by calls of `graphs` replays, run to the end after."""
    from emopt_amd.batch import Batch
    b = Batch(steps_per_graph=spg)
    sims = [_sim(c, limits, resident) for c in cases]
    for s, c in zip(sims, cases):
        b.add(s, adjoint=c["adjoint"], postprocess=False)
    done = []
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        for n in graphs:
            done += b.run(until="graphs", max_graphs=n)
        done += b.run()
    assert sorted(done) == list(range(len(cases))) and b.running == 0
    b.close()
    return [_result(s, c) for s, c in zip(sims, cases)]


@pytest.mark.parametrize("limits", LIMITS)
def test_result_does_not_depend_on_the_calls(limits):
    cases = [batch_case(q, n_fwd=2, **SMALL) for q in (1, 3)]
    assert all(_boxes(_sim(c, limits)) > 0 for c in cases)
    whole = _driven(cases, limits, [])
    for graphs in ([1], [20, 0, 3], [7] * 30, [1 << 20]):
        for got, ref in zip(_driven(cases, limits, graphs), whole):
            _same(got, ref)
    for c, ref in zip(cases, whole):           # and is the single solve's
        sim = _sim(c, limits)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")
            if c["adjoint"]:
                sim.solve_adjoint()
            else:
                sim._register(sim._sources)
                sim._solve(0)
        _same(_result(sim, c), ref)


def test_replays_count_steps():
    """Members are stepped in order of admission, a replay's steps each time."""
    from emopt_amd.batch import Batch
    cases = [batch_case(q, n_fwd=2, **SMALL) for q in (0, 1)]
    b = Batch(steps_per_graph=16)
    sims = [_sim(c, dict(fixed_n0=100)) for c in cases]
    for s, c in zip(sims, cases):
        b.add(s, adjoint=c["adjoint"], postprocess=False)
    total = [100 + 2 * s.Tn for s in sims]
    replays, ends = 0, {}
    while b.running:
        for m in b.run(until="graphs", max_graphs=1):
            ends[m] = replays
        replays += 1
        assert replays < 100
    assert abs(16 * ends[0] - total[0]) <= 80          # a replay, and a launch of up to 64 steps
    assert abs(16 * ends[1] - sum(total)) <= 80
    b.close()


def test_stall_between_calls():
    """A member whose launches stall (polls limited to one) takes the step kernels."""
    cases = [batch_case(1, n_fwd=2, **SMALL)]
    ref = _driven(cases, dict(fixed_n0=300), [], resident=(0, 0))[0]
    for graphs in ([], [20, 3], [7] * 30):
        got = _driven(cases, dict(fixed_n0=300), graphs, resident=(1, 1))[0]
        assert got[0] == ref[0]
        assert max(rel_l2(x, y) for x, y in zip(got[2], ref[2])) <= TOL


def test_any_is_bounded_by_replays():
    """until="any" returns after max_graphs replays where no member has finished."""
    from emopt_amd.batch import Batch
    cases = [batch_case(q, n_fwd=2, **SMALL) for q in (0, 1)]
    whole = _driven(cases, dict(fixed_n0=200), [])
    b = Batch(steps_per_graph=16)
    sims = [_sim(c, dict(fixed_n0=200)) for c in cases]
    for s in sims:
        b.add(s, postprocess=False)
    calls, done = 0, []
    while b.running:
        done += [(m, calls) for m in b.run(until="any", max_graphs=2)]
        calls += 1
        assert calls < 100
    assert [m for m, _ in done] == [0, 1]
    steps = [200 + 2 * s.Tn for s in sims]
    assert abs(32 * done[0][1] - steps[0]) <= 96       # a call, and a launch
    assert abs(32 * done[1][1] - sum(steps)) <= 160    # and the call that ended with the first
    b.close()
    for s, c, ref in zip(sims, cases, whole):
        _same(_result(s, c), ref)


def test_neither_kind_of_member_waits_for_ever():
    """A member that the graphs step finishes while members that fit on chip keep
    coming, and they while it runs; the results are those of each alone."""
    from emopt_amd.batch import Batch
    big, small = batch_case(0, n_fwd=2, **SMALL), batch_case(1, n_fwd=2, **SMALL)
    ref_big = _driven([big], dict(fixed_n0=600), [], spg=16, resident=(0, 0))[0]
    ref_small = _driven([small], dict(fixed_n0=20), [], spg=16)[0]
    b = Batch(steps_per_graph=16)
    sim = _sim(big, dict(fixed_n0=600), (0, 0))
    mid = b.add(sim, postprocess=False)
    limit = 3 * (600 + 2 * sim.Tn) // (4 * 16) + 4     # a turn of 4 replays in 3 calls
    live, got = {}, []
    for calls in range(limit):
        if not live:
            s = _sim(small, dict(fixed_n0=20))
            live[b.add(s, postprocess=False)] = s
        done = b.run(until="any", max_graphs=4)
        got += [live.pop(m) for m in done if m in live]
        if mid in done:
            break
    else:
        pytest.fail("the graphs' member has not finished after %d calls" % limit)
    print("big member done after %d of %d calls, %d small ones" % (calls + 1, limit, len(got)))
    assert len(got) >= 2
    b.run()
    b.close()
    _same(_result(sim, big), ref_big)
    for s in got:
        _same(_result(s, small), ref_small)
