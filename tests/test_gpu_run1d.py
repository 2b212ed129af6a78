"""1-D runs on chip (csrc/run1d.hpp) against the launches per stage they
replace: mara_block_run with graphs off launches every kernel from the host,
and both end in the same state, clock, step count and report, bit for bit --
at the lengths where a block fits one work-group of 256 or 512 threads or is
split (even and uneven), in both laws, every reconstruction, boundary and
form, at a final time, at a step limit, across calls, and through a failure."""
import numpy as np
import pytest

import oracle
from mara2_amd import abi, problems
from mara2_amd.runtime import Block

pytestmark = pytest.mark.gpu


def _random(desc, seed=5, guards=True):
    rng = np.random.default_rng(seed)
    P = problems.empty(desc)
    x = np.linspace(0, 8, P.shape[0])[:, None, None]
    P[..., 0] = 1 + 0.4 * np.sin(x) + 0.2 * rng.random(P.shape[:3])
    P[..., 4] = 1 + 0.4 * np.cos(x) + 0.2 * rng.random(P.shape[:3])
    P[..., 1:4] = 0.4 * rng.standard_normal(P.shape[:3] + (3,))
    if P.shape[3] >= 8:
        P[..., 5] = 0.5
        P[..., 6:8] = 0.4 * rng.standard_normal(P.shape[:3] + (2,))
    return problems.apply_bc(desc, P) if guards else P


def _both(desc, P, t_final=1e300, steps=40, cfl=0.4, calls=2):
    out = []
    for graphs in (True, False):
        with Block(desc) as blk:
            blk.set_graphs(graphs)
            blk.upload(P)
            t, seen = 0.0, []
            for _ in range(calls):
                t, n, rep = blk.run(cfl, t_final, steps, t=t, check=False)
                seen.append((t, n, rep.as_dict()))
            out.append((blk.download(), seen))
    (Pc, a), (Pl, b) = out
    assert a == b
    assert np.array_equal(Pc, Pl, equal_nan=True)
    return a


@pytest.mark.parametrize("n", [2, 3, 64, 251, 252, 253, 254, 500, 508, 509, 513, 744, 1024, 2999, 10007, 16384, 19840,
                               19841])
@pytest.mark.parametrize("law", ["hydro", "mhd"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lengths(n, law, precision):
    bc = ("outflow", "periodic", "reflecting")[n % 3]
    desc = abi.make_desc(law=law, bc=bc, cells=(n, 1, 1), precision=precision, pressure_floor=1e-6)
    _both(desc, _random(desc), steps=25)


@pytest.mark.parametrize("bc", ["outflow", "periodic", "reflecting"])
@pytest.mark.parametrize("recon", ["pcm", "plm", "weno5"])
@pytest.mark.parametrize("kind", ["hydro_hlle", "hydro_hllc", "mhd_ct", "mhd_no_ct"])
@pytest.mark.parametrize("n", [200, 700])
def test_schemes_and_boundaries(n, kind, recon, bc):
    law, opt = kind.split("_", 1)
    desc = abi.make_desc(law=law, recon=recon, riemann=opt if law == "hydro" else "hlle", bc=bc, cells=(n, 1, 1),
                         field_ct=1 if opt == "ct" else 0, pressure_floor=1e-6)
    _both(desc, _random(desc))


@pytest.mark.parametrize("n", [150, 900])
@pytest.mark.parametrize("precision", ["fp64", "fp64_fast", "mixed"])
def test_stops_at_the_final_time(n, precision):
    desc = abi.make_desc(law="hydro", riemann="hllc", bc="outflow", cells=(n, 1, 1), precision=precision)
    (t, steps, _), again = _both(desc, _random(desc), t_final=0.02, steps=10000)
    assert t == 0.02 and steps > 1 and again[:2] == (0.02, 0)


@pytest.mark.parametrize("n", [130, 2000])
@pytest.mark.parametrize("bc", ["periodic", "outflow"])
def test_guards_as_uploaded(n, bc):
    """Guards that are not the boundary condition's images count in the first step."""
    desc = abi.make_desc(law="hydro", bc=bc, cells=(n, 1, 1))
    _both(desc, _random(desc, guards=False), steps=3, calls=1)


@pytest.mark.parametrize("n", [190, 1300])
@pytest.mark.parametrize("stage_zone", [5, 100, 125, 160])
def test_a_failing_zone_ends_the_run(n, stage_zone):
    """No pressure floor and a zone the update cannot recover: the same zone is
    reported, the rest of the step stands, the zone keeps its old value."""
    desc = abi.make_desc(law="mhd", bc="periodic", cells=(n, 1, 1))
    P = _random(desc)
    P[stage_zone, 0, 0, 4] = 1e-9
    P[stage_zone - 1:stage_zone + 2, 0, 0, 1] = [-30.0, 0.0, 30.0]
    problems.apply_bc(desc, P)
    (t, steps, rep), again = _both(desc, P, steps=30)
    assert rep["c2p_failures"] > 0 and steps < 30


@pytest.mark.parametrize("law", ["hydro", "mhd"])
@pytest.mark.parametrize("n", [90, 252, 400])
def test_host_loop_equals_oracle(n, law):
    """courant_dt and advance of a block of one work-group, a launch each."""
    desc = abi.make_desc(law=law, bc="outflow", cells=(n, 1, 1), pressure_floor=1e-6)
    P = _random(desc)
    Po = P.copy()
    with Block(desc) as blk:
        blk.upload(P)
        for _ in range(5):
            dt = blk.courant_dt()
            err, do = oracle.courant_dt(desc, Po)
            assert err == 0 and dt == do
            blk.advance(0.4 * dt)
            err, _ = oracle.advance(desc, Po, 0.0, 0.4 * dt)
            assert err == 0
        assert np.array_equal(blk.download(), Po)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_solves_of_a_batch(precision):
    """1-D solves of every kind and length together on chip, some in more
    work-groups than one launch holds, one with guards that are not its
    boundary condition's (it goes by launches), against the batch that launches
    every kernel from the host: the same states, clocks, steps and statuses,
    whatever the steps per call."""
    from mara2_amd.runtime import Batch
    kinds = []
    for k, n in enumerate([3, 60, 248, 249, 252, 700, 1000, 3001, 16384, 16384, 16384, 16384, 49000, 51000]):
        law = "mhd" if k % 2 else "hydro"
        bc = ("outflow", "periodic", "reflecting")[k % 3]
        recon = ("plm", "plm", "weno5", "pcm")[k % 4]
        desc = abi.make_desc(law=law, recon=recon, bc=bc, cells=(n, 1, 1), precision=precision, pressure_floor=1e-6,
                             riemann="hllc" if law == "hydro" else "hlle")
        kinds.append((desc, _random(desc, seed=k, guards=k != 4), 1e300 if k % 2 else 0.3 / n, 40 + k))
    assert kinds[4][0].bc == abi.BC_PERIODIC
    seen = []
    for graphs, chunk in ((False, 16), (True, 16), (True, 1)):
        with Batch(1 << 29, precision=precision, max_solves=len(kinds)) as b:
            b.set_graphs(graphs)
            slots = [b.admit(d, P, 0.4, t, s) for d, P, t, s in kinds]
            assert None not in slots and all(b.lane(s) == 1 for s in slots)
            calls = 0
            while b.step(chunk):
                calls += 1
                assert calls < 200
            state = [b.query(s) for s in slots]
            seen.append(([(q[0], q[1], q[2], q[3], q[4].as_dict()) for q in state], [b.retire(s) for s in slots]))
    for info, states in seen[1:]:
        assert info == seen[0][0]
        assert all(np.array_equal(a, c) for a, c in zip(states, seen[0][1]))
