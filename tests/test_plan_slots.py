"""When a chained plan's results are handed over by value, and that it then is what the calls one after the other are: the
host's proof (plan_slots in oxh_plan.hip) over random dependent plans, run on a simulation of the workgroups."""
import numpy as np
import pytest

import plan_sim
from oxidize_amd import matvec as mv

Q4K = 13


def by_value_plans(rng, many):
    """(operations, words, draft) of that many random chains that go by value, and how many do not."""
    found, not_so = [], 0
    while len(found) < many:
        chain = plan_sim.random_chain(rng, mv.make_segments)
        if chain is None:
            continue
        try:
            draft = mv.plan_draft(chain[0], int(rng.choice([4, 5, 8, 16, 20])))
        except mv.OxhError:                 # more rows than so few workgroups can own
            continue
        if draft["by_value"]:
            found.append((chain[0], chain[1], draft))
        elif any(o["wait"] for o in draft["ops"]):
            not_so += 1
    return found, not_so


@pytest.mark.parametrize("seed", range(8))
def test_random_chains_by_value_read_what_the_calls_one_by_one_read(seed):
    rng = np.random.default_rng(100 + seed)
    found, not_so = by_value_plans(rng, 6)
    assert not_so > 0                       # and some of them are turned down
    for ops, cells, draft in found:
        sim = plan_sim.Sim(ops, draft, plan_sim.BASE, cells, plan_sim.rows_of, rng)
        for _ in range(3):                  # the slots carry over from launch to launch
            sim.launch()


@pytest.mark.parametrize("mistake", ["sets stay in place", "one slot for two results"])
def test_the_simulation_sees_a_wrong_hand_over(mistake):
    """The same chains with a mistake in the slots they were given: at least one has to come out wrong."""
    rng = np.random.default_rng(7)
    wrong = 0
    for ops, cells, draft in by_value_plans(rng, 12)[0]:
        for o in draft["ops"]:
            if mistake == "sets stay in place":
                o["seg_slot"] = [s & ~2 for s in o["seg_slot"]]
                o["slot"] = {k: v & ~2 if v < draft["set_bytes"] else v for k, v in o["slot"].items()}
            else:
                o["seg_slot"] = [s and (s & 3) + 4 for s in o["seg_slot"]]
        sim = plan_sim.Sim(ops, draft, plan_sim.BASE, cells, plan_sim.rows_of, rng)
        try:
            for _ in range(3):
                sim.launch()
        except plan_sim.Wrong:
            wrong += 1
    assert wrong > 0


def op(x, cols, out, rows, **more):
    return dict(qtype=Q4K, cols=cols, d_x=x, segs=mv.make_segments([(1 << 50, out, rows, 0)]), **more)


def test_which_chains_go_by_value():
    """On 256 compute units.  A result read whole or in part, a prologue's output and its sum do; an input made of two
    results, one whose address is no multiple of four into a result, a norm's weights written by the plan, an input stored
    over before everybody is known to have read it and results of different operations at one place do not, nor do
    chains of mostly long vectors."""
    v = [(1 << 40) + i * (1 << 20) for i in range(12)]
    first = op(v[0], 4096, v[1], 4096)

    def goes(*more):
        return mv.plan_draft([first] + list(more))["by_value"]
    assert goes(op(v[1], 4096, v[2], 4096))
    assert goes(op(v[1] + 400, 2048, v[2], 4096))
    assert not goes(op(v[1] - 400, 4096, v[2], 4096))                                  # half of it nobody's
    assert not goes(op(v[1] + 2, 2048, v[2], 4096))
    assert not mv.plan_draft([first, op(v[0], 4096, v[1] + 4 * 4096, 256), op(v[1] + 1024, 4096, v[2], 4096)])["by_value"]
    add = dict(kind=mv.PRO_RMSNORM, d_b=v[9], eps=1e-5, d_add=v[0], d_sum_out=v[3], d_pro_out=v[4])
    assert goes(op(v[1], 4096, v[2], 4096, **add), op(v[3], 4096, v[5], 64), op(v[4], 4096, v[6], 64))
    assert not goes(op(v[0], 4096, v[2], 4096, kind=mv.PRO_RMSNORM, d_b=v[1], eps=1e-5))
    assert goes(op(v[0], 4096, v[2], 4096, kind=mv.PRO_SWIGLU, d_b=v[1]))
    # v[0] stored over: by the operation that follows its reader, and one later, when everybody has read v[1]
    assert goes(op(v[1], 4096, v[0], 4096))
    assert not mv.plan_draft([op(v[0], 4096, v[1], 256), op(v[0], 4096, v[2], 4096), op(v[1], 256, v[0], 4096)])["by_value"]
    # two results at one place: of the same workgroups, and of others
    assert goes(op(v[1], 4096, v[2], 4096), op(v[2], 4096, v[1], 4096))
    assert not goes(op(v[0], 4096, v[2], 64), op(v[1], 4096, v[2], 4096))
    assert not mv.plan_draft([op(v[0], 4352, v[1], 4352), op(v[1], 4352, v[2], 4096)])["by_value"]
    assert not mv.plan_draft([first, op(v[1], 4096, v[2], 4352), op(v[2], 4352, v[3], 4352)])["by_value"]


def test_operations_that_share_the_place_of_their_quantised_bytes_go_by_value_only_apart():
    """A block of a vector of up to sixteen is stored by another workgroup than the same block of a longer one."""
    v = [(1 << 40) + i * (1 << 20) for i in range(6)]
    act = 1 << 45

    def chain(second):
        return [op(v[0], 4096, v[1], 4352 if second == 1 else 4096, d_act_out=act),
                op(v[1], 4352 if second == 1 else 4096, v[2], 4096, d_act_out=act if second == 1 else None),
                op(v[2], 4096, v[3], 4352 if second == 3 else 4096),
                op(v[3], 4352 if second == 3 else 4096, v[4], 4096, d_act_out=act if second == 3 else None),
                op(v[4], 4096, v[5], 4096)]
    assert not mv.plan_draft(chain(1))["by_value"] and mv.plan_draft(chain(3))["by_value"]
