"""Which runs replay the step graphs: a context that only fell back to launching its steps would still equal one
that launches them, so the captures and replays themselves are counted."""
import pytest

from cdns import config, fields

pytestmark = pytest.mark.gpu

STEPS, AFTER = 6, 40  # steps per graph, steady steps before the first capture


def small(gpu, precision="FP64"):
    cfg = dict(config.channel_32(), DT=2e-4)
    ch = gpu.Channel(cfg, precision=getattr(gpu, precision))
    ch.set_state("velocity", fields.seeded_velocity(cfg, seed=3))
    ch.run(2, it_begin=1)
    return ch


def counts(ch):
    n = ch.step_graphs()
    assert not n["failed"], ch.last_error()
    return n["captures"], n["replays"]


@pytest.mark.parametrize("precision", ["FP64", "MIXED"])
def test_steady_runs_are_replayed(gpu, precision):
    """Whole graphs as long as another step follows, one graph for each order of the swapped planes."""
    ch = small(gpu, precision)
    ch.run(AFTER)
    assert counts(ch) == (0, 0)
    ch.run(STEPS)  # the last step of a run is launched, so this run has none to replay
    assert counts(ch) == (0, 0)
    ch.run(20)  # 3 x 6 and two launched
    assert counts(ch) == (1, 3)
    ch.run(7)
    assert counts(ch) == (1, 4)
    ch.run(21)  # an odd number of steps later: the other order
    assert counts(ch) == (2, 7)
    ch.run(40)
    assert counts(ch) == (2, 13)


def test_timed_steps_and_first_steps_are_launched(gpu):
    ch = small(gpu)
    ch.profile(True)
    ch.run(100)
    assert counts(ch) == (0, 0)
    ch.profile(False)
    ch.run(100, it_begin=1)  # two launched, 16 x 6, two launched
    assert counts(ch) == (1, 16)
    for _ in range(20):
        ch.step()
    assert counts(ch) == (1, 16)


def test_a_body_force_set_and_removed_again_has_its_own_graphs(gpu):
    """Each state is captured once, however often the force comes and goes."""
    ch = small(gpu)
    force = 0.01 * fields.seeded_velocity(ch.cfg, seed=7, mean="laminar", kmax=4, amplitude=1.0)
    ch.run(AFTER)
    seen = []
    for k in range(4):
        for f in (None, force):
            ch.set_body_force(f)
            ch.run(20)
            seen.append(counts(ch))
    assert [c for c, _ in seen] == [1] + [2] * 7
    assert [r for _, r in seen] == [3 * (k + 1) for k in range(8)]
