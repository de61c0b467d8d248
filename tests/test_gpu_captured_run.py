"""A caller that captures the context's stream gets the steps themselves, no graph of the context's own, and can replay
them: against the same steps launched."""
import numpy as np
import pytest

from cdns import config, fields

pytestmark = pytest.mark.gpu


def test_run_in_a_callers_capture(gpu):
    import torch

    cfg = dict(config.channel_32(), DT=2e-4)
    u0 = fields.seeded_velocity(cfg, seed=3)
    captured, launched = gpu.Channel(cfg), gpu.Channel(cfg)
    launched.profile(True)  # never replayed
    for ch in (captured, launched):
        ch.set_state("velocity", u0)
        ch.run(60, it_begin=1)
        ch.sync()
    before = captured.step_graphs()
    assert before["captures"] == 1 and not before["failed"]
    stream = torch.cuda.ExternalStream(captured.stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        captured.run(20)
    assert captured.step_graphs() == before
    with torch.cuda.stream(stream):
        for k in range(3):  # an even number of steps: the planes are where they were captured
            graph.replay()
            captured.sync()
            launched.run(20)
            a, b = captured.get_state("velocity"), launched.get_state("velocity")
            assert np.isfinite(a).all() and np.array_equal(a, b), k
    captured.run(20)  # and its own replays go on from there
    launched.run(20)
    assert captured.step_graphs()["replays"] > before["replays"]
    assert np.array_equal(captured.get_state("velocity"), launched.get_state("velocity"))
