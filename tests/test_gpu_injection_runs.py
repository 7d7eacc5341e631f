"""Frozen runs whose injections go out several ticks ahead, against the oracle
stepping one byte at a time: input rows from one edge to more items than the
lane has threads, runs that end inside and at the edge of such a group, of the
64 step parameters held at a time, and of a launch; then learning steps on top
of the state the run left."""
from __future__ import annotations

import numpy as np
import pytest

from leo_amd import native
from leo_amd.model import Model
from tests.helpers import assert_models_equal, small_redundant_config, story

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cut", [0, 9])
@pytest.mark.parametrize("fanout", [1, 63, 65, 600])
def test_frozen_runs_match_oracle(require_gpu, oracle, monkeypatch, fanout, cut):
    from leo_amd.runtime import HipRuntime

    if cut:
        monkeypatch.setenv("LEO_HIP_MAX_STEPS_PER_LAUNCH", str(cut))
    cfg = small_redundant_config(neurons=1024, synapses=8, fanout=fanout, per_block=8, dropout=0.0)
    cfg.validate()
    model = Model.synthetic(cfg, weight_sigma=0.05)
    rng = np.random.default_rng(fanout)
    model.in_weight[:] = rng.uniform(0.2, 1.0, model.in_weight.size).astype(np.float32)
    model.validate()
    cpu = oracle.OracleRuntime(model)
    gpu = HipRuntime(model, device=0, max_lanes=1)
    text = story(fanout + 3, 200)
    try:
        for run in (1, 2, 8, 9, 10, 17, 63, 64, 65, 66, 131):
            cpu.begin_document()
            gpu.begin_document()
            for b in text[:run]:
                cpu.step(b, None, oracle.FROZEN)
            gpu.advance_frozen_batch([(b, None) for b in text[:run]])
            for name in ("membrane", "branches", "fatigue"):
                assert np.array_equal(gpu.read_state(name), cpu.read_f32(name)), f"run of {run}: {name}"
            c = [cpu.step(b, t, oracle.TRAINING) for b, t in zip(text[run:run + 10], text[run + 1:])]
            g = gpu.training_step_batch(list(zip(text[run:run + 10], text[run + 1:])), native.TRAINING)
            assert [m.loss for m in g] == [m.loss for m in c], f"after a run of {run}"
        assert_models_equal(gpu.model(), cpu.model(), f"fanout {fanout}")
    finally:
        gpu.close()
