"""The learning phase's lists (learning slots, inhibitory rows, output rows)
dealt as one round-robin, against the oracle: lists of none, of fewer and of
many more items than the lane has threads, on one, two and more workgroups.
Losses and the model bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from leo_amd import native
from leo_amd.model import BEGIN_DOCUMENT, END_DOCUMENT, Model
from tests.helpers import assert_models_equal, small_redundant_config, story

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workgroups", ["1", "2", "4"])
@pytest.mark.parametrize("per_block,low", [(6, -0.2), (8, 0.2), (40, 0.4)])
def test_learning_lists_match_oracle(require_gpu, oracle, monkeypatch, workgroups, per_block, low):
    from leo_amd.runtime import HipRuntime

    monkeypatch.setenv("LEO_HIP_WGS_PER_LANE", workgroups)
    monkeypatch.setenv("LEO_HIP_CANONICAL_WGS", workgroups)
    cfg = small_redundant_config(neurons=1024, synapses=24, fanout=300, per_block=per_block)
    model = Model.synthetic(cfg, weight_sigma=0.2)
    rng = np.random.default_rng(per_block)
    model.in_weight[:] = rng.uniform(max(low, 0.0), 1.0, model.in_weight.size).astype(np.float32)
    if low < 0:  # hardly any neuron fires: steps with empty lists
        model.in_weight[:] *= np.float32(0.1)
    model.validate()
    cpu = oracle.OracleRuntime(model)
    gpu = HipRuntime(model, device=0, max_lanes=1)
    try:
        for length in (1, 70):
            text = story(60 + length, length + 1)
            steps = list(zip([BEGIN_DOCUMENT] + list(text), list(text) + [END_DOCUMENT]))
            cpu.begin_document()
            gpu.begin_document()
            want = [cpu.step(s, t, oracle.TRAINING).loss for s, t in steps]
            got = [m.loss for m in gpu.training_step_batch(steps, native.TRAINING)]
            cpu.finish_document()
            gpu.finish_document()
            assert got == want
        assert_models_equal(gpu.model(), cpu.model(), f"{per_block} winners a block, {workgroups} workgroups")
    finally:
        gpu.close()
