"""Block selection at the edges of a wave's window against the oracle: touched
neurons below and past its 256 entries, few candidates (placed through lane
reads) and more (one block's compared as they are, several blocks' sorted
first), blocks smaller than a bitmap word,
not a multiple of one, and of the largest size. Inputs strong enough that most
injected neurons are candidates; losses, lists and the model bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from leo_amd import native
from leo_amd.config import Config
from leo_amd.config import test_toml_values as toml_values
from leo_amd.model import Model
from tests.helpers import assert_models_equal, story

pytestmark = pytest.mark.gpu

SHAPES = [  # neurons per block, blocks, input edges per symbol, winners per block
    (16, 64, 40, 2), (16, 640, 900, 3), (20, 96, 500, 5), (96, 40, 63, 4), (96, 40, 1500, 90),
    (200, 24, 65, 8), (256, 4, 64, 8), (256, 4, 700, 16), (256, 520, 4000, 1), (1024, 2, 1900, 64),
    (256, 4, 160, 16), (64, 64, 1300, 16),
]


RUNS = [  # one workgroup's four waves: groups of 64 blocks (40 of 320 neurons) in runs of many, few and one block
    (16, 260, 2200, 3), (64, 256, 3000, 4), (256, 66, 2400, 4), (256, 16, 3900, 8), (320, 48, 2500, 5),
]


@pytest.mark.parametrize("nb,blocks,fanout,limit", RUNS)
def test_runs_of_blocks_match_oracle(require_gpu, oracle, monkeypatch, nb, blocks, fanout, limit):
    monkeypatch.setenv("LEO_HIP_WGS_PER_LANE", "1")
    monkeypatch.setenv("LEO_HIP_CANONICAL_WGS", "1")
    test_selection_matches_oracle(require_gpu, oracle, nb, blocks, fanout, limit)


@pytest.mark.parametrize("nb,blocks,fanout,limit", SHAPES)
def test_selection_matches_oracle(require_gpu, oracle, nb, blocks, fanout, limit):
    from leo_amd.runtime import HipRuntime

    values = toml_values()
    n = nb * blocks
    values["model"].update(neuron_count=n, block_count=blocks, neurons_per_block=nb, synapses_per_neuron=6,
                           input_fanout=fanout, max_active_per_block=limit, max_active_global=blocks * limit)
    values["dynamics"].update(target_activity=min(0.5, 0.9 * limit / nb), population_inhibition_rate=0.001)
    model = Model.synthetic(Config.from_dict(values), weight_sigma=0.05)
    rng = np.random.default_rng(nb * 1000 + fanout)
    model.in_target.reshape(258, fanout)[:] = [rng.permutation(n)[:fanout] for _ in range(258)]
    model.in_branch[:] = 0
    model.in_weight[:] = rng.uniform(0.3, 1.0, model.in_weight.size).astype(np.float32)
    model.threshold[:] = np.float32(0.4)
    model.validate()
    cpu = oracle.OracleRuntime(model)
    gpu = HipRuntime(model, device=0, max_lanes=1)
    text = story(nb + blocks, 24)
    try:
        cpu.begin_document()
        gpu.begin_document()
        for b in text[:8]:
            c = cpu.step(b, None, oracle.FROZEN)
        gpu.advance_frozen_batch([(b, None) for b in text[:8]])
        assert gpu.active_neurons().size == c.active_neurons
        for b, t in zip(text[8:], text[9:]):
            c = cpu.step(b, t, oracle.TRAINING)
            g = gpu.step(b, t, native.TRAINING)
            assert (g.loss, g.active_neurons, g.suprathreshold_neurons) == (c.loss, c.active_neurons,
                                                                             c.suprathreshold_neurons)
        assert np.array_equal(gpu.read_state("membrane"), cpu.read_f32("membrane"))
        assert_models_equal(gpu.model(), cpu.model(), f"{blocks} blocks of {nb}")
    finally:
        gpu.close()
