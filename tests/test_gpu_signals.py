"""Learning signals at the edges of their batches (eight destinations a wave,
dealt over every wave of the lane) against the oracle: a step's destinations
are the targets of one input row of `fanout` distinct neurons, and the serial
257-term sums show in the updated input weights, compared bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from leo_amd import native
from leo_amd.model import Model
from tests.helpers import assert_models_equal, small_redundant_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fanout", [1, 7, 8, 9, 15, 17, 255, 256, 257, 521, 1000])
def test_signal_batches_match_oracle(require_gpu, oracle, fanout):
    from leo_amd.runtime import HipRuntime

    cfg = small_redundant_config(neurons=1024, synapses=4, fanout=fanout, per_block=8, dropout=0.0)
    cfg.validate()
    model = Model.synthetic(cfg, weight_sigma=0.05)
    rng = np.random.default_rng(fanout)
    model.in_target.reshape(258, fanout)[:] = [rng.permutation(1024)[:fanout] for _ in range(258)]
    model.in_weight[:] = rng.uniform(0.2, 1.0, model.in_weight.size).astype(np.float32)
    # a weight of -0.0 (in a row no step reads) makes every kept slot a learning
    # slot: with the zero-eligibility skip the touched neurons far from their
    # block's cutoff would claim no destination
    model.in_weight[0] = np.float32(-0.0)
    model.out_weight[:] = rng.uniform(-1.0, 1.0, model.out_weight.size).astype(np.float32)
    model.validate()
    cpu = oracle.OracleRuntime(model)
    gpu = HipRuntime(model, device=0, max_lanes=1)
    try:
        cpu.begin_document()
        gpu.begin_document()
        for symbol, target in ((65, 66), (66, 67), (65, 200)):
            c = cpu.step(symbol, target, oracle.TRAINING)
            g = gpu.step(symbol, target, native.TRAINING)
            assert g.loss == c.loss
        assert gpu.kernel_stats()["destinations"] >= fanout
        assert_models_equal(gpu.model(), cpu.model(), f"fanout {fanout}")
    finally:
        gpu.close()


@pytest.mark.parametrize("fanout", [32, 33, 63, 64, 65, 96, 97, 128, 136, 161, 500, 1000])
def test_many_batches_a_wave_match_oracle(require_gpu, oracle, monkeypatch, fanout):
    """One workgroup: four waves of eight destinations a batch, so that a wave
    takes one, two, an odd and an even number of batches, whole and ragged."""
    monkeypatch.setenv("LEO_HIP_CANONICAL_WGS", "1")
    monkeypatch.setenv("LEO_HIP_WGS_PER_LANE", "1")
    test_signal_batches_match_oracle(require_gpu, oracle, fanout)
