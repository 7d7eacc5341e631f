"""Kernel time of dense steps against sparse ones of the same model in the same
process: what a step does per candidate has to stay a small part of it. The
limits lie between the time ratios measured with a batched and with a serial
form of the work (both stated), near their geometric mean."""
from __future__ import annotations

import numpy as np
import pytest

from leo_amd import native
from leo_amd.config import Config
from leo_amd.config import test_toml_values as toml_values
from leo_amd.model import Model
from tests.helpers import story

pytestmark = pytest.mark.gpu


def _model(nb, blocks, fanout, limit, strength=1.0):
    """Input edges strong enough (at 1.0) that most injected neurons are above their threshold."""
    values = toml_values()
    n = nb * blocks
    values["model"].update(neuron_count=n, block_count=blocks, neurons_per_block=nb, synapses_per_neuron=6,
                           input_fanout=fanout, max_active_per_block=limit, max_active_global=blocks * limit)
    values["dynamics"].update(target_activity=min(0.5, 0.9 * limit / nb), population_inhibition_rate=0.001)
    model = Model.synthetic(Config.from_dict(values), weight_sigma=0.05)
    rng = np.random.default_rng(nb * 1000 + fanout)
    model.in_target.reshape(258, fanout)[:] = [rng.permutation(n)[:fanout] for _ in range(258)]
    model.in_branch[:] = 0
    model.in_weight[:] = (strength * rng.uniform(0.3, 1.0, model.in_weight.size)).astype(np.float32)
    model.threshold[:] = np.float32(0.4)
    model.validate()
    return model


def _best(model, run, value):
    """Smallest value of the kernel statistics of five passes."""
    from leo_amd.runtime import HipRuntime

    gpu = HipRuntime(model, device=0, max_lanes=1)
    try:
        best = float("inf")
        for _ in range(5):
            gpu.kernel_stats(reset=True)
            run(gpu)
            best = min(best, value(gpu.kernel_stats()))
        return best
    finally:
        gpu.close()


TEXT = story(5, 120)


def _step_us(model, run, steps):
    return _best(model, run, lambda stats: stats["kernel_ms"] * 1e3 / steps)


def _frozen(gpu):
    gpu.begin_document()
    gpu.advance_frozen_batch([(b, None) for b in TEXT])


# Frozen steps with nearly every neuron of a wave's one block a candidate,
# against the same deliveries with none. With one dependent pair of LDS reads a
# comparison 46 and 7.5 times; with independent reads 8.4 and 2.4 (6.5 and 2.2 with
# runs of blocks planned by one scan).
@pytest.mark.parametrize("nb,blocks,fanout,limit,most", [(1024, 2, 1900, 64, 20.0), (256, 4, 1000, 16, 4.2)])
def test_ranking_many_candidates(require_gpu, nb, blocks, fanout, limit, most):
    none = _step_us(_model(nb, blocks, fanout, limit, 0.001), _frozen, len(TEXT))
    dense = _step_us(_model(nb, blocks, fanout, limit), _frozen, len(TEXT))
    print(f"{blocks} blocks of {nb}: {none:.1f} us a step without candidates, {dense:.1f} us with", flush=True)
    assert dense < most * none


# The readout's own time (phase 2 of the workgroup that selects nothing) against
# that of two winners. Two waves' winners, 64 and 128 each: walked by one thread
# a wave 3.7 and 6.8 times; placed at once 2.2 and 3.4 (1.6 and 2.3 with the end
# class summed sixteen terms a round). 1,024 winners: with the end class summed
# one LDS read a term 11.6 times, sixteen a round 7.1.
@pytest.mark.parametrize("nb,blocks,fanout,winners,most",
                         [(1024, 2, 300, 64, 2.9), (1024, 2, 300, 128, 4.8), (256, 64, 1500, 16, 9.1)])
def test_reading_out_many_winners(require_gpu, monkeypatch, nb, blocks, fanout, winners, most):
    monkeypatch.setenv("LEO_HIP_PHASE_PROFILE", "1")
    monkeypatch.setenv("LEO_HIP_PROFILE_PART", "255")  # the last workgroup

    def run(gpu):
        gpu.evaluate([TEXT])

    def work(stats):
        return stats["phase_work_us"][2] / (len(TEXT) + 1)

    two = _best(_model(1024, 2, 300, 1), run, work)
    many = _best(_model(nb, blocks, fanout, winners), run, work)
    print(f"{winners} winners a block of {nb}: readout {many:.1f} us, of two winners {two:.1f}", flush=True)
    assert many < most * two
