"""Runs of scored frozen steps, whose next tick is delivered while the last
workgroup reads this one out, against the oracle stepping one byte at a time:
lanes of one, two and more workgroups, launches that end inside a run, after
unscored frozen steps and before learning ones; records, neuron state and the
model bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from leo_amd import native
from leo_amd.model import BEGIN_DOCUMENT, END_DOCUMENT, Model
from tests.helpers import assert_models_equal, small_redundant_config, story

pytestmark = pytest.mark.gpu

FIELDS = ("loss", "predicted_symbol", "active_neurons", "emitted_events", "population_inhibition", "context_cells")


@pytest.mark.parametrize("workgroups", ["1", "2", "5"])
@pytest.mark.parametrize("cut", ["", "1", "7"])
def test_scored_runs_match_oracle(require_gpu, oracle, monkeypatch, workgroups, cut):
    from leo_amd.runtime import HipRuntime

    monkeypatch.setenv("LEO_HIP_WGS_PER_LANE", workgroups)
    monkeypatch.setenv("LEO_HIP_CANONICAL_WGS", workgroups)
    if cut:
        monkeypatch.setenv("LEO_HIP_MAX_STEPS_PER_LAUNCH", cut)
    cfg = small_redundant_config(neurons=2048, fanout=200, dropout=0.0)
    model = Model.synthetic(cfg, weight_sigma=0.05)
    rng = np.random.default_rng(5)
    model.in_weight[:] = rng.uniform(0.2, 1.0, model.in_weight.size).astype(np.float32)
    model.validate()
    cpu = oracle.OracleRuntime(model)
    gpu = HipRuntime(model, device=0, max_lanes=3)
    texts = [story(41, 90), story(42, 33), story(43, 2)]
    document = lambda t: list(zip([BEGIN_DOCUMENT] + list(t), list(t) + [END_DOCUMENT]))  # noqa: E731
    try:
        for prefix, scored in ((0, 1), (0, 2), (11, 1), (20, 30), (3, 66)):
            cpu.begin_document()
            gpu.begin_document()
            steps = document(texts[0])
            for symbol, _ in steps[:prefix]:
                cpu.step(symbol, None, oracle.FROZEN)
            gpu.advance_frozen_batch([(s, None) for s, _ in steps[:prefix]])
            for permission, part in (("FROZEN", steps[prefix:prefix + scored]), ("TRAINING", steps[-9:])):
                c = [cpu.step(s, t, getattr(oracle, permission)) for s, t in part]
                g = gpu.training_step_batch(part, getattr(native, permission))
                for i, (a, b) in enumerate(zip(g, c)):
                    for f in FIELDS:
                        assert getattr(a, f) == getattr(b, f), f"{prefix}+{scored} {permission} step {i}: {f}"
                for name in ("membrane", "branches", "fatigue", "activation"):
                    assert np.array_equal(gpu.read_state(name), cpu.read_f32(name)), f"{permission}: {name}"
                assert np.array_equal(gpu.read_state("logits"), cpu.read_f32("logits"))
            cpu.finish_document()
            gpu.finish_document()
        losses = gpu.evaluate(texts)[1]
        for text, got in zip(texts, losses):
            cpu.begin_document()
            want = [cpu.step(s, t, oracle.FROZEN).loss for s, t in document(text)]
            cpu.finish_document()
            assert [float(v) for v in got] == want
        assert_models_equal(gpu.model(), cpu.model(), f"{workgroups} workgroups")
    finally:
        gpu.close()
