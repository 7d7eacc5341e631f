"""Deep delivery buckets of exact sizes against the oracle: one input row
sends `count` edges to one neuron, so that its bucket holds that many entries
in one tick, at the edges of the entries a lane ranks (64, 128, 256) and past
them (the radix sort). The sums are in delivery order, so they are compared
bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from leo_amd import native
from leo_amd.model import Model
from tests.helpers import small_redundant_config

pytestmark = pytest.mark.gpu

COUNTS = (8, 9, 63, 64, 65, 127, 128, 129, 191, 193, 255, 256, 257, 511)
HUB = 77


def _model():
    cfg = small_redundant_config(neurons=1024, synapses=8, fanout=512, per_block=8, dropout=0.0)
    cfg.validate()
    model = Model.synthetic(cfg, weight_sigma=0.05)
    rng = np.random.default_rng(5)
    rows = model.in_target.reshape(258, 512)
    for symbol, count in enumerate(COUNTS):
        others = rng.permutation([n for n in range(1024) if n != HUB])[: 512 - count]
        rows[symbol] = rng.permutation(np.concatenate([np.full(count, HUB), others]))
    model.in_weight[:] = rng.uniform(0.0, 1.0, model.in_weight.size).astype(np.float32)
    model.validate()
    return model


@pytest.mark.parametrize("permission", ["frozen", "training"])
def test_bucket_sizes_match_oracle(require_gpu, oracle, permission):
    from leo_amd.runtime import HipRuntime

    model = _model()
    cpu = oracle.OracleRuntime(model)
    gpu = HipRuntime(model, device=0, max_lanes=1)
    frozen = permission == "frozen"
    try:
        for symbol, count in enumerate(COUNTS):
            cpu.begin_document()
            gpu.begin_document()
            for sym in (symbol, 200, symbol):  # with recurrent deliveries beside the row the third time
                cpu.step(sym, 65, oracle.FROZEN if frozen else oracle.TRAINING)
                gpu.step(sym, 65, native.FROZEN if frozen else native.TRAINING)
            for name in ("branches", "membrane"):
                got, want = gpu.read_state(name), cpu.read_f32(name)
                assert np.array_equal(got, want), f"{count} entries: {name}"
        stats = gpu.kernel_stats()
        assert stats["deep_register_folds"] > 0 and stats["deep_radix_folds"] > 0
    finally:
        gpu.close()
