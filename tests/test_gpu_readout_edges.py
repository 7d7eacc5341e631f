"""The readout's context contribution at the edges of its loads against the
oracle: embeddings below, at and past a 16-dimension chunk, with rows that are
and are not whole 16-byte quarters, and the largest; documents learned (cells
appear and gain weight) and then scored frozen. Losses and the model bit for
bit."""
from __future__ import annotations

import numpy as np
import pytest

from leo_amd import native
from leo_amd.config import Config
from leo_amd.config import test_toml_values as toml_values
from leo_amd.model import BEGIN_DOCUMENT, END_DOCUMENT, Model
from tests.helpers import assert_models_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [1, 3, 4, 15, 16, 17, 20, 36, 64, 256])
def test_context_logits_match_oracle(require_gpu, oracle, dim):
    from leo_amd.runtime import HipRuntime

    values = toml_values()
    values["context"].update(embedding_dim=dim, max_order=6)
    model = Model.synthetic(Config.from_dict(values), weight_sigma=0.3)
    rng = np.random.default_rng(dim)
    model.ctx_out[:] = rng.uniform(-0.5, 0.5, model.ctx_out.size).astype(np.float32)
    model.validate()
    cpu = oracle.OracleRuntime(model)
    gpu = HipRuntime(model, device=0, max_lanes=1)
    text = b"abab abab acab."
    steps = list(zip([BEGIN_DOCUMENT] + list(text), list(text) + [END_DOCUMENT]))
    try:
        for permission in ("TRAINING", "TRAINING", "FROZEN"):
            cpu.begin_document()
            gpu.begin_document()
            for symbol, target in steps:
                c = cpu.step(symbol, target, getattr(oracle, permission))
                g = gpu.step(symbol, target, getattr(native, permission))
                assert (g.loss, g.predicted_symbol, g.context_cells) == (c.loss, c.predicted_symbol, c.context_cells)
            assert np.array_equal(gpu.read_state("logits"), cpu.read_f32("logits"))
            cpu.finish_document()
            gpu.finish_document()
        assert_models_equal(gpu.model(), cpu.model(), f"embedding {dim}")
    finally:
        gpu.close()
