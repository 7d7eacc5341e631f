"""The host mirror's synchronisation against a whole-model download: change
sets from nothing to a few rows around the 32-row transpose tile, repeated
synchronisations, a tracking restart in between, and more changed rows than
one download carries (64 MiB)."""
from __future__ import annotations

import numpy as np
import pytest

from leo_amd import native
from leo_amd.config import Config
from leo_amd.config import test_toml_values as toml_values
from leo_amd.model import Model
from tests.helpers import assert_models_equal, small_redundant_config, story

pytestmark = pytest.mark.gpu


def test_mirror_follows_training(require_gpu):
    from leo_amd.runtime import HipRuntime

    cfg = small_redundant_config(neurons=1024, synapses=8, fanout=48, per_block=8)
    model = Model.synthetic(cfg, weight_sigma=0.05)
    mirror = model.copy()
    gpu = HipRuntime(model, device=0, max_lanes=3)
    try:
        gpu.synchronize_model(mirror)
        assert_models_equal(mirror, model, "nothing changed")
        text = story(9, 400)
        sizes = set()
        for i, steps in enumerate((1, 1, 1, 2, 3, 5, 8, 13, 40, 90)):
            if i == 5:
                gpu.enable_parameter_tracking()
            gpu.begin_document()
            gpu.training_step_batch(list(zip(text[i:i + steps], text[i + 1:])), native.TRAINING)
            sizes.add(len(gpu.parameter_changes()["output_neurons"]))
            gpu.synchronize_model(mirror)
            assert_models_equal(mirror, gpu.model(), f"after {steps} steps")
        assert min(sizes) < 32 < max(sizes)
        gpu.train_batch([story(k, 40 + 9 * k) for k in range(3)], native.TRAINING)
        gpu.synchronize_model(mirror)
        assert_models_equal(mirror, gpu.model(), "after a batch")
    finally:
        gpu.close()


def _every_neuron_fires() -> Model:
    """69,632 neurons whose output rows (68 MiB) all change in a learning step."""
    values = toml_values()
    n = 272 * 256
    values["model"].update(neuron_count=n, block_count=272, neurons_per_block=256, synapses_per_neuron=1,
                           input_fanout=n, max_active_per_block=256, max_active_global=n)
    values["dynamics"].update(target_activity=0.5)
    model = Model.empty(Config.from_dict(values))
    rng = np.random.default_rng(3)
    model.rec_target[:] = (np.arange(n) + 1) % n
    model.rec_delay[:] = 1
    model.rec_weight[:] = np.float32(0.01)
    model.excitability[:] = np.float32(1.0)
    model.out_weight[:] = rng.uniform(-0.1, 0.1, model.out_weight.size).astype(np.float32)
    model.in_target.reshape(258, n)[:] = np.arange(n)  # every symbol drives every neuron
    model.in_weight[:] = np.float32(1.0)
    model.threshold[:] = np.float32(0.3)
    model.validate()
    return model


def test_mirror_of_more_rows_than_one_download(require_gpu):
    from leo_amd.runtime import HipRuntime

    model = _every_neuron_fires()
    mirror = model.copy()
    gpu = HipRuntime(model, device=0, max_lanes=1)
    try:
        gpu.begin_document()
        assert gpu.step(65, 66, native.TRAINING).active_neurons * 257 * 4 > (64 << 20)
        gpu.synchronize_model(mirror)
        assert_models_equal(mirror, gpu.model(), "every row")
    finally:
        gpu.close()



def test_mirror_gives_scratch_back(require_gpu):
    """A synchronisation keeps at most 128 MiB of device memory for the next."""
    import ctypes

    from leo_amd.runtime import HipRuntime

    hip = ctypes.CDLL("libamdhip64.so")

    def free_bytes():
        free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    model = _every_neuron_fires()
    mirror = model.copy()
    gpu = HipRuntime(model, device=0, max_lanes=1)
    try:
        gpu.synchronize_model(mirror)
        gpu.begin_document()
        gpu.step(65, 66, native.TRAINING)
        before = free_bytes()
        gpu.synchronize_model(mirror)
        kept = before - free_bytes()
        print(f"{kept / 2**20:.0f} MiB kept", flush=True)
        assert kept <= 130 << 20
    finally:
        gpu.close()
