"""Performance cases of Leo's per-byte step on one GPU: the work that a trainer,
an evaluator or a server has the backend do, through HipRuntime's public calls.

A case is a model shape (the benchmark's workloads A to D, an E-shaped
heavy-tailed model, and sizes between them) and one of seven paths:

  step      a line learned byte by byte, one `step` call per byte (online use)
  prompt    a frozen prompt (`advance_frozen_batch`), then one frozen step and
            the next byte's probabilities (serving)
  document  one document learned in place (`training_step_batch`)
  segment   one replay segment: reset, frozen prefix, supervised targets
  evaluate  a validation shard (`evaluate`)
  stories   a batch's story pass and its mean (`training_story_batch`)
  batch     a whole logical batch: story pass, mean and replay (`train_batch`)

Paths that learn also return what they learned: models of up to 2^17 neurons
through `synchronize_model` (the coordinator's host mirror), larger ones by the
losses of a short held-out line scored with the updated weights.

Every result of the framework is bit-identical to Leo's CPU executor, so
outputs are compared exactly; `exact` restates the step in 64 bits.
"""
from __future__ import annotations

import math
from typing import Dict, List

import numpy as np

from leo_amd import native
from leo_amd.config import Config
from leo_amd.model import BEGIN_DOCUMENT, END_DOCUMENT, Model
from leo_amd.runtime import HipRuntime
from leo_amd.workload import WORKLOADS, Workload, story_list, synthetic_stories, workload_config

LEARNED = ("threshold", "rec_weight", "in_weight", "out_weight", "bias", "ctx_keys", "ctx_emb", "ctx_obs", "ctx_out")
MIRROR_NEURONS = 1 << 17   # larger models are checked by a probe line instead of a host mirror
PROBE = b"the cat sat on the mat and\n"
TOPOLOGIES = {"uniform": native.TOPOLOGY_UNIFORM, "power_law": native.TOPOLOGY_POWER_LAW,
              "heavy_tail": native.TOPOLOGY_HEAVY_TAIL}


def _shape(letter: str) -> Dict[str, object]:
    w = WORKLOADS[letter]
    topology = {v: k for k, v in TOPOLOGIES.items()}[w.topology]
    return {"neurons": w.neurons, "block": 256, "fan_in": w.synapses, "fanout": w.fanout, "per_block": w.per_block,
            "cap": w.global_cap, "activity": w.target_activity, "topology": topology}


def _case(name: str, letter: str, path: str, stories: int, length: int, **more) -> Dict[str, object]:
    return {"name": name, "path": path, **_shape(letter), "stories": stories, "length": length, "prefix": 0,
            "replay_segment": 32, "stateful": False, **more}


# E's irregular shape (heavy-tailed in-degree, 30% activity, 80 winners per
# block) at a size whose host model is made in about a second.
_HEAVY = {"neurons": 65_536, "fan_in": 32, "fanout": 256, "per_block": 80, "cap": 20_480, "activity": 0.30,
          "topology": "heavy_tail"}


def listed() -> List[Dict[str, object]]:
    return [
        # the smallest calls: launch and host latency of one step at a time, as
        # an interactive user's program makes them
        _case("step_A", "A", "step", 1, 24),
        # one whole logical batch of the probe configuration: in-place document and replay
        _case("batch_A", "A", "batch", 1, 640),
        # a document learned in place, the coordinator's single-story path
        _case("document_B", "B", "document", 1, 200),
        # a validation shard of ordinary stories
        _case("evaluate_B", "B", "evaluate", 8, 800),
        # the ordinary training batch: 8 lanes, mean, classic replay
        _case("batch_B", "B", "batch", 8, 800),
        # prompt ingestion on a power-law model (hub targets receive many events)
        _case("prompt_C", "C", "prompt", 1, 400),
        # validation on the power-law model, more lanes than XCDs
        _case("evaluate_C", "C", "evaluate", 32, 120),
        # the story pass alone with 32 lanes: the batch-parallel half of training
        _case("stories_C", "C", "stories", 32, 96),
        # dense activity and hub targets (large delivery buckets)
        _case("stories_heavy", "E", "stories", 13, 48, **_HEAVY),
        # the serial half of training at a million neurons: one replay segment
        # behind the mean prefix of an 800-byte story
        _case("segment_D", "D", "segment", 1, 32, prefix=470),
        # a whole batch at a million neurons, short stories
        _case("batch_D", "D", "batch", 8, 128),
    ]


def draw(rng) -> Dict[str, object]:
    """A case of the same ranges: any path, sizes spread over their logarithm."""
    path = rng.choice(("step", "prompt", "document", "segment", "evaluate", "stories", "batch"))
    block = rng.choice((256, 256, 128, 200, 512, 96))
    blocks = max(4, int(round(math.exp(rng.uniform(math.log(1024), math.log(400_000))) / block)))
    neurons = blocks * block
    fan_in = rng.choice((8, 16, 24, 32, 37, 48, 64))
    fanout = int(round(math.exp(rng.uniform(math.log(48), math.log(512)))))
    per_block = rng.choice((2, 4, 8, 13, 16))
    # most configurations let every block winner through; some cap the whole
    cap = blocks * per_block if rng.random() < 0.8 else max(8, blocks * per_block // 2)
    activity = min(rng.choice((0.01, 0.02, 0.05)), 0.9 * cap / neurons)
    topology = rng.choice(("uniform", "uniform", "power_law", "heavy_tail"))
    serial = path in ("step", "prompt", "document", "segment")
    stories = 1 if serial else rng.choice((1, 2, 3, 5, 8, 11, 16)) if path != "stories" else rng.choice((2, 3, 7, 12, 24))
    longest = {"step": 40, "prompt": 700, "document": 300, "segment": 48, "evaluate": 400, "stories": 120, "batch": 200}
    length = int(round(math.exp(rng.uniform(math.log(8), math.log(longest[path])))))
    prefix = int(round(math.exp(rng.uniform(math.log(4), math.log(700))))) if path == "segment" else 0
    return {"path": path, "neurons": neurons, "block": block, "fan_in": fan_in, "fanout": fanout,
            "per_block": per_block, "cap": cap, "activity": activity, "topology": topology, "stories": stories,
            "length": length, "prefix": prefix, "replay_segment": rng.choice((8, 32, 64)),
            "stateful": rng.random() < 0.25}


# --- inputs -------------------------------------------------------------------
def _lengths(case) -> List[int]:
    """The texts' lengths, from the case alone: ragged around its length where there are several."""
    if case["path"] == "segment":
        return [case["prefix"] + case["length"]]
    if case["stories"] == 1:
        return [case["length"]]
    return [max(2, round(case["length"] * (0.5 + (0.618034 * (i + 1)) % 1.0))) for i in range(case["stories"])]


def _texts(case, seed: int) -> List[bytes]:
    """Zipf-ASCII stories of the seed, cut to the case's lengths."""
    lengths = _lengths(case)
    longest = max(lengths)
    source = Workload("text", seed & 0xFFFFFFFF, 0, 0, 0, 0, 0.0, 0, 0, 0, float(4 * longest + 64), 0.0, 64,
                      4 * longest + 128, native.TOPOLOGY_UNIFORM)
    return [text[:n] for text, n in zip(story_list(*synthetic_stories(source, len(lengths))), lengths)]


def _config(case) -> Config:
    base = workload_config(WORKLOADS["A"]).to_dict()
    base["model"].update(name="Leo-case", neuron_count=case["neurons"], block_count=case["neurons"] // case["block"],
                         neurons_per_block=case["block"], synapses_per_neuron=case["fan_in"],
                         input_fanout=case["fanout"], max_active_per_block=case["per_block"],
                         max_active_global=case["cap"])
    base["dynamics"].update(target_activity=case["activity"])
    base["replay"].update(segment_bytes=case["replay_segment"], stateful_batch=case["stateful"])
    return Config.from_dict(base)


# The model is the configuration's seeded synthetic one: like a checkpoint, the
# same for every input. Making a million-neuron model takes ten seconds of host
# time, so the last configuration's is kept for the next preparation.
_last_model: Dict[str, object] = {}


def _model(case) -> Model:
    config = _config(case)
    key = (repr(config), case["topology"])
    if _last_model.get("key") != key:
        _last_model.clear()
        exponent = {"uniform": 0.0, "power_law": 2.1, "heavy_tail": 1.1}[case["topology"]]
        cap = min(4096, case["neurons"] // 4) if case["topology"] == "heavy_tail" else 0
        _last_model.update(key=key, model=Model.synthetic(config, topology=TOPOLOGIES[case["topology"]],
                                                          exponent=exponent, in_degree_cap=cap, weight_sigma=0.05))
    return _last_model["model"]


def _document(text: bytes):
    """training.rs:1747-1757: BEGIN, the bytes, each with the next one (END last) as its target."""
    symbols = [BEGIN_DOCUMENT] + list(text)
    return list(zip(symbols, list(text) + [END_DOCUMENT]))


def prepare(case, seed: int):
    model = _model(case)
    lanes = case["stories"] if case["path"] in ("evaluate", "stories", "batch") else 1
    runtime = HipRuntime(model, device=0, max_lanes=lanes)
    state = {"case": case, "runtime": runtime, "texts": _texts(case, seed), "mirror": None}
    if case["path"] in ("step", "document", "stories", "batch") and case["neurons"] <= MIRROR_NEURONS:
        # the coordinator's host mirror: its own copy of what training changes
        state["mirror"] = Model(config=model.config, **{
            name: getattr(model, name).copy() if name in LEARNED else getattr(model, name)
            for name in Model.shapes(model.config)})
    return state


# --- one pass -----------------------------------------------------------------
def _learned(state):
    """What the pass learned: the updated host mirror, or a probe line's losses."""
    if state["mirror"] is not None:
        state["runtime"].synchronize_model(state["mirror"])
        return {name: getattr(state["mirror"], name) for name in LEARNED}
    return {"probe_losses": state["runtime"].evaluate([PROBE])[1][0]}


def _counts(report) -> Dict[str, int]:
    return {k: int(getattr(report, k)) for k in ("targets", "replay_segments", "replay_steps", "replay_prefix_steps",
                                                 "merge_fixed_parameter_updates", "merge_context_keys",
                                                 "active_neurons_sum", "emitted_events")}


def run(state):
    case, rt, texts = state["case"], state["runtime"], state["texts"]
    path = case["path"]
    if path == "step":
        rt.begin_document()
        losses = [rt.step(symbol, target, native.TRAINING).loss for symbol, target in _document(texts[0])]
        probabilities = rt.probabilities()
        rt.finish_document()
        return {"losses": np.array(losses, dtype=np.float32), "probabilities": probabilities,
                "learned": _learned(state)}
    if path == "prompt":
        rt.begin_document()
        rt.advance_frozen_batch([(BEGIN_DOCUMENT, None)] + [(b, None) for b in texts[0][:-1]])
        predicted = rt.step(texts[0][-1], None, native.FROZEN).predicted_symbol
        return {"probabilities": rt.probabilities(), "logits": rt.read_state("logits"), "predicted": predicted}
    if path == "document":
        rt.begin_document()
        metrics = rt.training_step_batch(_document(texts[0]), native.TRAINING)
        rt.finish_document()
        return {"losses": np.array([m.loss for m in metrics], dtype=np.float32),
                "active": np.array([m.active_neurons for m in metrics]), "learned": _learned(state)}
    if path == "segment":
        steps = _document(texts[0])
        at = case["prefix"]
        rt.begin_document()
        rt.advance_frozen_batch([(symbol, None) for symbol, _ in steps[:at]])
        metrics = rt.training_step_batch(steps[at:], native.TRAINING)
        probabilities = rt.probabilities()
        rt.finish_document()
        return {"losses": np.array([m.loss for m in metrics], dtype=np.float32),
                "active": np.array([m.active_neurons for m in metrics]), "probabilities": probabilities,
                "learned": _learned(state)}
    if path == "evaluate":
        report, losses = rt.evaluate(texts)
        return {"losses": np.concatenate(losses), "loss": report["loss"], "accuracy": report["accuracy"],
                "active_sum": int(report["active_neurons_sum"]), "events": int(report["emitted_events"])}
    if path == "stories":
        report, losses = rt.training_story_batch(texts, native.TRAINING)
    else:
        report, losses = rt.train_batch(texts, native.TRAINING, replay=True)
    return {"losses": np.concatenate(losses), "counts": _counts(report), "learned": _learned(state)}


# --- what a pass cannot do without ---------------------------------------------
def _steps(case):
    """(frozen, scored, learned) steps of a pass, about."""
    n = case["length"] + 1
    path = case["path"]
    if path == "prompt":
        return n - 1, 1, 0
    if path == "segment":
        return case["prefix"], len(PROBE), n
    if path == "evaluate":
        return 0, n * case["stories"], 0
    replayed, segments = 0.0, 0.0
    if path == "batch":
        replayed = 0.3 * n
        segments = 1.0 if case["stateful"] else max(1.0, replayed / case["replay_segment"])
    probe = len(PROBE) if case["neurons"] > MIRROR_NEURONS else 0
    return case["stories"] * segments * n / 2, probe, case["stories"] * (n + replayed)


def work(case):
    """Bytes and operations of one pass, each element that a step touches once (read, and written where it changes).

    A step injects F edges (9 B each) into as many neurons (state read and written 96 B, threshold and excitability
    8 B) and delivers about as many recurrent events again (13 B and a neuron each); about one neuron in
    twenty injected ones fires (S synapses of 8 B). A scored step reads the firing neurons' 257 output weights; a learning
    step also writes them and brings up the traces of the slots that delivered within the last few ticks (64 B each)."""
    F, S = case["fanout"], case["fan_in"]
    fire = max(1.0, min(F / 20.0, case["cap"]))
    frozen, scored, learned = _steps(case)
    sparse = F * 9 + 2 * F * 104 + fire * S * (13 + 8)
    readout = fire * 1028 + 257 * 12
    learning = 3 * fire * 1028 + 8 * (F + fire * S) * 64
    steps = frozen + scored + learned
    data = steps * sparse + (scored + learned) * readout + learned * learning
    flops = steps * (2 * F * 30 + 2 * fire * S) + (scored + learned) * (2 * 257 * fire + 257 * 6)
    flops += learned * (4 * 257 * fire + 8 * (F + fire * S) * 30)
    return {"bytes": data, "flops": flops}


def tolerance(case):
    """Exact: the framework's contract is the CPU executor's bits (a top-k winner that flips on a changed rounding
    changes everything after it)."""
    return "exact"


# --- the same in 64 bits --------------------------------------------------------
class _Exact:
    """Leo's step in float64 numpy, by its equations (sums in any order)."""

    def __init__(self, model: Model, learns: bool):
        config = model.config
        f = lambda v: float(np.float32(v))  # noqa: E731  (the configuration holds 32-bit values)
        self.config = config
        dyn, lrn, ctx = config.dynamics, config.learning, config.context
        self.N, self.S, self.F = config.model.neuron_count, config.model.synapses_per_neuron, config.model.input_fanout
        self.nb, self.E = config.model.neurons_per_block, ctx.embedding_dim
        self.decay = np.array([f(dyn.branch_decay), f(dyn.membrane_decay), f(dyn.fatigue_decay),
                               f(dyn.adaptation_fast_decay), f(dyn.adaptation_medium_decay),
                               f(dyn.adaptation_slow_decay)])
        self.gain = np.array([f(dyn.fatigue_gain), f(dyn.adaptation_fast_gain), f(dyn.adaptation_medium_gain),
                              f(dyn.adaptation_slow_gain)])
        self.dyn = {k: f(getattr(dyn, k)) for k in ("target_activity", "population_inhibition_rate",
                                                    "population_inhibition_max", "membrane_reset_fraction",
                                                    "threshold_homeostasis_rate")}
        self.lrn = {k: f(getattr(lrn, k)) for k in ("output_learning_rate", "recurrent_learning_rate",
                                                    "inhibitory_learning_rate", "eligibility_decay",
                                                    "eligibility_epsilon", "surrogate_width", "surrogate_gain",
                                                    "max_update", "weight_min", "weight_max", "training_strength",
                                                    "end_document_weight")}
        self.ctx_lr, self.confidence = f(ctx.learning_rate), float(ctx.confidence_observations)
        wide = (lambda a: a.astype(np.float64)) if learns else (lambda a: a)
        self.thr, self.rw, self.iw = wide(model.threshold), wide(model.rec_weight), wide(model.in_weight)
        self.ow = wide(model.out_weight).reshape(257, self.N)
        self.bias = model.bias.astype(np.float64)
        self.keys, self.obs = model.ctx_keys.copy(), model.ctx_obs.copy()
        self.emb = model.ctx_emb.astype(np.float64).reshape(-1, self.E)
        self.proj = model.ctx_out.astype(np.float64).reshape(257, self.E)
        self.exc, self.kind = model.excitability, model.neuron_type
        self.rt, self.rb, self.rd = model.rec_target, model.rec_branch, np.maximum(model.rec_delay, 1)
        self.it, self.ib = model.in_target, model.in_branch
        self.tick = 0
        self.reset()

    def reset(self):
        n, ns, ni = self.N, self.N * self.S, 258 * self.F
        self.state = np.zeros((n, 9))       # branches 0-3, membrane, fatigue, adaptation 0-2
        self.last = np.full(n, self.tick)
        self.act = np.zeros(n)
        self.refractory = np.zeros(n, dtype=np.int64)
        self.active = np.zeros(0, dtype=np.int64)
        self.due: Dict[int, list] = {}
        self.traces = {}                    # made by the first learning step
        self.trace_sizes = (ns, ni)
        self.listed = [np.zeros(0, dtype=np.int64), np.zeros(0, dtype=np.int64)]
        self.history: List[int] = []
        self.pi, self.phase = 0.0, 0

    def _bring(self, rows, last, idx):
        k = (self.tick - last[idx])[:, None].astype(np.float64)
        cols = np.array([0, 0, 0, 0, 1, 2, 3, 4, 5]) if rows.shape[1] == 9 else np.arange(6)
        rows[idx, : len(cols)] *= self.decay[cols] ** k
        last[idx] = self.tick

    def _activate(self, which, slots, pre):
        if which not in self.traces:        # branch, membrane, fatigue, adaptation 0-2, eligibility
            size = self.trace_sizes[which]
            self.traces[which] = (np.zeros((size, 7)), np.full(size, self.tick), np.zeros(size, dtype=bool))
        rows, last, mark = self.traces[which]
        self._bring(rows, last, slots)
        rows[slots, 0] += pre
        self.listed[which] = np.concatenate([self.listed[which], slots[~mark[slots]]])
        mark[slots] = True

    def _context(self, symbol, allocate, enabled):
        ctx = self.config.context
        self.history = (self.history + [symbol])[-ctx.max_order:]
        slots, scales = [], []
        for order in range(1, len(self.history) + 1) if enabled else ():
            h = 0xCBF29CE484222325 ^ order
            for s in self.history[-order:]:
                for b in range(4):
                    h = ((h ^ ((s >> (8 * b)) & 0xFF)) * 0x100000001B3) & 0xFFFFFFFFFFFFFFFF
            key, spo = max(h, 1), ctx.slots_per_order
            window = [(order - 1) * spo + (key % spo + off) % spo for off in range(ctx.probe_limit)]
            slot = next((s for s in window if int(self.keys[s]) == key), None)
            if slot is None:
                if not allocate:
                    continue
                slot = next((s for s in window if self.keys[s] == 0), min(window, key=lambda s: int(self.obs[s])))
                self.keys[slot], self.obs[slot], self.emb[slot] = key, 0, 0.0
            seen = float(self.obs[slot])
            slots.append(slot)
            scales.append(seen / (seen + self.confidence) * order)
        total = sum(scales)
        return slots, [s / total for s in scales] if total > 0 else scales

    def step(self, symbol, target, learn):
        """One step; (loss or None, probabilities)."""
        t, d, l = self.tick, self.dyn, self.lrn
        events = self.due.pop(t, [])
        rec = np.concatenate([e[0] for e in events]) if events else np.zeros(0, dtype=np.int64)
        pre = np.concatenate([e[1] for e in events]) if events else np.zeros(0)
        value = np.concatenate([e[2] for e in events]) if events else np.zeros(0)
        inj = symbol * self.F + np.arange(self.F)
        touched = np.unique(np.concatenate([self.active, self.rt[rec].astype(np.int64), self.it[inj].astype(np.int64)]))
        self.act[self.active] = 0.0
        self._bring(self.state, self.last, touched)
        np.add.at(self.state, (self.rt[rec].astype(np.int64), self.rb[rec]), value)
        np.add.at(self.state, (self.it[inj].astype(np.int64), self.ib[inj]), self.iw[inj].astype(np.float64))
        if learn:
            self._activate(0, rec, pre)
            self._activate(1, inj, 1.0)
        enabled = not learn or _survives(self.config.model.seed, t, symbol, self.config.context.dropout_rate)
        slots, scales = self._context(symbol, learn and enabled, enabled)
        # drive and selection
        live = touched[self.refractory[touched] <= t]
        s = self.state[live]
        net = s[:, 0] + s[:, 2] * np.clip(s[:, 3], 0.0, 1.0) + s[:, 1]
        self.state[live, 4] += self.exc[live].astype(np.float64) * net - s[:, 5] - s[:, 6:9].sum(1) - self.pi
        margin = self.state[live, 4] - self.thr[live]
        cand, act = live[margin > 0], np.clip(margin[margin > 0], 0.0, 1.0)
        tie = (cand + self.N - t % self.N) % self.N
        order = np.lexsort((tie, -act, cand // self.nb))
        cand, act, tie = cand[order], act[order], tie[order]
        blocks, first = np.unique(cand // self.nb, return_index=True)
        rank = np.arange(len(cand)) - first[np.searchsorted(blocks, cand // self.nb)] if len(cand) else np.zeros(0, int)
        limit, cap = self.config.model.max_active_per_block, self.config.model.max_active_global
        cutoff = dict(zip((cand // self.nb)[rank == limit], act[rank == limit]))
        win, wact, wtie = cand[rank < limit], act[rank < limit], tie[rank < limit]
        pop_cutoff = 0.0
        if cap < (self.N // self.nb) * limit:
            order = np.lexsort((wtie, -wact))
            win, wact = win[order], wact[order]
            if len(win) > cap:
                n = win[cap]
                pop_cutoff = min(max(self.state[n, 4] - self.thr[n], 0.0), d["population_inhibition_max"])
                win, wact = win[:cap], wact[:cap]
        self.active = win
        self.act[win] = wact
        activity = len(win) / self.N - d["target_activity"]
        self.pi = min(max(self.pi + d["population_inhibition_rate"] * activity, 0.0), d["population_inhibition_max"])
        if learn:
            is_touched, selected = np.zeros(self.N, dtype=bool), np.zeros(self.N, dtype=bool)
            is_touched[touched], selected[win] = True, True
            cuts = np.zeros(self.N // self.nb)
            for b, v in cutoff.items():
                cuts[b] = v
            self._eligibility(is_touched, selected, np.maximum(cuts, pop_cutoff))
        # post-activation state and emission
        self.state[win, 5:9] += wact[:, None] * self.gain
        self.state[win, 4] -= self.thr[win] * d["membrane_reset_fraction"]
        self.refractory[win] = t + self.config.dynamics.refractory_ticks + 1
        out = (win[:, None] * self.S + np.arange(self.S)).reshape(-1)
        source = np.repeat(wact, self.S)
        emitted = source * self.rw[out]
        for delay in (1, 2, 4, 8):
            m = self.rd[out] == delay
            self.due.setdefault(t + delay, []).append((out[m], source[m], emitted[m]))
        # readout
        logits = self.bias + self.ow[:, win].astype(np.float64) @ wact
        latent = sum((self.emb[k] * w for k, w in zip(slots, scales) if w > 0), np.zeros(self.E))
        if slots:
            logits = logits + self.proj @ latent
        self.logits = logits
        p = np.exp(logits - logits.max())
        p /= p.sum()
        index = None if target is None else min(target, 257) - (target == END_DOCUMENT)
        loss = None if index is None else -math.log(max(p[index], 1e-12))
        if learn and index is not None:
            self._learn(p, index, win, wact, slots, scales, latent, enabled)
        if learn:
            local = (self.act[touched] > 0) - d["target_activity"]
            self.thr[touched] = np.clip(self.thr[touched] + d["threshold_homeostasis_rate"] * (local + activity),
                                        0.05, 2.0)
        self.tick += 1
        return loss, p

    def _eligibility(self, touched, selected, cuts):
        l = self.lrn
        for which, targets, branches in ((0, self.rt, self.rb), (1, self.it, self.ib)):
            slots = self.listed[which]
            rows, last, mark = self.traces[which]
            self._bring(rows, last, slots)
            r, dst = rows[slots], targets[slots].astype(np.int64)
            open_ = touched[dst] & (self.refractory[dst] <= self.tick)
            r[~open_, 6] *= l["eligibility_decay"]
            o, n = r[open_], dst[open_]
            br, exc, s = branches[slots][open_], self.exc[n].astype(np.float64), self.state[n]
            inside = (s[:, 3] > 0) & (s[:, 3] < 1)
            jac = np.where(br == 2, exc * np.clip(s[:, 3], 0, 1), np.where(br == 3, exc * s[:, 2] * inside, exc))
            margin = s[:, 4] - self.thr[n]
            direct = selected[n] & (margin > 0) & (margin < 1)
            near = np.clip(1 - np.abs(margin - cuts[n // self.nb]) / l["surrogate_width"], 0, 1)
            o[:, 1] += jac * o[:, 0] - o[:, 2] - o[:, 3:6].sum(1)
            o[:, 6] = (direct + l["surrogate_gain"] * near) * o[:, 1]
            r[open_] = o
            won = touched[dst] & selected[dst]
            r[won, 2:6] += r[won, 6:7] * self.gain
            rows[slots] = r
            keep = np.abs(r).max(1) > l["eligibility_epsilon"] if len(r) else np.zeros(0, dtype=bool)
            mark[slots[~keep]] = False
            self.listed[which] = slots[keep]

    def _learn(self, p, index, win, wact, slots, scales, latent, enabled):
        l, d = self.lrn, self.dyn
        mu, lo, hi = l["max_update"], l["weight_min"], l["weight_max"]
        err = p.copy()
        err[index] -= 1.0
        strength = l["training_strength"] * (l["end_document_weight"] if index == 256 else 1.0)
        window = self.config.learning.plasticity_window
        size = min(self.phase, window - 1) + 1
        scale, self.phase = (float(size), 0) if size == window or index == 256 else (0.0, size)
        recs, ins = self.listed
        if scale > 0:
            dst = np.unique(np.concatenate([self.rt[recs], self.it[ins]])).astype(np.int64)
            signal = np.zeros(self.N)
            signal[dst] = err @ self.ow[:, dst]
        bounded = lambda v: np.clip(v, -mu, mu)  # noqa: E731
        olr = l["output_learning_rate"] * strength
        self.ow[:, win] = np.clip(self.ow[:, win] + bounded(-olr * err[:, None] * wact[None, :]), lo, hi)
        self.bias += bounded(-olr * err)
        if enabled and slots:
            gradient = err @ self.proj
            clr = self.ctx_lr * strength
            self.proj = np.clip(self.proj + bounded(-clr * err[:, None] * latent[None, :]), lo, hi)
            for k, w in zip(slots, scales):
                self.emb[k] = np.clip(self.emb[k] + bounded(-clr * w * gradient), lo, hi)
                self.obs[k] += 1
        if scale > 0:
            rate = l["recurrent_learning_rate"] * strength * scale
            for which, sl, targets, weights in ((0, recs, self.rt, self.rw), (1, ins, self.it, self.iw)):
                e = self.traces[which][0][sl, 6]
                w = weights[sl] + bounded(-rate * signal[targets[sl].astype(np.int64)] * e)
                if which == 1:
                    weights[sl] = np.clip(w, 0.0, hi)
                else:
                    w, excitatory = np.clip(w, lo, hi), self.kind[sl // self.S] == 0
                    weights[sl] = np.where(excitatory, np.maximum(w, 0.0), np.minimum(w, 0.0))
        inhibitory = self.kind[win] != 0
        sl = (win[inhibitory][:, None] * self.S + np.arange(self.S)).reshape(-1)
        fired = (self.act[self.rt[sl].astype(np.int64)] > 0) - d["target_activity"]
        delta = bounded(-l["inhibitory_learning_rate"] * l["training_strength"] * np.repeat(wact[inhibitory], self.S) * fired)
        self.rw[sl] = np.clip(self.rw[sl] + delta, lo, 0.0)

    def document(self, text, learn=True):
        self.reset()
        return [self.step(symbol, target, learn)[0] for symbol, target in _document(text)]

    def learned(self):
        values = (self.thr, self.rw, self.iw, self.ow, self.bias, self.emb, self.proj)
        names = ("threshold", "rec_weight", "in_weight", "out_weight", "bias", "ctx_emb", "ctx_out")
        return {**{k: None for k in LEARNED}, **{n: np.asarray(v, dtype=np.float64).reshape(-1) for n, v in zip(names, values)}}


def _survives(seed, tick, symbol, rate) -> bool:
    """runtime.rs:103-116: the context's dropout draw."""
    if rate <= 0.0:
        return True
    m = 0xFFFFFFFFFFFFFFFF
    v = (seed ^ (tick * 0x9E3779B97F4A7C15) ^ (symbol * 0xBF58476D1CE4E5B9)) & m
    v = ((v ^ (v >> 30)) * 0xBF58476D1CE4E5B9) & m
    v = ((v ^ (v >> 27)) * 0x94D049BB133111EB) & m
    v ^= v >> 31
    return (v >> 40) / float(1 << 24) >= float(np.float32(rate))


def exact(case, seed: int):
    path = case["path"]
    if path in ("stories", "batch"):  # many learning lanes, or a replay: minutes in numpy
        return None
    frozen, scored, learned = _steps(case)
    dense = case["activity"] >= 0.1 or case["neurons"] * case["fan_in"] > 80_000_000
    if (frozen + scored) * 0.002 + learned * (0.1 if dense else 0.02) > 15.0:
        return None
    sim = _Exact(_model(case), learns=path != "prompt" and path != "evaluate")
    text = _texts(case, seed)[0]
    if path == "evaluate":
        losses = []
        for story in _texts(case, seed):
            losses += sim.document(story, learn=False)
        return {"losses": np.array(losses), "loss": float(np.mean(losses)), "accuracy": None, "active_sum": None,
                "events": None}
    if path == "prompt":
        for symbol in [BEGIN_DOCUMENT] + list(text[:-1]):
            sim.step(symbol, None, False)
        _, p = sim.step(text[-1], None, False)
        return {"probabilities": p, "logits": sim.logits, "predicted": None}
    losses = []
    for i, (symbol, target) in enumerate(_document(text)):
        learn = i >= case["prefix"]
        loss, p = sim.step(symbol, target if learn else None, learn)
        losses += [loss] if learn else []
    if path != "segment" and case["neurons"] <= MIRROR_NEURONS:
        learned = sim.learned()
    else:
        learned = {"probe_losses": np.array(sim.document(PROBE, learn=False))}
    result = {"losses": np.array(losses), "probabilities": p, "active": None, "learned": learned}
    return {k: v for k, v in result.items() if k != {"step": "active", "document": "probabilities"}.get(path)}
