"""The calls a user of the engine makes, as measurable cases: decode steps of ragged batches, shared-prefix rollouts,
steps that mix decode rows with a portion of a prompt, and prompts, on quantised GGUF models and on bf16 layer-stack
models. Every case goes through `Engine.step` and `Engine.step_logits`; a pass is what a server or a rollout loop does
between two looks at its queue: it takes back what the last pass appended (`seq_rm`), runs its steps and reads tokens,
log-probabilities and logits.

Shapes are those of retrograd_amd/synth.py and retrograd_amd/bench_stack.py at a depth at which a model is made and
loaded in a second or two; layers repeat, so a step's cost per layer is that of the full depth. Weights are a fixed
checkpoint per model, as a user's are; prompts, context lengths and adapter routes come from the seed. Several states
of one model share its engine while it has free slots, each in slots of its own, as the sequences of a server do."""

from __future__ import annotations

import json
import math
import mmap
import os
import struct
import tempfile
from pathlib import Path

import numpy as np
import torch

from retrograd_amd import bench_stack, engine as E, synth, synth_stack

SLOTS = 256              # of an engine, the most that it takes
LORA_RANK, LORA_COUNT = 16, 8

# name: (shape or configuration, KV cells of an engine, n_batch)
MODELS = {
    "tiny": (synth.TINY_LLAMA, 64 * 128, 512),
    "llama": (bench_stack.llama_shape("w4096"), 440_000, 2048),
    "qwen2": (synth.scaled(synth.QWEN25_7B_Q8, n_layer=4, n_vocab=32000, name="qwen2.5-7b-shape-q8_0-4layers"), 300_000, 512),
    "qwen3moe": (synth.scaled(synth.QWEN3_30B_A3B, n_layer=4, n_vocab=32000, name="qwen3-30b-a3b-shape-mxfp4-4layers"), 260_000, 2048),
    "pomisun": (bench_stack.pomisun_config("w2048"), 300_000, 4096),
    "dibosun": (bench_stack.dibosun_config("w2048"), 60_000, 4096),
}


def listed():
    return [
        # the smallest step: a two-layer test model, eight short conversations; launches and host time are all there is
        {"name": "tiny_decode", "kind": "decode", "model": "tiny", "kv": "f16", "rows": 8, "lo": 8, "hi": 64, "steps": 8},
        # one user waiting for the next token of a chat
        {"name": "llama_decode_1", "kind": "decode", "model": "llama", "kv": "f16", "rows": 1, "lo": 500, "hi": 1100, "steps": 8},
        # a busy server's decode step: 64 sequences of very different lengths
        {"name": "llama_decode_64", "kind": "decode", "model": "llama", "kv": "f16", "rows": 64, "lo": 128, "hi": 4096, "steps": 8},
        # GRPO rollouts: 32 prompts over one system prompt, each continued eight times from shared pages
        {"name": "llama_rollout_256", "kind": "rollout", "model": "llama", "kv": "f16", "rows": 32, "samples": 8, "prefix": 2048, "lo": 32, "hi": 512, "steps": 4},
        # continuous batching on a Q8_0 cache: decode rows and a newcomer's portion of a prompt in one step
        {"name": "llama_mixed_q8kv", "kind": "mixed", "model": "llama", "kv": "q8_0", "rows": 48, "lo": 128, "hi": 2048, "chunk": 397, "at": 512},
        # a long document's prompt
        {"name": "llama_prefill_4001", "kind": "prefill", "model": "llama", "kv": "f16", "rows": 1, "lo": 4001, "hi": 4001, "scored": 32},
        # several fine-tunes served at once: rows of one step routed to eight adapters or the base
        {"name": "qwen2_lora_decode_64", "kind": "decode", "model": "qwen2", "kv": "f16", "rows": 64, "lo": 256, "hi": 2048, "steps": 8},
        # mixture of experts, decode: every expert is touched
        {"name": "qwen3moe_decode_128", "kind": "decode", "model": "qwen3moe", "kv": "f16", "rows": 128, "lo": 64, "hi": 2048, "steps": 4},
        # mixture of experts, admission of a few prompts at once
        {"name": "qwen3moe_prefill", "kind": "prefill", "model": "qwen3moe", "kv": "f16", "rows": 3, "lo": 300, "hi": 1000, "scored": 16},
        # bf16 layer-stack models: decode of a batch ...
        {"name": "pomisun_decode_64", "kind": "decode", "model": "pomisun", "kv": "f16", "rows": 64, "lo": 128, "hi": 2048, "steps": 8},
        # ... a long prompt through attention, dense and expert feed-forwards
        {"name": "pomisun_prefill_3900", "kind": "prefill", "model": "pomisun", "kv": "f16", "rows": 1, "lo": 3900, "hi": 3900, "scored": 32},
        # ... and several prompts through latent attention and Mamba-2
        {"name": "dibosun_prefill", "kind": "prefill", "model": "dibosun", "kv": "f16", "rows": 5, "lo": 200, "hi": 1500, "scored": 16},
    ]


def draw(rng):
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["tiny", "decode", "decode", "lora", "moe", "rollout", "mixed", "prefill", "moe_prefill", "stack_decode", "stack_prefill", "dibosun"])
    kv = rng.choice(["f16", "f16", "q8_0"])
    if kind == "tiny":
        return {"kind": "decode", "model": "tiny", "kv": kv, "rows": rng.randint(1, 8), "lo": 8, "hi": 64, "steps": 8}
    if kind == "decode":
        return {"kind": "decode", "model": "llama", "kv": kv, "rows": log(1, 64), "lo": log(32, 512), "hi": log(512, 4096), "steps": 8}
    if kind == "lora":
        return {"kind": "decode", "model": "qwen2", "kv": kv, "rows": log(1, 64), "lo": log(32, 256), "hi": log(256, 2048), "steps": 8}
    if kind == "moe":
        return {"kind": "decode", "model": "qwen3moe", "kv": kv, "rows": log(1, 128), "lo": log(32, 256), "hi": log(256, 2048), "steps": 4}
    if kind == "rollout":
        return {"kind": "rollout", "model": "llama", "kv": "f16", "rows": rng.randint(2, 32), "samples": rng.randint(2, 8), "prefix": log(100, 2048),
                "lo": 32, "hi": log(64, 512), "steps": 4}
    if kind == "mixed":
        return {"kind": "mixed", "model": rng.choice(["llama", "qwen3moe"]), "kv": kv, "rows": rng.randint(4, 64), "lo": log(32, 256), "hi": log(256, 2048),
                "chunk": log(17, 448), "at": rng.choice([0, log(100, 1500)])}
    if kind == "prefill":
        n = log(24, 4096)
        return {"kind": "prefill", "model": "llama", "kv": kv, "rows": 1 if n > 2000 else rng.randint(1, 2), "lo": max(16, n // 2), "hi": n, "scored": 16}
    if kind == "moe_prefill":
        return {"kind": "prefill", "model": "qwen3moe", "kv": kv, "rows": rng.randint(1, 4), "lo": 64, "hi": log(65, 1000), "scored": 16}
    if kind == "stack_decode":
        return {"kind": "decode", "model": "pomisun", "kv": "f16", "rows": log(1, 64), "lo": log(32, 256), "hi": log(256, 2048), "steps": 8}
    if kind == "stack_prefill":
        n = log(64, 3900)
        return {"kind": "prefill", "model": "pomisun", "kv": "f16", "rows": 1, "lo": n, "hi": n, "scored": 16}
    return {"kind": "prefill", "model": "dibosun", "kv": "f16", "rows": rng.randint(1, 5), "lo": 100, "hi": log(101, 1500), "scored": 16}


# ---- inputs ---------------------------------------------------------------------------

def _is_stack(model):
    return isinstance(MODELS[model][0], dict)


def _vocab(model):
    m = MODELS[model][0]
    return m["vocab"] if _is_stack(model) else m.n_vocab


class _Inputs:
    """A case's sequences and steps. `nodes`: (parent, tokens), a tree of token runs in which a child continues its
    parent; `home`: the slot that holds a node's run; `setup`: nodes to bring into the cache beforehand, in order;
    `steps`: rows (node, first index, count) of every step, with the (row, index) places whose logits it returns, or
    None where it samples every row."""

    def __init__(self, case, seed):
        rng = np.random.default_rng([seed, 11])
        v = _vocab(case["model"])
        text = lambda n: rng.integers(0, v, n).astype(np.int32)
        lens = [int(round(x)) for x in np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["rows"]))]
        self.route = rng.integers(0, LORA_COUNT + 1, case["rows"])
        self.nodes, self.setup, self.fork, self.steps = [], [], [], []
        kind, n_batch = case["kind"], MODELS[case["model"]][2]
        if kind == "decode":
            for n in lens:
                self.nodes.append((None, text(n)))
                self.nodes.append((len(self.nodes) - 1, text(case["steps"])))
            tails = range(1, len(self.nodes), 2)
            self.home = [i // 2 for i in range(len(self.nodes))]
            self.setup = list(range(0, len(self.nodes), 2))
        elif kind == "rollout":
            # a prompt's first sample continues in the prompt's slot, the first prompt in the system prompt's
            self.nodes.append((None, text(case["prefix"])))
            for n in lens:
                self.nodes.append((0, text(n)))
            for p in range(case["rows"]):
                for _ in range(case["samples"]):
                    self.nodes.append((1 + p, text(case["steps"])))
            tails = range(1 + case["rows"], len(self.nodes))
            first = [p * case["samples"] for p in range(case["rows"])]
            self.home = [0] + first + list(range(case["rows"] * case["samples"]))
            self.setup = [0] + list(range(case["rows"], 0, -1))
        elif kind == "mixed":
            for n in lens + [case["at"]]:
                self.nodes.append((None, text(n)))
                self.nodes.append((len(self.nodes) - 1, text(1)))
            self.nodes[-1] = (len(self.nodes) - 2, text(case["chunk"]))
            tails = range(1, len(self.nodes), 2)
            self.home = [i // 2 for i in range(len(self.nodes))]
            self.setup = [i for i in range(0, len(self.nodes), 2) if len(self.nodes[i][1])]
        else:
            self.nodes = [(None, text(n)) for n in lens]
            tails = range(len(self.nodes))
            self.home = list(range(len(self.nodes)))
        self.tails = list(tails)
        if kind in ("decode", "rollout"):
            for s in range(case["steps"]):
                self.steps.append(([(i, s, 1) for i in tails], [(r, 0) for r in range(len(tails))] if s + 1 == case["steps"] else None))
        elif kind == "mixed":
            rows = [(i, 0, len(self.nodes[i][1])) for i in tails]
            self.steps.append((rows, [(r, n - 1) for r, (_, _, n) in enumerate(rows)]))
        else:                            # prompts in order, packed into steps of at most n_batch tokens
            rows, room = [], n_batch
            todo = [(i, len(self.nodes[i][1])) for i in tails]
            def flush():
                want = []
                for r, (i, at, n) in enumerate(rows):
                    first = max(len(self.nodes[i][1]) - case["scored"], 0)
                    want += [(r, k - at) for k in range(max(first, at), at + n)]
                self.steps.append((list(rows), want))
            for i, n in todo:
                at = 0
                while at < n:
                    take = min(room, n - at)
                    rows.append((i, at, take))
                    at, room = at + take, room - take
                    if room == 0:
                        flush()
                        rows, room = [], n_batch
            if rows:
                flush()
        self.start = []                  # position of a node's first token
        for parent, _ in self.nodes:
            self.start.append(0 if parent is None else self.start[parent] + len(self.nodes[parent][1]))

    def adapter_of(self, case, node):
        """Index of the adapter the node's tokens run under, or -1."""
        if case["model"] != "qwen2":
            return -1
        return int(self.route[self.home[node]]) - 1


# ---- models and engines -----------------------------------------------------------------

def _model_path(model):
    m = MODELS[model][0]
    folder = Path(os.environ.get("RETRO_BENCH_MODEL_DIR", tempfile.gettempdir())) / ("retro-cases-%d" % os.getuid())
    folder.mkdir(parents=True, exist_ok=True)
    if _is_stack(model):
        path = folder / ("%s-w%d" % (model, m["width"]))
        if not (path / "done").exists():
            synth_stack.write_random_checkpoint(path, m, 1234, device="cuda")
            (path / "done").write_text("")
        return path
    path = folder / ("%s.gguf" % m.name)
    if not path.exists():
        tmp = path.with_suffix(".%d" % os.getpid())
        synth.write_model(tmp, m, seed=1234, device="cuda")
        os.replace(tmp, path)
    return path


def _adapter_paths():
    shape = MODELS["qwen2"][0]
    out = []
    for i in range(LORA_COUNT):
        path = _model_path("qwen2").with_name("qwen2-lora-%d.gguf" % i)
        if not path.exists():
            tmp = path.with_suffix(".%d" % os.getpid())
            synth.write_lora_adapter(tmp, shape, rank=LORA_RANK, alpha=float(LORA_RANK), seed=1334 + i, std_a=0.02, std_b=0.01)
            os.replace(tmp, path)
        out.append(path)
    return out


class _Server:
    """A loaded model and which of its slots and cells are taken."""

    def __init__(self, model, kv):
        _, self.cells, n_batch = MODELS[model]
        path = _model_path(model)
        torch.cuda.empty_cache()
        self.engine = E.Engine(path, E.EngineConfig(n_ctx=self.cells, n_seq_max=SLOTS if model != "dibosun" else 32, n_batch=n_batch, n_ubatch=n_batch,
                                                    kv_dtype=E.KV_Q8_0 if kv == "q8_0" else E.KV_F16))
        self.adapters = [self.engine.adapter_load(p, 1.0) for p in _adapter_paths()] if model == "qwen2" else []
        self.taken = []                  # (first slot, slots, cells)

    def take(self, count, cells):
        """A block of slots, or None."""
        at = 0
        for first, n, _ in sorted(self.taken):
            if first - at >= count:
                break
            at = first + n
        if at + count > self.engine.config.n_seq_max or cells + sum(t[2] for t in self.taken) > self.cells:
            return None
        self.taken.append((at, count, cells))
        return self.taken[-1]


_servers = {}


def _place(model, kv, count, cells):
    """A server with room, and the block of its slots that is now taken."""
    if (model, kv) not in _servers:
        _servers.clear()                 # one model resides at a time; states that are alive keep theirs
        _servers[(model, kv)] = []
    for server in _servers[(model, kv)]:
        block = server.take(count, cells)
        if block is not None:
            return server, block
    _servers[(model, kv)].append(_Server(model, kv))
    return _servers[(model, kv)][-1], _servers[(model, kv)][-1].take(count, cells)


class _State:
    def __init__(self, case, seed):
        self.inputs = x = _Inputs(case, seed)
        self.bf16 = _is_stack(case["model"])
        self.server, self.block = _place(case["model"], case["kv"], max(x.home) + 1, sum(len(t) + 64 for _, t in x.nodes))
        self.eng = eng = self.server.engine
        self.out = E.StepOutput(self.block[1])
        slot = [self.block[0] + h for h in x.home]
        greedy = E.SamplingParamsV2.greedy()
        base = E.RowAdapter.base() if case["model"] == "qwen2" else E.RowAdapter.context()
        adapter = lambda i: base if x.adapter_of(case, i) < 0 else E.RowAdapter.loaded(self.server.adapters[x.adapter_of(case, i)])
        n_batch = eng.config.n_batch
        for i in x.setup:
            parent, tokens = x.nodes[i]
            if parent is not None and slot[i] != slot[parent]:
                eng.seq_cp(slot[parent], slot[i])
            for at in range(0, len(tokens), n_batch):
                eng.step([E.StepRow(slot[i], slot[i], tokens[at:at + n_batch], x.start[i] + at, adapter=adapter(i))], self.out)
        if case["kind"] == "rollout":    # forked and already past their first token, so their last pages are their own
            for i in x.tails:
                if slot[i] != slot[x.nodes[i][0]]:
                    eng.seq_cp(slot[x.nodes[i][0]], slot[i])
            eng.step([E.StepRow.decode(slot[i], slot[i], int(x.nodes[i][1][0]), x.start[i], greedy) for i in x.tails], self.out)
        self.back = [(slot[i], x.start[i]) for i in x.tails]
        self.plan = []
        for rows, want in x.steps:
            if want is None or case["model"] == "qwen2":
                step = []
                for i, at, n in rows:
                    step.append(E.StepRow(slot[i], slot[i], x.nodes[i][1][at:at + n], x.start[i] + at, sample=want is None or n == 1,
                                          sampling=greedy, adapter=adapter(i)))
                self.plan.append((step, None))
            else:
                self.plan.append(([(slot[i], x.nodes[i][1][at:at + n], x.start[i] + at) for i, at, n in rows], want))

    def __del__(self):
        try:
            for s in range(self.block[0], self.block[0] + self.block[1]):
                self.eng.seq_rm(s)
                self.eng.request_free(s)
            self.server.taken.remove(self.block)
        except Exception:
            pass


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    eng, out = state.eng, state.out
    for slot, pos in state.back:
        eng.seq_rm(slot, pos)
    tokens, logprobs, logits = [], [], []
    for rows, want in state.plan:
        if want is None:
            eng.step(rows, out)
            got = out.rows()
            tokens.append([r.token for r in got])
            logprobs.append([r.logprob for r in got])
        elif want:
            logits.append(eng.step_logits(rows, want))
        else:
            eng.step([E.StepRow.prefill(-1, s, t, p) for s, t, p in rows], out)
    if state.server.adapters:            # rows routed to adapters go through step(): its logits stay on the device until asked for
        logits.append(eng.debug_logits())
    got = {"logprobs": np.array(logprobs, np.float32), "logits": logits}
    if not state.bf16:                   # under bf16 products the order of a sum decides which of two near-equal logits leads
        got["tokens"] = np.array(tokens, np.int64)
    return got


# ---- what a pass cannot do without ---------------------------------------------------------

def _keys(model, pos):
    """Keys a token at position pos attends, of the layers that attend."""
    if model == "pomisun":
        return pos % bench_stack.CHUNK + 1
    return min(pos + 1, bench_stack.WINDOW) if model == "dibosun" else pos + 1


def work(case):
    x = _Inputs(case, 0)
    model, m = case["model"], MODELS[case["model"]][0]
    by = fl = 0.0
    for rows, want in x.steps:
        T = sum(n for _, _, n in rows)
        n_out = len(want) if want is not None else len(rows)
        attended = 0                     # pairs of a token and a key
        cells = {}                       # cells read, by the node that owns them
        for i, at, n in rows:
            p0 = x.start[i] + at
            attended += sum(_keys(model, p) for p in range(p0, p0 + n))
            cells[i] = max(cells.get(i, 0), at + n)
            first = p0 + n - _keys(model, p0 + n - 1)
            up = x.nodes[i][0]
            while up is not None:
                cells[up] = max(cells.get(up, 0), min(len(x.nodes[up][1]), x.start[up] + len(x.nodes[up][1]) - first))
                up = x.nodes[up][0]
        cells = sum(max(c, 0) for c in cells.values())
        if _is_stack(model):
            w = getattr(bench_stack, model + "_work")(m, T, (attended / T, cells, len(rows)), n_out)
            by += sum(v[0] for v in w.values())
            fl += sum(sum(v[1:]) for v in w.values())
            continue
        s = m
        QD, KD, V = s.n_head * s.head_dim, s.n_head_kv * s.head_dim, s.n_vocab
        attn = s.n_embd * (2 * QD + 2 * KD)
        bpw = {synth.gw.GGML_Q4_K: 144 / 256, synth.gw.GGML_Q8_0: 34 / 32}[s.matrix_type]
        by += s.n_layer * attn * bpw + (V * s.n_embd * bpw + n_out * V * 4 if n_out else 0)
        fl += 2 * T * s.n_layer * attn + 2 * n_out * V * s.n_embd
        if s.n_expert:
            expert = 3 * s.n_embd * s.n_ff_exp
            by += s.n_layer * (bench_stack.chosen_experts(s.n_expert, s.n_expert_used, T) * expert * 17 / 32 + 4 * s.n_expert * s.n_embd)
            fl += 2 * T * s.n_layer * (s.n_expert_used * expert + s.n_expert * s.n_embd)
        else:
            by += s.n_layer * 3 * s.n_embd * s.n_ff * bpw
            fl += 2 * T * s.n_layer * 3 * s.n_embd * s.n_ff
        if model == "qwen2":
            per = LORA_RANK * (4 * s.n_embd + 2 * QD + 2 * KD)
            by += s.n_layer * per * 2 * len({x.adapter_of(case, i) for i, _, _ in rows} - {-1})
            fl += 2 * s.n_layer * per * sum(n for i, _, n in rows if x.adapter_of(case, i) >= 0)
        by += s.n_layer * 2 * KD * cells * (34 / 32 if case["kv"] == "q8_0" else 2)
        fl += s.n_layer * 4 * QD * attended
    return {"bytes": by, "flops": fl}


def tolerance(case):
    # About four times what the 64-bit results below differ by. GGUF models: f32 accumulation over activations of about
    # 22 bits, 4e-5 to 1.6e-4, most of it values of the cache that another order of the sums puts on the other side of a
    # rounding boundary (Q8_0 cache: a step of 1/127, 1.5e-3); with experts a near tie in the routing takes another
    # expert for a token, 4e-4 to 4.5e-3. bf16 products: every activation is rounded to 8 bits, 4e-3 to 7e-3.
    if _is_stack(case["model"]):
        return {"rel": 0.028, "max": 0.5}
    if case["model"] == "qwen3moe":
        return {"rel": 0.018, "max": 0.3, "differ": 0.01}
    if case["kv"] == "q8_0":
        return {"rel": 6e-3, "max": 0.1, "differ": 0.01}
    return {"rel": 5e-4, "max": 0.01, "differ": 0.005}


# ---- the same in 64 bits ------------------------------------------------------------------

class _Gguf:
    """Tensors of a GGUF file, as float64 on the GPU."""
    GEOMETRY = {0: (1, 4), 1: (1, 2), 8: (32, 34), 12: (256, 144), 39: (32, 17)}

    def __init__(self, path):
        self.f = open(path, "rb")
        self.map = mmap.mmap(self.f.fileno(), 0, access=mmap.ACCESS_READ)
        self.at = 8
        n_tensors, n_kv = self.take("<QQ")
        for _ in range(n_kv):
            self.text()
            self.value(self.take("<I")[0])
        self.info = {}
        for _ in range(n_tensors):
            name = self.text()
            ne = self.take("<%dQ" % self.take("<I")[0])
            self.info[name] = (ne, *self.take("<IQ"))
        self.base = (self.at + 31) // 32 * 32

    def take(self, fmt):
        v = struct.unpack_from(fmt, self.map, self.at)
        self.at += struct.calcsize(fmt)
        return v

    def text(self):
        n = self.take("<Q")[0]
        self.at += n
        return self.map[self.at - n:self.at].decode()

    def value(self, t):
        if t == 8:
            return self.text()
        if t == 9:
            kind, n = self.take("<IQ")
            for _ in range(n):
                self.value(kind)
            return None
        return self.take("<" + {0: "B", 1: "b", 2: "H", 3: "h", 4: "I", 5: "i", 6: "f", 7: "?", 10: "Q", 11: "q", 12: "d"}[t])

    def __call__(self, name, part=None):
        """[rows, columns] (a vector: [columns]); `part`: one matrix of a stack of them."""
        ne, kind, off = self.info[name]
        el, nb = self.GEOMETRY[kind]
        rows, k = int(np.prod(ne[1:])) if len(ne) > 1 else 1, ne[0]
        at, n = self.base + off, rows * k // el * nb
        if part is not None:
            n //= ne[2]
            rows //= ne[2]
            at += part * n
        raw = torch.from_numpy(np.frombuffer(self.map, np.uint8, n, at).copy()).cuda().reshape(-1, nb)
        half = lambda a: raw[:, a:a + 2].contiguous().view(torch.float16).double()
        if kind == 0:
            v = raw.view(torch.float32).double()
        elif kind == 1:
            v = raw.view(torch.float16).double()
        elif kind == 8:
            v = half(0) * raw[:, 2:].contiguous().view(torch.int8).double()
        elif kind == 39:
            grid = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device="cuda")
            codes = torch.cat([raw[:, 1:] & 15, raw[:, 1:] >> 4], 1).long()
            v = grid[codes] * torch.exp2(raw[:, :1].double() - 127)
        else:
            s = raw[:, 4:16].int()
            sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
            mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
            q = raw[:, 16:].reshape(-1, 4, 32)
            q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
            v = (half(0) * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
        return v.reshape(rows, k) if len(ne) > 1 else v.reshape(k)


class _Safetensors:
    def __init__(self, folder):
        with open(Path(folder) / "model.safetensors", "rb") as f:
            n = struct.unpack("<Q", f.read(8))[0]
            self.head, self.base = json.loads(f.read(n)), 8 + n
            self.map = mmap.mmap(f.fileno(), 0, access=mmap.ACCESS_READ)

    def __call__(self, name):
        d = self.head[name]
        a, b = d["data_offsets"]
        bits = torch.from_numpy(np.frombuffer(self.map, np.int16, (b - a) // 2, self.base + a).copy()).cuda()
        return bits.view(torch.bfloat16).double().reshape(d["shape"])


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _silu(x):
    return x * torch.sigmoid(x)


def _stored(x, kv):
    """[tokens, heads, dim] as the cache holds it."""
    if kv == "f16":
        return x.half().double()
    b = x.reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    q = torch.where(d > 0, b / d, b)
    q = torch.sign(q) * torch.floor(q.abs() + 0.5)
    return (q * d.half().double()).reshape(x.shape)


def _attend(q, k, v, scale, first, span, cap=None):
    """q [n, H, D] at positions first.., k and v [m, G, .] from position 0; span(p): the first position that p sees."""
    n, H, _ = q.shape
    G = k.shape[1]
    out = torch.empty(n, H, v.shape[2], dtype=q.dtype, device=q.device)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    j = torch.arange(k.shape[0], device=q.device)
    for a in range(0, n, 512):
        p = torch.arange(first + a, first + min(n, a + 512), device=q.device)
        seen = (j[None, :] <= p[:, None]) & (j[None, :] >= span(p)[:, None])
        for g in range(G):
            qs = q[a:a + 512, g * (H // G):(g + 1) * (H // G)]
            s = qs.reshape(-1, q.shape[2]) @ kt[g] * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            s = s.reshape(len(p), H // G, -1).masked_fill(~seen[:, None], -math.inf)
            out[a:a + 512, g * (H // G):(g + 1) * (H // G)] = (torch.softmax(s, -1).reshape(-1, s.shape[-1]) @ vt[g]).reshape(len(p), H // G, -1)
    return out


def _mixture(h, sel, weight, expert):
    out = torch.zeros_like(h)
    for e in sel.unique().tolist():
        t, slot = (sel == e).nonzero(as_tuple=True)
        out.index_add_(0, t, expert(e, h[t]) * weight[t, slot][:, None])
    return out


class _Runs:
    """The case's token runs laid end to end."""

    def __init__(self, x):
        self.x = x
        self.at = np.cumsum([0] + [len(t) for _, t in x.nodes])
        self.tokens = torch.from_numpy(np.concatenate([t for _, t in x.nodes]).astype(np.int64)).cuda()
        self.pos = torch.from_numpy(np.concatenate([s + np.arange(len(t)) for s, (_, t) in zip(x.start, x.nodes)])).cuda()

    def of(self, i):
        return slice(int(self.at[i]), int(self.at[i + 1]))

    def line(self, i):
        """Nodes from the root to i."""
        up = []
        while i is not None:
            up.insert(0, i)
            i = self.x.nodes[i][0]
        return up

    def attend(self, q, k, v, scale, span, cap=None):
        out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=q.dtype, device=q.device)
        for i in range(len(self.x.nodes)):
            s = self.of(i)
            if s.stop > s.start:
                past = [self.of(j) for j in self.line(i)]
                out[s] = _attend(q[s], torch.cat([k[p] for p in past]), torch.cat([v[p] for p in past]), scale, self.x.start[i], span, cap)
        return out


def _in_parts(f, x, size=16384):
    return torch.cat([f(x[a:a + size]) for a in range(0, len(x), size)])


def _gguf_stream(case, x, runs):
    """The residual stream behind the last layer, and the head."""
    s, W = MODELS[case["model"]][0], _Gguf(_model_path(case["model"]))
    neox = s.arch != "llama"
    H, G, D = s.n_head, s.n_head_kv, s.head_dim
    lora = [_Gguf(p) for p in _adapter_paths()] if case["model"] == "qwen2" else []
    rows_of = [torch.cat([torch.arange(runs.of(i).start, runs.of(i).stop, device="cuda") for i in range(len(x.nodes)) if x.adapter_of(case, i) == a]
                         or [torch.empty(0, dtype=torch.long, device="cuda")]) for a in range(len(lora))]
    ang = runs.pos.double()[:, None] * torch.from_numpy(s.rope_base ** (-2.0 * np.arange(D // 2) / D)).cuda()[None, :]
    c, sn = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

    def turn(t):
        if neox:
            a, b = t[..., :D // 2], t[..., D // 2:]
            return torch.cat([a * c - b * sn, b * c + a * sn], -1)
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack([a * c - b * sn, b * c + a * sn], -1).reshape(t.shape)

    def product(h, l, name, bias=False):
        y = h @ W("blk.%d.%s.weight" % (l, name)).T
        if bias:
            y = y + W("blk.%d.%s.bias" % (l, name))
        for f, r in zip(lora, rows_of):
            if len(r):
                n = "blk.%d.%s.weight.lora_" % (l, name)
                y[r] += h[r] @ f(n + "a").T @ f(n + "b").T
        return y

    h = W("token_embd.weight")[runs.tokens]
    for l in range(s.n_layer):
        b = "blk.%d." % l
        a = _rms(h, W(b + "attn_norm.weight"), s.eps)
        q = product(a, l, "attn_q", s.qkv_bias).reshape(-1, H, D)
        k = product(a, l, "attn_k", s.qkv_bias).reshape(-1, G, D)
        v = product(a, l, "attn_v", s.qkv_bias).reshape(-1, G, D)
        if s.arch == "qwen3moe":
            q, k = _rms(q, W(b + "attn_q_norm.weight"), s.eps), _rms(k, W(b + "attn_k_norm.weight"), s.eps)
        o = runs.attend(turn(q), _stored(turn(k), case["kv"]), _stored(v, case["kv"]), D ** -0.5, lambda p: torch.zeros_like(p))
        h = h + product(o.reshape(-1, H * D), l, "attn_output")
        a = _rms(h, W(b + "ffn_norm.weight"), s.eps)
        if s.n_expert:
            z = a @ W(b + "ffn_gate_inp.weight").T
            top, sel = z.topk(s.n_expert_used, 1)
            mats = lambda e: [W(b + "ffn_%s_exps.weight" % n, e) for n in ("gate", "up", "down")]

            def expert(e, t):
                g, u, d = mats(e)
                return (_silu(t @ g.T) * (t @ u.T)) @ d.T
            h = h + _mixture(a, sel, torch.softmax(top, 1), expert)
        else:
            g, u, d = (W(b + "ffn_%s.weight" % n) for n in ("gate", "up", "down"))
            h = h + _in_parts(lambda t: (_silu(t @ g.T) * (t @ u.T)) @ d.T, a)
    return lambda rows: _rms(h[rows], W("output_norm.weight"), s.eps) @ W("output.weight").T


def _pomisun_stream(case, x, runs):
    cfg, W = MODELS["pomisun"][0], _Safetensors(_model_path("pomisun"))
    eps, span = cfg["norm"]["eps"], lambda p: p // bench_stack.CHUNK * bench_stack.CHUNK
    norm = lambda t, name: _rms(t, 1 + W(name), eps)
    h = W("embed")[runs.tokens]
    for i, layer in enumerate(cfg["layers"]):
        p, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
        H, G, D, rot = m["heads"], m["kv_heads"], m["dim"], m["rot"]
        freq = rot["base"] ** (-np.arange(0, rot["dims"], 2) / rot["dims"])
        sc = rot["scaling"]
        edge = lambda turns: rot["dims"] * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))
        lo, hi = max(math.floor(edge(sc["fast"])), 0), min(math.ceil(edge(sc["slow"])), rot["dims"] - 1)
        ramp = np.clip((np.arange(rot["dims"] // 2) - lo) / max(hi - lo, 0.001), 0, 1)
        ang = runs.pos.double()[:, None] * torch.from_numpy(freq / sc["factor"] * ramp + freq * (1 - ramp)).cuda()
        mag = 0.1 * math.log(sc["factor"]) + 1
        c, s = (torch.cos(ang) * mag)[:, None], (torch.sin(ang) * mag)[:, None]
        turn = lambda t: torch.cat([t[..., :D // 2] * c - t[..., D // 2:] * s, t[..., D // 2:] * c + t[..., :D // 2] * s], -1)
        a = norm(h, p + "norm1")
        v = (a @ W(p + "mix.k").T).reshape(-1, G, D)
        o = runs.attend(turn((a @ W(p + "mix.q").T).reshape(-1, H, D)), turn(v), v, m["scale"], span, m["softcap"])
        h = h + o.reshape(-1, H * D) @ W(p + "mix.o").T
        a, p = norm(h, p + "norm2"), p + "mlp."
        gated = lambda t, q, act: (act(t @ W(q + "gate").T) * (t @ W(q + "up").T)) @ W(q + "down").T
        if mlp["kind"] == "dense":
            h = h + _in_parts(lambda t: gated(t, p, lambda z: torch.nn.functional.gelu(z, approximate="tanh")), a)
            continue
        top, sel = (a @ W(p + "router").T).topk(mlp["router"]["top"], 1)
        y = _mixture(a, sel, torch.softmax(top, 1), lambda e, t: gated(t, p + "e%d." % e, _silu))
        h = h + y + gated(a, p + "shared.", _silu) * torch.sigmoid(a @ W(p + "shared.sg").T)
    return lambda rows: norm(h[rows], "final.norm") @ W("embed").T


def _dibosun_stream(case, x, runs):
    cfg, W = MODELS["dibosun"][0], _Safetensors(_model_path("dibosun"))
    eps = cfg["norm"]["eps"]
    norm = lambda t, name: torch.nn.functional.layer_norm(t, t.shape[-1:], W(name), None, eps)
    h, latents = W("embed")[runs.tokens], {}
    for i, layer in enumerate(cfg["layers"]):
        p, m = "l%d." % i, layer["mixer"]
        a, x_ = norm(h, p + "norm1"), p + "mix."
        if layer["type"] == "latent_attention":
            H, D, V, size = m["heads"], m["dim"], m["vdim"], m["mask"]["size"]
            src = m.get("kv_from")
            if src is None:
                latents[i] = _rms(a @ W(x_ + "dkv").T, W(x_ + "dkv.norm"), eps)
            lat = latents[i if src is None else src]
            q = (_rms(a @ W(x_ + "dq").T, W(x_ + "dq.norm"), eps) @ W(x_ + "uq").T).reshape(-1, H, D)
            k, v = (lat @ W(x_ + "uk").T).reshape(-1, H, D), (lat @ W(x_ + "uv").T).reshape(-1, H, V)
            o = runs.attend(q, k, v, m["scale"], lambda p: torch.clamp(p - size + 1, min=0))
            mix = (o * torch.sigmoid(a @ W(x_ + "g").T)[:, :, None]).reshape(-1, H * V) @ W(x_ + "o").T
        else:
            H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            inner = H * P
            z, xbc, dt = (a @ W(x_ + "in").T).split([inner, inner + 2 * G * N, H], 1)
            taps, y = W(x_ + "conv"), torch.empty(len(a), inner, dtype=a.dtype, device=a.device)
            dt = torch.nn.functional.softplus(dt + W(x_ + "dt_bias"))
            decay, skip = torch.exp(-torch.exp(W(x_ + "A_log")) * dt), W(x_ + "D")
            longest = max(len(t) for _, t in x.nodes)
            pad = lambda t: torch.stack([torch.nn.functional.pad(t[runs.of(j)], (0, 0, 0, longest - len(t[runs.of(j)]))) for j in range(len(x.nodes))])
            u = torch.nn.functional.pad(pad(xbc), (0, 0, taps.shape[1] - 1, 0))
            u = _silu(sum(u[:, j:j + longest] * taps[:, j] for j in range(taps.shape[1])) + W(x_ + "conv.b"))
            xs, B, C = u.split([inner, G * N, G * N], 2)
            xs = xs.reshape(*xs.shape[:2], H, P)
            B, C = (t.reshape(*t.shape[:2], G, N).repeat_interleave(H // G, 2) for t in (B, C))
            decay, dt = pad(decay), pad(dt)
            S = torch.zeros(len(x.nodes), H, N, P, dtype=a.dtype, device=a.device)
            ys = []
            for t in range(longest):
                S = S * decay[:, t, :, None, None] + (dt[:, t, :, None] * B[:, t])[..., None] * xs[:, t, :, None, :]
                ys.append((S * C[:, t, ..., None]).sum(2) + skip[:, None] * xs[:, t])
            ys = torch.stack(ys, 1).reshape(len(x.nodes), longest, inner)
            for j in range(len(x.nodes)):
                y[runs.of(j)] = ys[j, :len(x.nodes[j][1])]
            y = (y * _silu(z)).reshape(len(a), m["norm_groups"], -1)
            mix = _rms(y, W(x_ + "norm").reshape(m["norm_groups"], -1), eps).reshape(len(a), inner) @ W(x_ + "o").T
        ff = torch.relu(a @ W(p + "mlp.up").T) ** 2 @ W(p + "mlp.down").T
        h = h + mix * W(p + "ls1") + ff * W(p + "ls2")
    return lambda rows: norm(h[rows], "final.norm") @ W("embed").T


def exact(case, seed):
    x = _Inputs(case, seed)
    runs = _Runs(x)
    with torch.no_grad():
        head = {"pomisun": _pomisun_stream, "dibosun": _dibosun_stream}.get(case["model"], _gguf_stream)(case, x, runs)
        logprobs, logits = [], []
        for rows, want in x.steps:
            sampled = want is None or case["model"] == "qwen2"
            places = [(r, 0) for r in range(len(rows))] if sampled else want
            if not places:
                continue
            z = head(torch.tensor([runs.of(rows[r][0]).start + rows[r][1] + k for r, k in places], device="cuda"))
            if sampled:
                logprobs.append(torch.log_softmax(z, 1).amax(1).cpu().numpy())
            if not sampled or want is not None:
                logits.append(z.cpu().numpy())
    got = {"logprobs": np.array(logprobs), "logits": logits}
    return got if _is_stack(case["model"]) else dict(got, tokens=None)
