"""Timed workloads of this framework, through its public entry points.

What a program that uses the framework has it do:

* the backward cycle (``LoraSftTrainerService.process_backward``): final norm, LM head and loss,
  the decoder layers from the last to the first (forward recompute and backward), the per-layer
  clip, AdamW and the publish into the served LoRA slots. One pass is one cycle on one filled
  activation store. The widths, ranks, vocabularies and packings are those of
  ``deltaserve_amd.configs``; the layer count is cut to 2-4 (a whole model repeats the same layer),
  the LM head is whole.
* the serving worker's half of the handoff: the save of one forward step's finetuning rows.
* the single ops of ``deltaserve_amd.ops`` (attention forward and backward, the gate/up product
  with SwiGLU, a dX product, the streamed LM head, the batched LoRA pass).

A case is a dict of plain values; ``prepare`` builds from it and a seed what a user's program holds
before the call, ``run`` makes one pass, ``exact`` states the same result in 64 bits.
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "deltaserve-vllm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
BF16 = torch.bfloat16
F64 = torch.float64

# Model widths the repository configures (deltaserve_amd.configs.CONFIGS).
MODELS = {
    "qwen3-0.6b": dict(family="qwen3", D=1024, Hq=16, Hkv=8, Hd=128, I=3072, V=151936, theta=1e6,
                       eps=1e-6, tie=True, rope=None),
    "llama3.2-1b": dict(family="llama3", D=2048, Hq=32, Hkv=8, Hd=64, I=8192, V=128256, theta=5e5,
                        eps=1e-5, tie=True, rope=32.0),
    "llama3-8b": dict(family="llama3", D=4096, Hq=32, Hkv=8, Hd=128, I=14336, V=128256, theta=5e5,
                      eps=1e-5, tie=False, rope=None),
    "llama3-8b-long": dict(family="llama3", D=4096, Hq=32, Hkv=8, Hd=128, I=14336, V=128256,
                           theta=5e5, eps=1e-5, tie=False, rope=8.0),
    "qwen3-14b": dict(family="qwen3", D=5120, Hq=40, Hkv=8, Hd=128, I=17408, V=151936, theta=1e6,
                      eps=1e-6, tie=False, rope=None),
}
ALL_PROJS = ("q", "k", "v", "o", "gate", "up", "down")
# the most algorithmic flops a drawn cycle takes (the largest listed one has about 67e12)
MOST_FLOPS = 60e12


def listed():
    return [
        # One serving step's save: 256 finetuning rows picked out of a flat batch of 384, for 8
        # layers (the residual stream as the fused add-norm leaves it, x + r, and the gate/up
        # output), the final hidden row and the ids. The smallest calls: copies of a few MB.
        dict(name="save-step-256", kind="save", model="qwen3-14b", layers=8, rows=384, ft=256,
             max_saved=256, resid=True, gate_up=True, dtype="bf16"),
        # Attention over a packed cycle of 32 sequences of 64-512 tokens, 8192 in all (the headline
        # packing): many short ragged sequences, no multiple of a tile among them.
        dict(name="attn-fwd-packed", kind="attn_fwd", Hq=32, Hkv=8, Hd=128, nseq=32, lo=64, hi=512,
             total=8192, lens=0),
        # Attention's backward over one long and one ragged sequence: the long-context packing,
        # where attention is a third of a layer.
        dict(name="attn-bwd-long", kind="attn_bwd", Hq=32, Hkv=8, Hd=128, nseq=2, lo=4001, hi=8192,
             total=12193, lens=1),
        # The MLP's gate/up product with its LoRA term and SwiGLU, at the narrow model's widths and
        # a ragged row count: a forward block whose reduction is short.
        dict(name="mlp-glu-4718", kind="glu", D=1024, I=3072, r=16, M=4718),
        # The gate/up dX product of a 256-token serving cycle (fp32 out, weight in its own layout,
        # LoRA factor as a second segment): a product that streams its weights.
        dict(name="mlp-dx-256", kind="dx", D=5120, I=17408, r=16, M=256),
        # The streamed LM head, loss and gradient of 2048 packed rows over a 128256-word vocabulary.
        dict(name="head-2048", kind="head", D=2048, V=128256, nseq=8, lo=64, hi=512, total=2048,
             lens=0),
        # The MLP's three rank-16 LoRA passes (grad_Z and grad_B of gate and up, Z and grad_A of
        # down) of a headline-size cycle: memory-bound.
        dict(name="lora-mlp-8192", kind="lora", C=14336, r=16, n=8192, count=3),
        # A cycle of the smallest configuration: 4 sequences, about 500 tokens, rank 8; latency and
        # launches count.
        dict(name="cycle-0.6b-r8", kind="cycle", model="qwen3-0.6b", L=4, r=8, nseq=4, lo=32, hi=256,
             total=504, lens=0, projs="all", saved=False, pause=False),
        # The serving preset's cycle: 256 tokens of the 14B model, rank 16; every product streams
        # its weights.
        dict(name="cycle-14b-256", kind="cycle", model="qwen3-14b", L=4, r=16, nseq=2, lo=64, hi=192,
             total=256, lens=0, projs="all", saved=False, pause=False),
        # A co-located cycle as the worker's default capture leaves it: gate/up saved by the forward,
        # pause points on (one graph per segment), head_dim 64, tied head, rank 8.
        dict(name="cycle-1b-saved-pause", kind="cycle", model="llama3.2-1b", L=4, r=8, nseq=8, lo=64,
             hi=512, total=2048, lens=0, projs="all", saved=True, pause=True),
        # The headline cycle: Llama-3-8B widths, rank 16, 32 sequences, 8192 tokens.
        dict(name="cycle-8b-8192", kind="cycle", model="llama3-8b", L=4, r=16, nseq=32, lo=64, hi=512,
             total=8192, lens=0, projs="all", saved=False, pause=False),
        # The long-context cycle: two sequences of 8192 tokens, rank 64, scaled RoPE; the largest.
        dict(name="cycle-8b-long-r64", kind="cycle", model="llama3-8b-long", L=2, r=64, nseq=2,
             lo=8192, hi=8192, total=16384, lens=0, projs="all", saved=False, pause=False),
    ]


# ---------------------------------------------------------------- drawing

def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_packing(rng, most):
    """nseq, lo, hi, total: 1-32 sequences of up to 8192 tokens, at most `most` in all."""
    total = _logint(rng, 96, most)
    nseq = max(1, min(_logint(rng, 1, 32), total // 8))
    mean = total / nseq
    if mean > 8192:
        nseq = -(-total // 8192)
        mean = total / nseq
    return dict(nseq=nseq, lo=max(1, int(mean / 3)), hi=min(8192, max(2, int(mean * 2) + 1)),
                total=total, lens=rng.randrange(1 << 20))


def draw(rng):
    kind = rng.choice(["save", "attn_fwd", "attn_bwd", "glu", "dx", "head", "lora", "cycle", "cycle",
                       "cycle", "cycle"])
    if kind == "save":
        ft = _logint(rng, 16, 8192)
        big = ft > 1024
        return dict(kind=kind, model=rng.choice(sorted(MODELS)), layers=rng.randint(1, 2 if big else 8),
                    rows=ft + rng.randrange(0, ft + 1), ft=ft, max_saved=ft + rng.randrange(0, 65),
                    resid=rng.random() < 0.7, gate_up=rng.random() < 0.5,
                    dtype=rng.choice(["bf16", "bf16", "f16", "f32"]))
    if kind in ("attn_fwd", "attn_bwd"):
        Hq, Hkv, Hd = rng.choice([(16, 8, 128), (32, 8, 128), (40, 8, 128), (32, 8, 64)])
        return dict(kind=kind, Hq=Hq, Hkv=Hkv, Hd=Hd, **_draw_packing(rng, 12288))
    m = MODELS[rng.choice(sorted(MODELS))]
    if kind in ("glu", "dx"):
        return dict(kind=kind, D=m["D"], I=m["I"], r=rng.choice([8, 16, 32, 64]), M=_logint(rng, 32, 8192))
    if kind == "head":
        return dict(kind=kind, D=m["D"], V=m["V"], **_draw_packing(rng, 4096))
    if kind == "lora":
        case = dict(kind=kind, C=rng.choice([m["D"], m["I"], m["Hq"] * m["Hd"]]), r=rng.choice([16, 32]),
                    n=_logint(rng, 64, 8192), count=rng.randint(1, 3))
        # the allocation-free entry holds 64 MiB of partial sums: up to ceil(C/512)·n·r of them and
        # 256 column blocks' worth of C·r per pass
        while case["count"] * (-(-case["C"] // 512) * case["n"] * case["r"]) + 256 * 512 * case["r"] > 16 << 20:
            case["n"] = case["n"] * 3 // 4
        return case
    name = rng.choice(sorted(MODELS))
    case = dict(kind="cycle", model=name, L=rng.randint(1, 4), r=rng.choice([4, 8, 12, 16, 32, 64]),
                **_draw_packing(rng, 12288), projs=rng.choice(["all", "all", "all", "qkvo"]),
                saved=rng.random() < 0.35, pause=rng.random() < 0.25)
    while work(case)["flops"] > MOST_FLOPS:
        if case["L"] > 1:
            case["L"] -= 1
        else:
            case["total"] = max(case["nseq"], case["total"] * 3 // 4)
            mean = case["total"] / case["nseq"]
            case["lo"], case["hi"] = max(1, int(mean / 3)), min(8192, max(2, int(mean * 2) + 1))
    return case


def lengths(case):
    """The case's sequence lengths: uniform in [lo, hi], then walked by one to the total."""
    rng = random.Random(1000003 * case["lens"] + case["nseq"])
    lo, hi, total = case["lo"], case["hi"], case["total"]
    lens = [rng.randint(lo, hi) for _ in range(case["nseq"])]
    i = 0
    while sum(lens) != total:
        d = 1 if sum(lens) < total else -1
        if lo <= lens[i] + d <= hi:
            lens[i] += d
        i = (i + 1) % len(lens)
    return lens


# ---------------------------------------------------------------- inputs

class _Rng:
    """Seeded device tensors; each call takes the next stream of the seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 7919 + 12345)

    def randn(self, *shape, std=1.0, dtype=BF16):
        t = torch.randn(*shape, generator=self.g, device=DEV, dtype=torch.float32)
        return (t if std == 1.0 else t.mul_(std)).to(dtype)

    def uniform(self, *shape, bound):
        return (torch.rand(*shape, generator=self.g, device=DEV) * 2 - 1) * bound

    def ids(self, n, high):
        return torch.randint(0, high, (n,), generator=self.g, device=DEV)


def _proj_shapes(m):
    q, kv = m["Hq"] * m["Hd"], m["Hkv"] * m["Hd"]
    return {"q": (q, m["D"]), "k": (kv, m["D"]), "v": (kv, m["D"]), "o": (m["D"], q),
            "gate": (m["I"], m["D"]), "up": (m["I"], m["D"]), "down": (m["D"], m["I"])}


def _projs(case):
    return ALL_PROJS if case["projs"] == "all" else ("q", "k", "v", "o")


def _cycle_inputs(case, seed):
    """Frozen bf16 weights, fp32 LoRA factors and a filled activation store."""
    m, r = MODELS[case["model"]], case["r"]
    rng = _Rng(seed)
    D, I, q, kv = m["D"], m["I"], m["Hq"] * m["Hd"], m["Hkv"] * m["Hd"]
    lens = lengths(case)
    n = sum(lens)
    w = {"lm": rng.randn(m["V"], D, std=0.02), "norm": 1 + rng.randn(D, std=0.05)}
    layers = []
    for _ in range(case["L"]):
        lw = {"qkv": rng.randn(q + 2 * kv, D, std=0.02), "o": rng.randn(D, q, std=0.02),
              "gate_up": rng.randn(2 * I, D, std=0.02), "down": rng.randn(D, I, std=0.02),
              "in_ln": 1 + rng.randn(D, std=0.05), "post_ln": 1 + rng.randn(D, std=0.05)}
        if m["family"] == "qwen3":
            lw["q_norm"], lw["k_norm"] = 1 + rng.randn(m["Hd"], std=0.05), 1 + rng.randn(m["Hd"], std=0.05)
        for p in _projs(case):
            out, inp = _proj_shapes(m)[p]
            lw[p + "A"] = rng.uniform(r, inp, bound=1.0 / math.sqrt(inp))
            lw[p + "B"] = rng.randn(out, r, std=0.01, dtype=torch.float32)
        layers.append(lw)

    def rows(width):
        t = torch.zeros(n + 1, width, dtype=BF16, device=DEV)
        t[:n] = rng.randn(n, width)
        return t

    acts = {"layer_in": [rows(D) for _ in range(case["L"])], "final_in": rows(D),
            "concat_input_ids": rng.ids(n, m["V"])}
    if case["saved"]:
        acts["mlp_gate_up"] = [rows(2 * I) for _ in range(case["L"])]
    return m, w, layers, acts, lens


def _rope_scaling(m):
    if m["rope"] is None:
        return None
    return {"rope_type": "llama3", "factor": m["rope"], "low_freq_factor": 1.0, "high_freq_factor": 4.0,
            "original_max_position_embeddings": 8192.0}


class _Cycle:
    """A built backward service with its activation store, closed when dropped."""

    def __init__(self, case, seed):
        from deltaserve_amd.bwd_services.registry import get_service

        m, w, layers, acts, lens = _cycle_inputs(case, seed)
        r, projs = case["r"], _projs(case)
        head = "model.embed_tokens.weight" if m["tie"] else "lm_head.weight"
        base = {head: w["lm"], "model.norm.weight": w["norm"]}
        ft, served = {}, {}
        for i, lw in enumerate(layers):
            p = f"model.layers.{i}."
            base[p + "self_attn.qkv_proj.weight"], base[p + "self_attn.o_proj.weight"] = lw["qkv"], lw["o"]
            base[p + "mlp.gate_up_proj.weight"], base[p + "mlp.down_proj.weight"] = lw["gate_up"], lw["down"]
            base[p + "input_layernorm.weight"] = lw["in_ln"]
            base[p + "post_attention_layernorm.weight"] = lw["post_ln"]
            if "q_norm" in lw:
                base[p + "self_attn.q_norm.weight"], base[p + "self_attn.k_norm.weight"] = lw["q_norm"], lw["k_norm"]
            served[i] = {}
            for x in projs:
                out, inp = _proj_shapes(m)[x]
                key = f"base_model.model.model.layers.{i}.{'mlp' if x in ('gate', 'up', 'down') else 'self_attn'}.{x}_proj.lora_"
                ft[key + "A.weight"], ft[key + "B.weight"] = lw[x + "A"], lw[x + "B"]
                served[i][x] = {"a": torch.zeros(2, 1, r, inp, dtype=BF16, device=DEV),
                                "b": torch.zeros(2, 1, out, r, dtype=BF16, device=DEV)}
        n = sum(lens)
        meta = dict(hidden_size=m["D"], num_hidden_layers=case["L"], num_attention_heads=m["Hq"],
                    num_key_value_heads=m["Hkv"], head_dim=m["Hd"], intermediate_size=m["I"],
                    vocab_size=m["V"], rope_theta=m["theta"], rope_scaling=_rope_scaling(m),
                    rms_norm_eps=m["eps"], lora_scaling=2.0, learning_rate=1e-4, weight_decay=0.0,
                    gamma=1.0, lm_head_key=head, norm_weight_key="model.norm.weight",
                    max_saved_finetuning_tokens=n)
        if case["pause"]:
            meta["backward_pause_boundaries"] = True
        self.svc = get_service(m["family"])(0)
        self.svc.shared = {"base": base, "ft": ft, "meta": meta}
        err = self.svc._on_weights_shared()
        if err:
            raise RuntimeError(err)
        self.svc.lora_buffers = {"slot": 1, "layers": served}
        self.svc._on_lora_buffers()
        self.acts, self.lens, self.n, self.L, self.projs = acts, lens, n, case["L"], projs

    def __del__(self):
        svc = getattr(self, "svc", None)
        if svc is not None:
            svc.close()

    def run(self):
        loss, nv = self.svc.process_backward(self.acts, self.lens, self.n, epoch=0)
        pairs = [self.svc.lora[i][p][ab] for i in range(self.L) for p in self.projs for ab in "AB"]
        out = {"loss": loss, "n_valid": nv, "grads": [t.grad for t in pairs]}
        if 2 * len(pairs) + 2 <= 64:
            out["masters"] = [t.detach() for t in pairs]
        return out


class _SaveStep:
    """One forward step of the serving worker as the save points see it."""

    def __init__(self, case, seed):
        from deltaserve_amd import capture

        m, rng = MODELS[case["model"]], _Rng(seed)
        dt = {"bf16": BF16, "f16": torch.float16, "f32": torch.float32}[case["dtype"]]
        self.capture, self.layers = capture, case["layers"]
        self.store = capture.ActivationStore(
            case["layers"], m["D"], case["max_saved"], device=DEV,
            intermediate_size=m["I"] if case["gate_up"] else 0)
        T = case["rows"]
        self.x = [rng.randn(T, m["D"], dtype=dt) for _ in range(case["layers"] + 1)]
        self.r = [rng.randn(T, m["D"], dtype=dt) if case["resid"] else None for _ in range(case["layers"] + 1)]
        self.gu = [rng.randn(T, 2 * m["I"], dtype=dt) for _ in range(case["layers"])] if case["gate_up"] else []
        self.ids = rng.ids(T, m["V"])
        self.pos = torch.randperm(T, generator=torch.Generator().manual_seed(seed))[:case["ft"]].sort().values
        self.state = self.store.arm_op_step(self.pos, case["ft"], 0)

    def run(self):
        C, st = self.capture, self.store
        with C.active_state(self.state):
            for i in range(self.layers):
                C.dserve_save_rows(self.x[i], self.r[i], st.marker, st.slot(i, C.SLOT_LAYER_IN))
                if self.gu:
                    C.dserve_save_rows(self.gu[i], None, st.marker, st.slot(i, C.SLOT_GATE_UP))
            C.dserve_save_rows(self.x[-1], self.r[-1], st.marker, st.final_slot)
        st.save_final_ids(self.ids, self.state)
        return {"layer_in": st.layer_in, "final_in": st.final_in, "gate_up": st.mlp_gate_up,
                "ids": st.concat_input_ids}


class _Op:
    """Inputs of one op of deltaserve_amd.ops and the call."""

    def __init__(self, case, seed):
        from deltaserve_amd import ops

        self.t = t = _op_inputs(case, seed)
        kind = case["kind"]
        if kind == "attn_fwd":
            self.call = lambda: ops.attn_forward(t["q"], t["k"], t["v"], t["lens"], case["Hq"], case["Hkv"])
        elif kind == "attn_bwd":
            _, o32, lse = ops.attn_forward(t["q"], t["k"], t["v"], t["lens"], case["Hq"], case["Hkv"])
            self.call = lambda: ops.attn_backward(t["q"], t["k"], t["v"], o32, lse, t["g"], t["lens"],
                                                  case["Hq"], case["Hkv"])
        elif kind == "glu":
            self.call = lambda: ops.gemm_glu(t["x"], t["w"], t["z"], t["b"])
        elif kind == "dx":
            self.call = lambda: ops.gemm_nt(t["g"], t["w"], t["z"], t["a"], out_dtype=torch.float32, b_kn=True)
        elif kind == "head":
            self.call = lambda: ops.head_backward(t["x"], t["w"], t["ids"], t["lens"])
        else:
            passes = [(g, z, w, gz, gb, 2.0, i < 2) for i, (g, z, w, gz, gb) in enumerate(t["passes"])]

            def call():
                ops.lora_dual_batch(passes, case["n"], entry="dsb_op_lora_dual_noalloc")
                return [(p[3], p[4]) for p in passes]

            self.call = call

    def run(self):
        return self.call()


def _op_inputs(case, seed):
    rng, kind = _Rng(seed), case["kind"]
    if kind in ("attn_fwd", "attn_bwd"):
        lens, hd = lengths(case), case["Hd"]
        n = sum(lens)
        t = {"lens": lens, "q": rng.randn(n, case["Hq"] * hd), "k": rng.randn(n, case["Hkv"] * hd),
             "v": rng.randn(n, case["Hkv"] * hd)}
        if kind == "attn_bwd":
            t["g"] = rng.randn(n, case["Hq"] * hd)
        return t
    if kind == "glu":
        D, I, r, M = case["D"], case["I"], case["r"], case["M"]
        return {"x": rng.randn(M, D), "w": rng.randn(2 * I, D, std=0.02), "z": rng.randn(M, 2 * r, std=0.5),
                "b": rng.randn(2 * I, 2 * r, std=0.02)}
    if kind == "dx":
        D, I, r, M = case["D"], case["I"], case["r"], case["M"]
        return {"g": rng.randn(M, 2 * I), "w": rng.randn(2 * I, D, std=0.02),
                "z": rng.randn(M, 2 * r, std=0.5), "a": rng.randn(2 * r, D, std=0.02)}
    if kind == "head":
        lens = lengths(case)
        n = sum(lens)
        return {"lens": lens, "x": rng.randn(n, case["D"]), "w": rng.randn(case["V"], case["D"], std=0.02),
                "ids": rng.ids(n, case["V"])}
    n, C, r = case["n"], case["C"], case["r"]
    return {"passes": [(rng.randn(n, C), rng.randn(n, r), rng.randn(r, C, std=0.02),
                        torch.zeros(n, r, dtype=BF16, device=DEV),
                        torch.zeros(*((C, r) if i < 2 else (r, C)), device=DEV))
                       for i in range(case["count"])]}


def prepare(case, seed):
    if case["kind"] == "cycle":
        return _Cycle(case, seed)
    return _SaveStep(case, seed) if case["kind"] == "save" else _Op(case, seed)


def run(state):
    return state.run()


# ---------------------------------------------------------------- work and tolerance

def work(case):
    """Bytes (each input read once, each output written once) and operations of one pass."""
    kind = case["kind"]
    if kind == "save":
        m, e = MODELS[case["model"]], {"bf16": 2, "f16": 2, "f32": 4}[case["dtype"]]
        rows = case["ft"]
        per = m["D"] * (e * (2 if case["resid"] else 1) + 2)
        b = (case["layers"] + 1) * per + case["layers"] * (2 * m["I"] * (e + 2) if case["gate_up"] else 0)
        return {"bytes": rows * (b + 16) + 16 * case["max_saved"], "flops": 0}
    if kind in ("attn_fwd", "attn_bwd"):
        lens, hd = lengths(case), case["Hd"]
        n, S = sum(lens), sum(x * (x + 1) for x in lens)
        q, kv = case["Hq"] * hd, case["Hkv"] * hd
        if kind == "attn_fwd":  # q, k, v in; ctx, its fp32 copy and the row statistics out
            return {"bytes": n * (2 * (q + 2 * kv) + 6 * q + 4 * case["Hq"]), "flops": 2 * q * S}
        return {"bytes": n * (2 * (q + 2 * kv) + 6 * q + 4 * case["Hq"] + 2 * (q + 2 * kv)), "flops": 5 * q * S}
    if kind == "glu":
        D, I, r2, M = case["D"], case["I"], 2 * case["r"], case["M"]
        return {"bytes": 2 * (M * (D + r2) + 2 * I * (D + r2) + 3 * M * I), "flops": 4 * M * I * (D + r2)}
    if kind == "dx":
        D, I, r2, M = case["D"], case["I"], 2 * case["r"], case["M"]
        return {"bytes": 2 * (M * (2 * I + r2) + D * (2 * I + r2)) + 4 * M * D, "flops": 2 * M * D * (2 * I + r2)}
    if kind == "head":
        lens = lengths(case)
        n, D, V = sum(lens), case["D"], case["V"]
        return {"bytes": 2 * n * D + 2 * V * D + 4 * n * D + 8 * n,
                "flops": 4 * sum(max(x - 1, 0) for x in lens) * D * V}
    if kind == "lora":
        n, C, r = case["n"], case["C"], case["r"]
        return {"bytes": case["count"] * (2 * n * C + 4 * n * r + 6 * r * C), "flops": case["count"] * 4 * n * C * r}
    m, L, r, lens = MODELS[case["model"]], case["L"], case["r"], lengths(case)
    D, I, V, q, kv = m["D"], m["I"], m["V"], m["Hq"] * m["Hd"], m["Hkv"] * m["Hd"]
    n, M, S = sum(lens), sum(max(x - 1, 0) for x in lens), sum(x * (x + 1) for x in lens)
    shapes = _proj_shapes(m)
    dense = L * n * (4 * D * (q + 2 * kv) + 4 * D * q + (6 if case["saved"] else 10) * D * I)
    lora = L * n * 6 * r * sum(a + b for p, (a, b) in shapes.items() if p in _projs(case))
    params = L * (D * (q + 2 * kv) + D * q + 3 * D * I) + V * D
    adapter = L * r * sum(a + b for p, (a, b) in shapes.items() if p in _projs(case))
    # weights once, the store once, and per LoRA parameter the master, both moments and the
    # gradient (read and written, 32 bytes) and the served bf16 copy
    return {"bytes": 2 * params + 2 * n * ((L + 1) * D + (2 * I * L if case["saved"] else 0)) + 34 * adapter,
            "flops": dense + lora + L * 7 * q * S + 4 * M * D * V}


def tolerance(case):
    kind = case["kind"]
    if kind == "save":
        return "exact"
    # Measured against 64 bits and, for the cycles, between two orders of every product's sums
    # (other tiles and vocabulary slices): attention 0.0019-0.0024 (bf16 results and operands), gate/up
    # and h 0.0017 and 0.0031, the fp32 dX 1.2e-6, the head's fp32 dH 8e-6 (its softmax term passes
    # bf16), the LoRA pass 0.0017 (bf16 grad_Z); a cycle's gradients 0.0065-0.0116 between two orders
    # (largest single difference 0.03-0.09) and 0.009-0.016 against 64 bits over 2-4 layers.
    return {"attn_fwd": {"rel": 0.008}, "attn_bwd": {"rel": 0.01}, "glu": {"rel": 0.008},
            "dx": {"rel": 1e-5}, "head": {"rel": 4e-5, "max": 2e-3}, "lora": {"rel": 0.006},
            "cycle": {"rel": 0.03, "max": 0.35}}[kind]


# ---------------------------------------------------------------- the same in 64 bits

def _attention(q, k, v, lens, Hq, Hkv, fn):
    """fn(q_h, k_h, v_h, mask, h, rows) per sequence and q-head over packed fp64 rows."""
    hd, st = q.shape[1] // Hq, 0
    for s in lens:
        rows = slice(st, st + s)
        mask = torch.ones(s, s, dtype=torch.bool, device=DEV).triu(1)
        for h in range(Hq):
            g = h // (Hq // Hkv)
            fn(q[rows, h * hd:(h + 1) * hd].double(), k[rows, g * hd:(g + 1) * hd].double(),
               v[rows, g * hd:(g + 1) * hd].double(), mask, h, rows)
        st += s


def _attn_fwd64(q, k, v, lens, Hq, Hkv):
    n, hd = q.shape[0], q.shape[1] // Hq
    o = torch.empty(n, Hq * hd, dtype=F64, device=DEV)
    lse = torch.empty(Hq, n, dtype=F64, device=DEV)

    def head(qh, kh, vh, mask, h, rows):
        s = (qh @ kh.t()).mul_(1 / math.sqrt(hd)).masked_fill_(mask, -math.inf)
        z = torch.logsumexp(s, 1, keepdim=True)
        o[rows, h * hd:(h + 1) * hd] = s.sub_(z).exp_() @ vh
        lse[h, rows] = z[:, 0] / math.log(2.0)

    _attention(q, k, v, lens, Hq, Hkv, head)
    return o, lse


def _attn_bwd64(q, k, v, g, lens, Hq, Hkv):
    hd = q.shape[1] // Hq
    dq, dk, dv = (torch.zeros(t.shape, dtype=F64, device=DEV) for t in (q, k, v))

    def head(qh, kh, vh, mask, h, rows):
        c = 1 / math.sqrt(hd)
        gk = slice((h // (Hq // Hkv)) * hd, (h // (Hq // Hkv) + 1) * hd)
        gh = g[rows, h * hd:(h + 1) * hd].double()
        p = torch.softmax((qh @ kh.t()).mul_(c).masked_fill_(mask, -math.inf), 1)
        dv[rows, gk] += p.t() @ gh
        ds = gh @ vh.t()
        ds = ds.sub_((ds * p).sum(1, keepdim=True)).mul_(p)
        dq[rows, h * hd:(h + 1) * hd] = (ds @ kh) * c
        dk[rows, gk] += (ds.t() @ qh) * c

    _attention(q, k, v, lens, Hq, Hkv, head)
    return dq, dk, dv


class _Attention64(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, lens, Hq, Hkv):
        ctx.save_for_backward(q, k, v)
        ctx.args = (lens, Hq, Hkv)
        return _attn_fwd64(q, k, v, lens, Hq, Hkv)[0]

    @staticmethod
    def backward(ctx, g):
        return (*_attn_bwd64(*ctx.saved_tensors, g, *ctx.args), None, None, None)


def _norm64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope64(m, lens):
    hd = m["Hd"]
    inv = 1.0 / m["theta"] ** (torch.arange(0, hd, 2, dtype=F64) / hd)
    if m["rope"] is not None:
        wl = 2 * math.pi / inv
        smooth = ((8192.0 / wl - 1.0) / 3.0).clamp(0, 1)
        inv = (1 - smooth) * inv / m["rope"] + smooth * inv
    pos = torch.cat([torch.arange(s, dtype=F64) for s in lens])
    ang = pos[:, None] * inv[None]
    return ang.cos().to(DEV)[:, None], ang.sin().to(DEV)[:, None]


def _rotate(x, cos, sin):
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _head64(x, w, ids, lens):
    """(loss, n_valid, dH) of the packed rows x in 64 bits, the vocabulary in slices."""
    n, V, dev = x.shape[0], w.shape[0], x.device
    valid = torch.cat([torch.arange(s) < s - 1 for s in lens]).to(dev)
    rows = valid.nonzero()[:, 0]
    tgt = ids[rows + 1]
    xr, nv = x[rows].double(), len(rows)
    step = 16384
    lse = torch.full((nv,), -math.inf, dtype=F64, device=dev)
    at = torch.empty(nv, dtype=F64, device=dev)
    for c in range(0, V, step):
        s = xr @ w[c:c + step].double().t()
        lse = torch.logaddexp(lse, torch.logsumexp(s, 1))
        here = ((tgt >= c) & (tgt < c + step)).nonzero()[:, 0]
        at[here] = s[here, tgt[here] - c]
    d = torch.zeros(nv, x.shape[1], dtype=F64, device=dev)
    for c in range(0, V, step):
        wc = w[c:c + step].double()
        d += (xr @ wc.t()).sub_(lse[:, None]).exp_() @ wc
    d -= w[tgt].double()
    dH = torch.zeros(n, x.shape[1], dtype=F64, device=dev)
    dH[rows] = d / max(nv, 1)
    return float((lse - at).sum() / max(nv, 1)), nv, dH


def _cycle64(case, seed):
    m, w, layers, acts, lens = _cycle_inputs(case, seed)
    n, projs, eps, scale = sum(lens), _projs(case), m["eps"], 2.0
    hd, Hq, Hkv, I = m["Hd"], m["Hq"], m["Hkv"], m["I"]
    q, kv = Hq * hd, Hkv * hd
    cos, sin = _rope64(m, lens)
    fin = acts["final_in"][:n].double().requires_grad_()
    normed = _norm64(fin, w["norm"], eps)
    loss, nv, dH = _head64(normed.detach(), w["lm"], acts["concat_input_ids"], lens)
    g, = torch.autograd.grad(normed, fin, dH)
    del normed, dH
    grads = [None] * case["L"]
    for i in reversed(range(case["L"])):
        lw = layers[i]
        A = {p + ab: lw[p + ab].double().requires_grad_() for p in projs for ab in "AB"}
        x = acts["layer_in"][i][:n].double().requires_grad_()

        def proj(p, t, wt):
            y = t @ wt.double().t()
            return y + scale * (t @ A[p + "A"].t()) @ A[p + "B"].t() if p in projs else y

        xn = _norm64(x, lw["in_ln"], eps)
        wq, wk, wv = lw["qkv"].split([q, kv, kv])
        qh, kh = proj("q", xn, wq).view(n, Hq, hd), proj("k", xn, wk).view(n, Hkv, hd)
        if m["family"] == "qwen3":
            qh, kh = _norm64(qh, lw["q_norm"], eps), _norm64(kh, lw["k_norm"], eps)
        c = _Attention64.apply(_rotate(qh, cos, sin).reshape(n, q), _rotate(kh, cos, sin).reshape(n, kv),
                               proj("v", xn, wv), lens, Hq, Hkv)
        mid = x + proj("o", c, lw["o"])
        xn2 = _norm64(mid, lw["post_ln"], eps)
        gate, up = proj("gate", xn2, lw["gate_up"][:I]), proj("up", xn2, lw["gate_up"][I:])
        if case["saved"]:  # the forward's values in place of the recomputed ones, same derivative
            sg, su = acts["mlp_gate_up"][i][:n].double().split(I, 1)
            gate, up = gate + (sg - gate).detach(), up + (su - up).detach()
        y = mid + proj("down", torch.nn.functional.silu(gate) * up, lw["down"])
        keys = [p + ab for p in projs for ab in "AB"]
        got = torch.autograd.grad(y, [x] + [A[k] for k in keys], g)
        del xn, qh, kh, c, mid, xn2, gate, up, y
        g, gl = got[0], got[1:]
        norm = math.sqrt(sum(float((t * t).sum()) for t in gl))
        grads[i] = [t * min(1.0, 1.0 / (norm + 1e-6)) for t in gl]
    flat = [t for per in grads for t in per]
    out = {"loss": loss, "n_valid": nv, "grads": flat}
    if 2 * len(flat) + 2 <= 64:  # AdamW's first step, no decay
        masters = [layers[i][p + ab].double() for i in range(case["L"]) for p in projs for ab in "AB"]
        out["masters"] = [t - 1e-4 * x / (x.abs() + 1e-8) for t, x in zip(masters, flat)]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "save":
        return None  # copies: compared bit by bit
    if kind == "cycle":
        return _cycle64(case, seed)
    t = _op_inputs(case, seed)
    if kind == "attn_fwd":
        o, lse = _attn_fwd64(t["q"], t["k"], t["v"], t["lens"], case["Hq"], case["Hkv"])
        return o, o, lse
    if kind == "attn_bwd":
        return _attn_bwd64(t["q"], t["k"], t["v"], t["g"], t["lens"], case["Hq"], case["Hkv"])
    if kind == "glu":
        gu = t["x"].double() @ t["w"].double().t() + t["z"].double() @ t["b"].double().t()
        gate, up = gu.split(case["I"], 1)
        return gu, torch.nn.functional.silu(gate) * up
    if kind == "dx":
        return t["g"].double() @ t["w"].double() + t["z"].double() @ t["a"].double()
    if kind == "head":
        return _head64(t["x"], t["w"], t["ids"], t["lens"])
    out = []
    for i, (g, z, w, _, _) in enumerate(t["passes"]):
        gb = 2.0 * (g.double().t() @ z.double())
        out.append((g.double() @ w.double().t(), gb if i < 2 else gb.t()))
    return out
