"""The work a user of this framework has it do, as measurable cases.

A PLM decoder runs ``M = k + k^2`` rows per round (42 at k = 6, 56 at k = 7, 110 at k = 10) through
every linear of the model, ends the round with the LM-head verify and the auxiliary decode of its k
verify rows, and reads the prompt in prefill chunks of 64 to 640 rows. Rounds and chunks are captured
once as HIP graphs and replayed, as the decoder does; the chained round is one launch of its own.
Weights are kept as a served model keeps them: one packed copy (``fast_gemm.release``), the tile
tables installed, workspaces sized once. Several layers with weights of their own are run per pass, so
that weights come from memory and not from a cache that a whole model would not fit.

Kinds of case (``"kind"``):

* ``linear``  — one call of the dispatch (``fast_gemm``), eager;
* ``round``   — the linears of ``layers`` decoder blocks, one launch per linear, captured;
* ``chain``   — the linears of ``layers`` GPT-style blocks in one chained launch (``LinearChain``);
* ``lora``    — the gated-LoRA QKV projection of ``layers`` layers, captured;
* ``verify``  — the fused LM-head verify (packed or row-major weights), eager;
* ``end``     — the end of a round: verify with the verify rows' logits, then their auxiliary decode;
* ``prefill`` — the linears of ``layers`` decoder blocks at a prefill chunk's width, captured.

``block`` is the decoder block: ``gpt`` (QKV H -> 3H, out H -> H, up H -> F, down F -> H) or ``llama``
(fused grouped QKV, out, and the MLP ``down(silu(gate) * up)`` through ``llama_mlp``).
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "plm-anon_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from plm_amd import _lib, fast_gemm, gated_lora, gemm_tables, tiles, verify, voronoi  # noqa: E402
from plm_amd.chain import Link, LinearChain  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
WORKSPACE = 256 << 20   # reserved once, so that no captured graph outlives a workspace that grew

# (hidden, qkv columns, MLP width) of the Llama-style models and (hidden, MLP width) of the GPT-style ones.
LLAMA = {512: (768, 1408), 768: (1152, 2048), 1024: (1536, 2560), 2048: (3072, 5632), 3072: (4608, 8192)}
GPT = {1024: 4096, 2048: 8192, 2560: 10240}


def listed() -> list[dict]:
    return [
        # The smallest call: one MLP up-projection of a 350M-class model at k = 6, launched eagerly.
        {"name": "linear_350m_k6", "kind": "linear", "M": 42, "N": 4096, "K": 1024, "dtype": "bf16"},
        # A linear no table knows, with ragged sizes: what a width or model outside the tuned set gets.
        {"name": "linear_untuned", "kind": "linear", "M": 33, "N": 5003, "K": 1416, "dtype": "fp16"},
        # A small released model's round: short linears, where launches and latency are all there is.
        {"name": "round_llama512_k6", "kind": "round", "block": "llama", "hidden": 512, "M": 42, "layers": 8,
         "dtype": "fp16"},
        # The 1.3B-shape round at k = 7, launch per linear.
        {"name": "round_gpt2048_k7", "kind": "round", "block": "gpt", "hidden": 2048, "M": 56, "layers": 6,
         "dtype": "bf16"},
        # The relaxed setting's wide round (k = 10) on the 3B-class model.
        {"name": "round_llama3072_k10", "kind": "round", "block": "llama", "hidden": 3072, "M": 110, "layers": 2,
         "dtype": "bf16"},
        # The 1.3B-shape round as one chained launch, in the decoder's default dtype.
        {"name": "chain_gpt2048_k7", "kind": "chain", "block": "gpt", "hidden": 2048, "M": 56, "layers": 6,
         "dtype": "fp16"},
        # The adapter's fused QKV projections at k = 7 (rank 16, rows from the seventh gated).
        {"name": "lora_qkv2048_k7", "kind": "lora", "hidden": 2048, "M": 56, "gate": 7, "rank": 16, "layers": 8,
         "dtype": "bf16"},
        # The verify of a k = 6 round under the floor rule, padded vocabulary.
        {"name": "verify_floor_k6", "kind": "verify", "R": 42, "V": 50304, "K": 2048, "rule": "floor", "packed": True,
         "dtype": "fp16"},
        # The verify on a weight that is still being trained, so that no packed copy can be kept.
        {"name": "verify_rowmajor_k7", "kind": "verify", "R": 56, "V": 50257, "K": 2048, "rule": "nucleus",
         "packed": False, "dtype": "bf16"},
        # The whole end of a k = 7 round: verify, the verify rows' logits, their auxiliary decode.
        {"name": "end_k7", "kind": "end", "k": 7, "V": 50257, "K": 2048, "A": 1024, "dtype": "bf16"},
        # The widest prefill chunk of the 1.3B-shape model.
        {"name": "prefill_gpt2048_640", "kind": "prefill", "block": "gpt", "hidden": 2048, "M": 640, "layers": 2,
         "dtype": "bf16"},
        # A ragged, shorter chunk of the 3B-class model.
        {"name": "prefill_llama3072_200", "kind": "prefill", "block": "llama", "hidden": 3072, "M": 200, "layers": 1,
         "dtype": "fp16"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _layers(rng, kind: str, block: str, hidden: int, M: int, most: int) -> int:
    """Up to ``most`` layers, within the listed cases' cost."""
    if kind == "prefill":
        fit = int(120e9 // (2 * M * _block_params(block, hidden)))
    else:
        fit = int(600e6 // (2 * _block_params(block, hidden)))
    return rng.randint(1, max(1, min(most, fit)))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "round", "round", "chain", "lora", "verify", "verify", "end", "prefill", "prefill"])
    dtype = rng.choice(["bf16", "fp16"])
    widths = [2, 6, 12, 20, 30, 42, 56, 72, 90, 110]   # k + k^2
    if kind == "linear":
        return {"kind": kind, "M": _log_int(rng, 1, 128), "N": _log_int(rng, 64, 16384),
                "K": 8 * _log_int(rng, 16, 1024), "dtype": dtype}
    if kind == "round":
        block = rng.choice(["gpt", "llama"])
        hidden = rng.choice(sorted(GPT if block == "gpt" else LLAMA))
        M = rng.choice(widths) if rng.random() < 0.7 else rng.randint(1, 128)
        return {"kind": kind, "block": block, "hidden": hidden, "M": M,
                "layers": _layers(rng, kind, block, hidden, M, 8), "dtype": dtype}
    if kind == "chain":
        hidden = rng.choice(sorted(GPT))
        M = rng.choice(widths)
        return {"kind": kind, "block": "gpt", "hidden": hidden, "M": M,
                "layers": _layers(rng, kind, "gpt", hidden, M, 6), "dtype": dtype}
    if kind == "lora":
        k = rng.choice([6, 7, 10])
        hidden = rng.choice([2048, 3072] if k != 6 else sorted(LLAMA))
        return {"kind": kind, "hidden": hidden, "M": k + k * k, "gate": k, "rank": 8 * rng.randint(1, 8),
                "layers": rng.randint(1, 8), "dtype": dtype}
    if kind == "verify":
        return {"kind": kind, "R": rng.randint(1, 64), "V": _log_int(rng, 2000, 50304),
                "K": 8 * rng.randint(64, 256), "rule": rng.choice(["nucleus", "floor"]),
                "packed": rng.random() < 0.6, "dtype": dtype}
    if kind == "end":
        return {"kind": kind, "k": rng.randint(2, 7), "V": _log_int(rng, 8000, 50304), "K": 8 * rng.randint(64, 256),
                "A": rng.choice([256, 512, 1024, 2048]), "dtype": dtype}
    block = rng.choice(["gpt", "llama"])
    hidden = rng.choice([1024, 2048] if block == "gpt" else sorted(LLAMA))
    M = rng.choice([64, 128, 192, 256, 320, 384, 448, 512, 576, 640]) if rng.random() < 0.5 else rng.randint(64, 640)
    return {"kind": kind, "block": block, "hidden": hidden, "M": M,
            "layers": _layers(rng, kind, block, hidden, M, 2), "dtype": dtype}


# ------------------------------------------------------------------------------------------ inputs


def _block_shapes(block: str, hidden: int) -> list[tuple[str, int, int]]:
    if block == "gpt":
        return [("qkv", 3 * hidden, hidden), ("out", hidden, hidden), ("up", GPT[hidden], hidden),
                ("down", hidden, GPT[hidden])]
    qkv, mlp = LLAMA[hidden]
    return [("qkv", qkv, hidden), ("out", hidden, hidden), ("gate_up", 2 * mlp, hidden), ("down", hidden, mlp)]


def _block_params(block: str, hidden: int) -> int:
    return sum(n * k for _, n, k in _block_shapes(block, hidden))


class _Inputs:
    """Seeded tensors on the GPU, drawn in fp32 and rounded to the case's dtype."""

    def __init__(self, case: dict, seed: int):
        self.device = torch.device("cuda", torch.cuda.current_device())
        self.dtype = DTYPES[case["dtype"]]
        self.gen = torch.Generator(device=self.device).manual_seed(1_000_003 * seed + 17)

    def normal(self, *shape: int, std: float = 1.0) -> torch.Tensor:
        return (std * torch.randn(*shape, generator=self.gen, device=self.device)).to(self.dtype)

    def weight(self, n: int, k: int, gain: float = 1.0) -> torch.Tensor:
        return self.normal(n, k, std=gain / math.sqrt(k))

    def ids(self, n: int, below: int) -> torch.Tensor:
        return torch.randint(0, below, (n,), generator=self.gen, device=self.device, dtype=torch.int64)


def _draw_inputs(case: dict, seed: int) -> dict:
    """The case's tensors, the same for ``prepare`` and ``exact``."""
    g = _Inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        return {"x": g.normal(case["M"], case["K"]), "w": g.weight(case["N"], case["K"])}
    if kind in ("round", "prefill"):
        hidden, M = case["hidden"], case["M"]
        # Each block's two inputs as the norms before them give them.
        return {"layers": [{"x": g.normal(M, hidden), "h": g.normal(M, hidden),
                            "w": [g.weight(n, k) for _, n, k in _block_shapes(case["block"], hidden)]}
                           for _ in range(case["layers"])]}
    if kind == "chain":
        return {"x": g.normal(case["M"], case["hidden"]),
                "w": [g.weight(n, k) for _ in range(case["layers"]) for _, n, k in _block_shapes("gpt", case["hidden"])]}
    if kind == "lora":
        hidden, rank = case["hidden"], case["rank"]
        kv = (LLAMA[hidden][0] - hidden) // 2
        return {"layers": [{"x": g.normal(case["M"], hidden), "w": g.weight(hidden + 2 * kv, hidden),
                            "a": g.weight(3 * rank, hidden), "b": [g.weight(n, rank) for n in (hidden, kv, kv)]}
                           for _ in range(case["layers"])]}
    if kind == "verify":
        # Logits with a language model's spread (std about 2.5); proposals over the whole vocabulary.
        return {"x": g.normal(case["R"], case["K"]), "w": g.weight(case["V"], case["K"], 2.5),
                "pending": g.ids(case["R"], case["V"])}
    k = case["k"]
    return {"x": g.normal(k + k * k, case["K"]), "w": g.weight(case["V"], case["K"], 2.5),
            "pending": g.ids(k, case["V"])[: k - 1].contiguous(), "cells": g.normal(case["A"], case["K"]),
            "values": g.ids(k, case["A"])}


def _install_tables(hidden: int) -> None:
    """Every tuned tile of this model width, as ``gemm_tables.install`` does for one round width."""
    fast_gemm.install(gemm_tables.read_table(hidden))
    fast_gemm.ACT_CONFIGS.update(gemm_tables.read_act_table(hidden))


def _captured(fn) -> dict:
    """``fn`` run once eagerly (first-use packing), then captured; its outputs are the graph's."""
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = fn()
    return {"graph": graph, "outputs": outputs}


def _block(block: str, layer: dict) -> list[torch.Tensor]:
    """One decoder block's linears through the dispatch; attention-out reads the queries' columns."""
    w = layer["w"]
    hidden = layer["x"].shape[1]
    qkv = fast_gemm.fast_gemm(None, layer["x"], w[0])
    out = fast_gemm.fast_gemm(None, qkv[:, :hidden], w[1])
    if block == "llama":
        return [qkv, out, fast_gemm.llama_mlp(layer["h"], w[2], w[3])]
    up = fast_gemm.fast_gemm(None, layer["h"], w[2])
    return [qkv, out, up, fast_gemm.fast_gemm(None, up, w[3])]


def prepare(case: dict, seed: int) -> dict:
    state = _draw_inputs(case, seed)
    kind = case["kind"]
    device = torch.device("cuda", torch.cuda.current_device())
    state["case"] = case
    state["workspace"] = fast_gemm.workspace(device, WORKSPACE)
    if kind == "linear":
        if case["K"] in (512, 768, 1024, 2048, 2560, 3072):
            _install_tables(case["K"])
        fast_gemm.release(state["w"])
    elif kind in ("round", "prefill"):
        _install_tables(case["hidden"])
        for layer in state["layers"]:
            for w in layer["w"]:
                fast_gemm.release(w)
        state.update(_captured(lambda: [y for layer in state["layers"] for y in _block(case["block"], layer)]))
    elif kind == "chain":
        state["chain"], state["outputs"] = _chain(case, state)
    elif kind == "lora":
        _install_tables(case["hidden"])
        for layer in state["layers"]:
            fast_gemm.release(layer["w"])
            layer["stacked"] = gated_lora.stack_b(layer["b"])
        state.update(_captured(lambda: [
            gated_lora.gated_linear(la["x"], la["w"], la["a"], la["b"], case["gate"], lora_b=la["stacked"])
            for la in state["layers"]]))
    elif kind == "verify":
        if case["packed"]:
            fast_gemm.release(state["w"])
    else:
        scheme = voronoi.LogitVoronoiAuxiliary(case["A"], case["K"], case["V"], dtype=DTYPES[case["dtype"]])
        scheme.auxiliary_vocabulary = state["cells"]
        state["scheme"] = scheme.to(device)
        state["logits"] = torch.empty(case["k"], (case["V"] + 7) // 8 * 8, dtype=state["x"].dtype, device=device)
        run(state)   # packs the LM head (its row-major form stays: the embedding is tied to it) and
        #              builds the scheme's cost table, each once per weight
    return state


def _chain(case: dict, state: dict) -> tuple[LinearChain, list[torch.Tensor]]:
    M, hidden, weights = case["M"], case["hidden"], state["w"]
    outs = [torch.empty(M, w.shape[0], dtype=w.dtype, device=w.device) for w in weights]
    cfg = gemm_tables.round_chain_tile(hidden, M)
    resident = _lib.lib().plm_gemm_packed_resident_workgroups(_lib.DTYPE_CODES[state["x"].dtype], M,
                                                              _lib.Tile.from_config(cfg))
    links = [Link(state["x"] if i == 0 else outs[i - 1][:, : w.shape[1]], w, outs[i], i - 1,
                  tiles.packed_chain_split(w.shape[0], w.shape[1], cfg, resident))
             for i, w in enumerate(weights)]
    return LinearChain(links, cfg), outs


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return fast_gemm.fast_gemm(None, state["x"], state["w"])
    if kind == "chain":
        state["chain"].run()
        return state["outputs"]
    if kind == "verify":
        return verify.lm_head_verify(state["x"], state["w"], state["pending"], _threshold(case["rule"]),
                                     round_to=case["dtype"], packed=case["packed"], rule=case["rule"])
    if kind == "end":
        accept, argmax = verify.lm_head_verify_logits(state["x"], state["w"], state["pending"], case["k"] - 1,
                                                      _threshold("nucleus"), state["logits"], case["k"])
        logits = state["logits"][:, : case["V"]]
        tokens = state["scheme"].decode_unmasked(logits, None, state["w"], state["values"])
        return accept, argmax, logits, tokens
    state["graph"].replay()
    return state["outputs"]


def _threshold(rule: str) -> float:
    return 0.94 if rule == "nucleus" else 1e-4   # top-p, or the floor rule's epsilon


# ------------------------------------------------------------------------------- what is measured


def _linear_work(M: int, shapes) -> dict:
    return {"bytes": sum(2 * (n * k + M * k + M * n) for n, k in shapes), "flops": sum(2 * M * n * k for n, k in shapes)}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "linear":
        return _linear_work(case["M"], [(case["N"], case["K"])])
    if kind in ("round", "chain", "prefill"):
        M, hidden = case["M"], case["hidden"]
        one = _linear_work(M, [(n, k) for _, n, k in _block_shapes(case["block"], hidden)])
        if case["block"] == "llama":
            # The MLP is one call: its activations [M, F] are not among its inputs and outputs.
            one["bytes"] -= 2 * M * 3 * LLAMA[hidden][1]
        return {key: case["layers"] * value for key, value in one.items()}
    if kind == "lora":
        M, n, k, r = case["M"], LLAMA[case["hidden"]][0], case["hidden"], case["rank"]
        one = _linear_work(M, [(n, k)])
        gated = M - case["gate"]
        return {"bytes": case["layers"] * (one["bytes"] + 2 * (3 * r * k + n * r)),
                "flops": case["layers"] * (one["flops"] + 2 * gated * (3 * r * k + n * r))}
    if kind == "verify":
        R, V, K = case["R"], case["V"], case["K"]
        return {"bytes": 2 * (V * K + R * K) + 17 * R, "flops": 2 * R * V * K}
    k, V, K, A = case["k"], case["V"], case["K"], case["A"]
    R = k + k * k
    # The decode reads each verify row's logits and its 128 shortlisted tokens' costs.
    return {"bytes": 2 * (V * K + R * K) + 17 * R + 2 * 2 * k * V + 2 * k * 128 * A, "flops": 2 * R * V * K}


def tolerance(case: dict):
    kind = case["kind"]
    bf16 = case["dtype"] == "bf16"
    if kind == "verify":
        return "exact"
    # A sum in another order moves a result across a rounding midpoint now and then: one output step
    # (2^-8 or 2^-11 of the value at most), for few of them.
    step = 2.0 ** -7 if bf16 else 2.0 ** -10
    if kind == "chain":
        # Every block's output is the next one's input, so steps spread over the blocks that follow.
        return {"rel": 2e-2 if bf16 else 5e-3, "max": 0.15 if bf16 else 0.03}
    if kind == "end":
        return {"rel": 4e-4 if bf16 else 2e-4, "max": 2 * step, "differ": 0.0}
    return {"rel": 1.2e-3 if bf16 else 4e-4, "max": 4 * step}


# ---------------------------------------------------------------------------------- in 64 bits


def _mm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x.double() @ w.double().t()


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "verify":
        return None   # decisions and token ids
    t = _draw_inputs(case, seed)
    if kind == "linear":
        return _mm(t["x"], t["w"])
    if kind in ("round", "prefill"):
        got = []
        for layer in t["layers"]:
            w = layer["w"]
            qkv = _mm(layer["x"], w[0])
            out = _mm(qkv[:, : case["hidden"]], w[1])
            up = _mm(layer["h"], w[2])
            if case["block"] == "llama":
                gate, up = up.chunk(2, dim=1)
                got += [qkv, out, _mm(gate * torch.sigmoid(gate) * up, w[3])]
            else:
                got += [qkv, out, up, _mm(up, w[3])]
        return got
    if kind == "chain":
        got, x = [], t["x"]
        for w in t["w"]:
            x = _mm(x[:, : w.shape[1]], w)
            got.append(x)
        return got
    if kind == "lora":
        got = []
        for la in t["layers"]:
            y, g, r = _mm(la["x"], la["w"]), case["gate"], case["rank"]
            h = _mm(la["x"][g:], la["a"])
            y[g:] += torch.cat([_mm(h[:, i * r:(i + 1) * r], b) for i, b in enumerate(la["b"])], dim=1)
            got.append(y)
        return got
    return None, None, _mm(t["x"][: case["k"]], t["w"]), None
