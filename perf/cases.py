"""The work this package is measured on: cases of its public entry points at the served decoder's sizes.

The decoder has hidden size 1280, 12 layers (layer 0 a dense SwiGLU of width 6848, the others a mixture of
64 routed experts of width 896, top 6, with 2 shared experts), 10 attention heads of 128 and a vocabulary
of 129280.  A case is a dict of plain values:

``kind``    what is called: ``decode`` (``MoE.decode_rows``), ``prefill`` (``MoE.__call__``), ``dense``
            (``dense_bf16_qmv`` of one of the decoder's projections), ``attention``
            (``paged_decode_attention_qkv``) or ``decoder`` (``Decoder.decode`` and ``logits_rows``).
``rows``    tokens of the call: requests of a decode step, or the tokens of a prefill.
``weights`` ``int8`` or ``bf16`` routed experts (decode, prefill).
``routing`` ``plain`` (random hidden states) or ``zipf`` (a bias over the experts that makes a few of them
            hot, as a page of similar image tokens does) (prefill).
``proj``    which projection (dense).
``attend``  the longest request's attended rows (attention, decoder).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "unlimited-ocr-max_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

E, TOPK, H, F, FS, GROUP = 64, 6, 1280, 896, 1792, 128
HEADS, HEAD_DIM, LAYERS, FFN, VOCAB, PAGE = 10, 128, 12, 6848, 129280, 128
MAX_SEQ, EPS = 2048, 1e-6
POOL_LAYERS = 2  # of the attention cases' page pool (a whole decoder's holds 12)
ZIPF = 0.75 * 1.1
PROJECTIONS = {  # name: (outputs, inputs)
    "qkv": (3 * H, H),
    "o": (H, H),
    "gate_up": (2 * FFN, H),
    "down": (H, FFN),
    "lm_head": (VOCAB, H),
}
DEV = "cuda:0"


def listed() -> list[dict]:
    return [
        # One request's decode step: the smallest call, bound by latency.
        {"name": "decode-int8-b1", "kind": "decode", "rows": 1, "weights": "int8"},
        # The serving batch cap of 8 requests.
        {"name": "decode-int8-b8", "kind": "decode", "rows": 8, "weights": "int8"},
        # The unquantised checkpoint at an odd batch.
        {"name": "decode-bf16-b5", "kind": "decode", "rows": 5, "weights": "bf16"},
        # A decode batch past the serving cap (decode_rows takes up to 64 rows): several requests per expert.
        {"name": "decode-int8-b37", "kind": "decode", "rows": 37, "weights": "int8"},
        # The lm_head of a full serving batch: the largest single weight read of a step.
        {"name": "dense-lm-head-m8", "kind": "dense", "rows": 8, "proj": "lm_head"},
        # The fused q/k/v projection of a larger batch: a narrow output, many rows.
        {"name": "dense-qkv-m20", "kind": "dense", "rows": 20, "proj": "qkv"},
        # RoPE and paged attention of a full batch: a 512-token prompt and the 128-slot ring.
        {"name": "attention-b8", "kind": "attention", "rows": 8, "attend": 640},
        # One page of 273 image rows and a short instruction.
        {"name": "prefill-int8-t291", "kind": "prefill", "rows": 291, "weights": "int8", "routing": "plain"},
        # A 512-token prompt with hot and cold experts.
        {"name": "prefill-int8-t512", "kind": "prefill", "rows": 512, "weights": "int8", "routing": "zipf"},
        # A few prompts together, unquantised checkpoint, ragged length.
        {"name": "prefill-bf16-t1531", "kind": "prefill", "rows": 1531, "weights": "bf16", "routing": "plain"},
        # Eight 512-token prompts together: the largest call.
        {"name": "prefill-int8-t4096", "kind": "prefill", "rows": 4096, "weights": "int8", "routing": "zipf"},
        # The whole decode step of a full batch, replayed from a captured graph as a serving loop does.
        {"name": "decoder-b8", "kind": "decoder", "rows": 8, "attend": 640},
    ]


def _log_int(rng, low: int, high: int) -> int:
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng) -> dict:
    known = [{k: v for k, v in case.items() if k != "name"} for case in listed()]
    while True:
        case = _draw(rng)
        if case not in known:
            return case


def _draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "dense", "dense", "attention", "prefill", "prefill", "prefill", "decoder"])
    if kind == "decode":
        return {"kind": kind, "rows": _log_int(rng, 1, 64), "weights": rng.choice(["int8", "int8", "bf16"])}
    if kind == "dense":
        return {"kind": kind, "rows": _log_int(rng, 1, 64), "proj": rng.choice(sorted(PROJECTIONS))}
    if kind == "attention":
        return {"kind": kind, "rows": rng.randint(1, 8), "attend": _log_int(rng, 16, 1280)}
    if kind == "prefill":
        return {"kind": kind, "rows": _log_int(rng, 16, 4096), "weights": rng.choice(["int8", "int8", "bf16"]),
                "routing": rng.choice(["plain", "zipf"])}
    return {"kind": kind, "rows": rng.randint(1, 8), "attend": _log_int(rng, 16, 1280)}


# ------------------------------------------------------------------------------------------ inputs


class _Draws:
    """Seeded tensors on the GPU."""

    def __init__(self, seed: int) -> None:
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape: int, std: float = 1.0) -> torch.Tensor:
        return torch.randn(shape, generator=self.g, device=DEV) * std

    def weight(self, *shape: int) -> torch.Tensor:
        return self.normal(*shape, std=0.02).to(torch.bfloat16)

    def hidden(self, rows: int) -> torch.Tensor:
        """Hidden states as an RMSNorm leaves them."""
        x = self.normal(rows, H)
        return x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + EPS)


def _quantised(w: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    groups = w.float().unflatten(-1, (-1, GROUP))
    scale = groups.abs().amax(dim=-1) / 127.0
    q = (groups / scale.unsqueeze(-1)).round().clamp(-127, 127).to(torch.int8)
    return q.flatten(-2), scale


def _moe_weights(d: _Draws, int8: bool, zipf: bool = False) -> dict[str, torch.Tensor]:
    """One MoE layer's state dict.  With ``zipf`` the router's column 0 is a bias over the experts (the
    inputs then hold 1 there): ln(rank) steps, a few hot experts and some that are hardly chosen."""
    w = {"gate.gate_score.weight": d.weight(E, H).float()}
    if zipf:
        rank = torch.randperm(E, generator=d.g, device=DEV) + 1
        w["gate.gate_score.weight"][:, 0] = -ZIPF * rank.float().log()
    for proj, n, k in (("gate_proj", F, H), ("up_proj", F, H), ("down_proj", H, F)):
        stack = d.weight(E, n, k)
        if int8:
            w[f"experts.{proj}"], w[f"experts.{proj}_scales"] = _quantised(stack)
        else:
            w[f"experts.{proj}"] = stack
    for proj, n, k in (("gate_proj", FS, H), ("up_proj", FS, H), ("down_proj", H, FS)):
        w[f"shared_experts.{proj}.weight"] = _kblocked(d.weight(n, k))
    return w


def _kblocked(w: torch.Tensor) -> torch.Tensor:
    n, k = w.shape
    return w.view(n, k // 16, 16).permute(1, 0, 2).contiguous()


def _moe_inputs(case: dict, seed: int) -> tuple[dict[str, torch.Tensor], torch.Tensor]:
    d = _Draws(seed)
    zipf = case.get("routing") == "zipf"
    w = _moe_weights(d, case["weights"] == "int8", zipf)
    x = d.hidden(case["rows"])
    if zipf:
        x[:, 0] = 1.0
    return w, x


def _dense_inputs(case: dict, seed: int) -> tuple[torch.Tensor, torch.Tensor]:
    d = _Draws(seed)
    n, k = PROJECTIONS[case["proj"]]
    return d.weight(k // 16, n, 16), d.hidden(case["rows"]) if k == H else d.normal(case["rows"], k)


def _lengths(case: dict) -> list[int]:
    """The attended rows of each request: the first has ``attend``, the others less."""
    rows, attend = case["rows"], case["attend"]
    return [max(1, attend - (r * attend) // (3 * rows)) for r in range(rows)]


def _pool_inputs(d: _Draws, case: dict, layers: int) -> dict[str, torch.Tensor]:
    """A page pool and one step's metadata; each request appends its new row at the end."""
    rows = case["rows"]
    lengths = _lengths(case)
    per = -(-case["attend"] // PAGE)
    pages = rows * per + 1
    order = torch.randperm(pages - 1, generator=d.g, device=DEV)
    table = torch.full((rows, per + 1), pages - 1, dtype=torch.int32, device=DEV)  # the last page is the null page
    table[:, :per] = order.view(rows, per).to(torch.int32)
    last = torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device=DEV)
    return {"pool": d.normal(pages, 2, layers, PAGE, HEADS, HEAD_DIM), "table": table, "last": last}


def _attention_inputs(case: dict, seed: int) -> dict[str, torch.Tensor]:
    d = _Draws(seed)
    return {**_pool_inputs(d, case, POOL_LAYERS), "qkv": d.normal(case["rows"], 3 * H)}


def _rope_tables(dtype: torch.dtype) -> tuple[torch.Tensor, torch.Tensor]:
    inv = 10000.0 ** -(torch.arange(0, HEAD_DIM, 2, dtype=torch.float64, device=DEV) / HEAD_DIM)
    angle = torch.arange(MAX_SEQ, dtype=torch.float64, device=DEV)[:, None] * inv[None, :]
    angle = torch.cat([angle, angle], dim=1)
    return angle.cos().to(dtype), angle.sin().to(dtype)


def _decoder_inputs(case: dict, seed: int):
    d = _Draws(seed)
    w: dict[str, torch.Tensor] = {}
    for i in range(LAYERS):
        p = f"layers.{i}."
        for c in "qkvo":
            w[f"{p}self_attn.{c}_proj.weight"] = _kblocked(d.weight(H, H))
        for norm in ("input_layernorm", "post_attention_layernorm"):
            w[f"{p}{norm}.weight"] = 1 + d.normal(H, std=0.1)
        if i == 0:
            for name, n, k in (("gate_proj", FFN, H), ("up_proj", FFN, H), ("down_proj", H, FFN)):
                w[f"{p}mlp.{name}.weight"] = _kblocked(d.weight(n, k))
        else:
            w.update({f"{p}mlp.{k}": v for k, v in _moe_weights(d, True).items()})
    w["norm.weight"] = 1 + d.normal(H, std=0.1)
    w["lm_head.weight"] = _kblocked(d.weight(VOCAB, H))
    return w, d.hidden(case["rows"]), _pool_inputs(d, case, LAYERS)


# ------------------------------------------------------------------------------------------ the calls


def _paged(pool: dict[str, torch.Tensor], attend: int):
    import uocr_moe

    return uocr_moe.PagedKv(kv_blocks=pool["pool"], lookup_table=pool["table"], attend_lengths=pool["last"],
                            attend_max=attend, write_index=pool["last"])


def prepare(case: dict, seed: int) -> dict:
    import uocr_moe

    kind = case["kind"]
    if kind in ("decode", "prefill"):
        w, x = _moe_inputs(case, seed)
        config = uocr_moe.MoeConfig(int8_experts=case["weights"] == "int8")
        return {"kind": kind, "moe": uocr_moe.MoE(config, w), "x": x}
    if kind == "dense":
        w, x = _dense_inputs(case, seed)
        return {"kind": kind, "w": w, "x": x}
    if kind == "attention":
        i = _attention_inputs(case, seed)
        cos, sin = _rope_tables(torch.float32)
        return {"kind": kind, "qkv": i["qkv"], "kv": _paged(i, case["attend"]), "positions": i["last"].clone(),
                "cos": cos, "sin": sin}
    w, hidden, pool = _decoder_inputs(case, seed)
    decoder = uocr_moe.Decoder(uocr_moe.DecoderConfig(), w, max_seq_len=MAX_SEQ)
    # The residual stream is held in the input: a step starts from a copy, as from a token's embedding.
    state = {"kind": kind, "decoder": decoder, "hidden": hidden, "kv": _paged(pool, case["attend"]),
             "positions": pool["last"].clone(), "buffer": torch.empty_like(hidden)}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(state)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    state["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(state["graph"], stream=side):
        state["logits"] = _step(state)
    return state


def _step(state: dict) -> torch.Tensor:
    state["buffer"].copy_(state["hidden"])
    normed = state["decoder"].decode(state["buffer"], positions=state["positions"], kv=state["kv"])
    return state["decoder"].logits_rows(normed)


def run(state: dict):
    import uocr_moe

    kind = state["kind"]
    if kind == "decode":
        return state["moe"].decode_rows(state["x"])
    if kind == "prefill":
        return state["moe"](state["x"])
    if kind == "dense":
        return uocr_moe.dense_bf16_qmv(state["x"], state["w"])
    if kind == "attention":
        out = uocr_moe.paged_decode_attention_qkv(
            state["qkv"], state["positions"], state["cos"], state["sin"], heads=HEADS, kv=state["kv"], layer_idx=1,
            scale=HEAD_DIM ** -0.5)
        return out, state["kv"].kv_blocks
    state["graph"].replay()
    return state["logits"]


# ------------------------------------------------------------------------------------------ what a pass needs


def _expert_bytes(weights: str) -> int:
    return 3 * F * H * (2 if weights == "bf16" else 1) + (0 if weights == "bf16" else 4 * 3 * F * H // GROUP)


def _moe_work(rows: int, weights: str, routing: str = "plain") -> tuple[float, float]:
    """Bytes and operations of one MoE layer.  The experts chosen are those expected of random rows; under
    the skewed routing about nine in ten of these are."""
    chosen = E * (1 - (1 - TOPK / E) ** rows) * (0.9 if routing == "zipf" else 1.0)
    nbytes = chosen * _expert_bytes(weights) + 3 * FS * H * 2 + E * H * 4 + 2 * rows * H * 4
    return nbytes, 2.0 * rows * (TOPK * 3 * F * H + 3 * FS * H + E * H)


def _dense_work(rows: int, n: int, k: int) -> tuple[float, float]:
    return 2 * n * k + 4 * rows * (n + k), 2.0 * rows * n * k


def _attention_work(case: dict) -> tuple[float, float]:
    rows, total = case["rows"], sum(_lengths(case))
    return 2 * total * H * 4 + rows * (3 + 1 + 2) * H * 4, 4.0 * total * H


def work(case: dict) -> dict:
    kind, rows = case["kind"], case["rows"]
    if kind in ("decode", "prefill"):
        parts = [_moe_work(rows, case["weights"], case.get("routing", "plain"))]
    elif kind == "dense":
        parts = [_dense_work(rows, *PROJECTIONS[case["proj"]])]
    elif kind == "attention":
        parts = [_attention_work(case)]
    else:
        layer = [_dense_work(rows, *PROJECTIONS["qkv"]), _dense_work(rows, *PROJECTIONS["o"]), _attention_work(case)]
        parts = layer * LAYERS + [_moe_work(rows, "int8")] * (LAYERS - 1)
        parts += [_dense_work(rows, *PROJECTIONS[p]) for p in ("gate_up", "down", "lm_head")]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case: dict) -> dict:
    """About four times what the path is off its 64-bit value."""
    if case["kind"] == "prefill":  # bf16 activations, dequantised weights and intermediate
        return {"rel": 1.4e-2}
    if case["kind"] == "decoder":  # 32-bit sums through twelve layers
        return {"rel": 3e-6}
    return {"rel": 2e-6}  # 32-bit sums


# ------------------------------------------------------------------------------------------ the 64-bit values


def _plain(w: torch.Tensor) -> torch.Tensor:
    """A K-blocked weight as float64 [N, K]."""
    kb, n, b = w.shape
    return w.permute(1, 0, 2).reshape(n, kb * b).double()


def _silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    return gate / (1 + torch.exp(-gate)) * up


def _exact_moe(w: dict[str, torch.Tensor], x: torch.Tensor) -> torch.Tensor:
    x = x.double()

    def stack(proj: str, e: int) -> torch.Tensor:
        q = w[f"experts.{proj}"][e].double()
        if f"experts.{proj}_scales" in w:
            q = q * w[f"experts.{proj}_scales"][e].double().repeat_interleave(GROUP, dim=1)
        return q

    probs = torch.softmax(x @ w["gate.gate_score.weight"].double().T, dim=1)
    weight, ids = probs.topk(TOPK, dim=1)
    gate, up, down = (_plain(w[f"shared_experts.{p}.weight"]) for p in ("gate_proj", "up_proj", "down_proj"))
    out = _silu_mul(x @ gate.T, x @ up.T) @ down.T
    for e in ids.unique().tolist():
        row, slot = (ids == e).nonzero(as_tuple=True)
        h = _silu_mul(x[row] @ stack("gate_proj", e).T, x[row] @ stack("up_proj", e).T)
        out.index_add_(0, row, (h @ stack("down_proj", e).T) * weight[row, slot, None])
    return out


def _exact_attention(qkv: torch.Tensor, i: dict[str, torch.Tensor], layer: int) -> torch.Tensor:
    """Rotates q and k, stores the new k and v rows in the (float64) pool and attends."""
    rows = qkv.shape[0]
    cos, sin = (t.double() for t in _rope_tables(torch.float32))
    q, k, v = qkv.double().view(rows, 3, HEADS, HEAD_DIM).unbind(1)
    half = HEAD_DIM // 2
    out = torch.empty_like(q)
    for r, last in enumerate(i["last"].tolist()):
        c, s = cos[last], sin[last]

        def turn(t: torch.Tensor) -> torch.Tensor:
            return t * c + torch.cat([-t[:, half:], t[:, :half]], dim=1) * s

        pages = i["table"][r].long()
        pool = i["pool"]
        pool[pages[last // PAGE], 0, layer, last % PAGE] = turn(k[r])
        pool[pages[last // PAGE], 1, layer, last % PAGE] = v[r]
        keys, values = (pool[pages, j, layer].flatten(0, 1)[: last + 1] for j in (0, 1))
        score = (keys * turn(q[r])).sum(dim=2) * HEAD_DIM ** -0.5
        out[r] = (torch.softmax(score, dim=0).unsqueeze(2) * values).sum(dim=0)
    return out


def _exact_norm(x: torch.Tensor, gamma: torch.Tensor) -> torch.Tensor:
    return x / torch.sqrt(x.square().mean(dim=1, keepdim=True) + EPS) * gamma.double()


def _exact_decoder(case: dict, seed: int) -> torch.Tensor:
    w, hidden, pool = _decoder_inputs(case, seed)
    pool["pool"] = pool["pool"].double()
    x = hidden.double()
    for layer in range(LAYERS):
        p = f"layers.{layer}."
        normed = _exact_norm(x, w[p + "input_layernorm.weight"])
        qkv = torch.cat([normed @ _plain(w[f"{p}self_attn.{c}_proj.weight"]).T for c in "qkv"], dim=1)
        attended = _exact_attention(qkv, pool, layer).flatten(1)
        x = x + attended @ _plain(w[p + "self_attn.o_proj.weight"]).T
        normed = _exact_norm(x, w[p + "post_attention_layernorm.weight"])
        if layer == 0:
            gate, up, down = (_plain(w[f"{p}mlp.{c}_proj.weight"]) for c in ("gate", "up", "down"))
            x = x + _silu_mul(normed @ gate.T, normed @ up.T) @ down.T
        else:
            x = x + _exact_moe({k[len(p) + 4:]: v for k, v in w.items() if k.startswith(p + "mlp.")}, normed)
    return _exact_norm(x, w["norm.weight"]) @ _plain(w["lm_head.weight"]).T


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_moe(*_moe_inputs(case, seed))
    if kind == "dense":
        w, x = _dense_inputs(case, seed)
        return x.double() @ _plain(w).T
    if kind == "attention":
        i = _attention_inputs(case, seed)
        i["pool"] = i["pool"].double()
        return _exact_attention(i["qkv"], i, 1), i["pool"]
    return _exact_decoder(case, seed)
