"""The prefill layer's one GEMM launch (gate/up tiles, then down tiles that wait for their rows), and a phase alone.

Weights at an odd address take the fragment-load kernel, a launch per phase and the same bits, so the two
paths are compared bit for bit: at the edges of the tiles (32-row blocks, 64- and 128-row tiles), with one
expert or more tiles than workgroups, and as the launch meets itself: replayed, and on two streams at once.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _gpu import DEV, bits_equal, layer_weights, moe_for, n, t

pytestmark = pytest.mark.gpu

SHAPES = {  # experts, hidden, ffn (top 2, 2 shared experts)
    "small": (8, 256, 128),
    "many": (64, 256, 256),
    "one": (1, 128, 128),
    "fine gate/up": (8, 1152, 256),  # at int8 group 64: 18 groups a row, down 4
    "fine down": (8, 256, 1152),
    "wide": (8, 2176, 256),
}


def _pair(oracle, shape: str, int8: bool, group: int = 128):
    """A layer with aligned weights, and the same one with its gate stack at an odd (2-byte for bf16) address."""
    from uocr_moe import MoE

    E, H, F = SHAPES[shape]
    layer = oracle.make_layer(5, E=E, H=H, F=F, topk=min(2, E), int8=int8, group=group, std=0.05, router_std=0.1)
    moe = moe_for(layer)
    w = layer_weights(layer)
    gate = w["experts.gate_proj"]
    raw = torch.empty(gate.numel() * gate.element_size() + 16, dtype=torch.uint8, device=DEV)
    off = gate.element_size()
    odd = raw[off:off + gate.numel() * gate.element_size()].view(gate.dtype).view(gate.shape)
    odd.copy_(gate)
    w["experts.gate_proj"] = odd
    other = MoE(moe.config, w)
    assert other.stacks["gate_proj"].data_ptr() % 16 != 0
    return moe, other


def _x(T: int, H: int) -> torch.Tensor:
    return t(np.random.default_rng(T).standard_normal((T, H)).astype(np.float32))


@pytest.mark.parametrize("int8", [True, False])
@pytest.mark.parametrize(("shape", "T"), [("one", 1), ("one", 64), ("one", 129), ("one", 300), ("small", 1),
                                          ("small", 31), ("small", 130), ("small", 515), ("many", 65),
                                          ("many", 2049), ("many", 6000)])
def test_one_launch_is_the_two(oracle, shape, T, int8) -> None:
    moe, other = _pair(oracle, shape, int8)
    x = _x(T, SHAPES[shape][1])
    assert bits_equal(n(moe(x)), n(other(x)))


def test_many_down_tiles(oracle) -> None:
    """Few gate/up tiles and more down tiles than the by-class plan holds."""
    from uocr_moe import MoE, MoeConfig

    E, H, F, T = 64, 4608, 128, 2048
    g = torch.Generator(device=DEV).manual_seed(1)

    def w(*shape: int) -> torch.Tensor:
        return (torch.randn(shape, generator=g, device=DEV) * 0.05).to(torch.bfloat16)

    weights = {"gate.gate_score.weight": w(E, H).float(), "experts.gate_proj": w(E, F, H),
               "experts.up_proj": w(E, F, H), "experts.down_proj": w(E, H, F),
               "shared_experts.gate_proj.weight": w(H // 16, 2 * F, 16),
               "shared_experts.up_proj.weight": w(H // 16, 2 * F, 16),
               "shared_experts.down_proj.weight": w(2 * F // 16, H, 16)}
    config = MoeConfig(hidden_size=H, moe_intermediate_size=F, n_routed_experts=E, num_experts_per_tok=1,
                       n_shared_experts=2, int8_experts=False)
    x = _x(T, H)
    got = n(MoE(config, weights)(x))
    raw = torch.empty(E * F * H + 8, dtype=torch.bfloat16, device=DEV)
    odd = raw[1:1 + E * F * H].view(E, F, H)
    odd.copy_(weights["experts.gate_proj"])
    assert bits_equal(got, n(MoE(config, {**weights, "experts.gate_proj": odd})(x)))


def test_replays_and_streams(oracle) -> None:
    """A captured layer replayed between eager calls, then calls on two streams at once."""
    moe, _ = _pair(oracle, "many", True)
    xs = [_x(T, 256) for T in (700, 1900)]
    want = [n(moe(x)) for x in xs]
    side = torch.cuda.Stream()
    ws = moe.workspace(700, True)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        moe(xs[0], workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = moe(xs[0], workspace=ws)
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert bits_equal(n(moe(xs[1])), want[1])
        assert bits_equal(n(out), want[0])
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got: list[list[torch.Tensor]] = [[], []]
    torch.cuda.synchronize()
    for _ in range(8):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(moe(xs[i]))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(bits_equal(n(o), want[i]) for o in got[i])


def test_routing_launches_agree(oracle) -> None:
    """The served router's two sets of routing launches (one token apart) route the same tokens alike."""
    layer = oracle.make_layer(7, E=64, H=1280, F=128, topk=6, int8=True)
    moe = moe_for(layer)
    x = _x(1400, 1280)
    out, ids, wts = (n(v) for v in moe(x, routing=True))
    few, ids_few, wts_few = (n(v) for v in moe(x[:1399].contiguous(), routing=True))
    assert np.array_equal(ids[:1399], ids_few) and bits_equal(wts[:1399], wts_few)
    assert bits_equal(out[:1399], few)


@pytest.mark.parametrize("T", [40, 6000])
def test_a_wait_without_an_end_is_nan(oracle, monkeypatch, T) -> None:
    """The down tiles' wait, forced to give up from the host (a limit of 0 polls; every workgroup still exits):
    the call writes NaN everywhere, and the next one on the same workspace is right again."""
    moe, other = _pair(oracle, "many", True)
    x = _x(T, 256)
    ws = moe.workspace(T, True)
    monkeypatch.setenv("UOCR_MOE_SPIN_LIMIT", "0")
    out, _, wts = moe(x, workspace=ws, routing=True)
    assert np.isnan(n(out)).all() and np.isnan(n(wts)).all()
    monkeypatch.delenv("UOCR_MOE_SPIN_LIMIT")
    assert bits_equal(n(moe(x, workspace=ws)), n(other(x)))


@pytest.mark.parametrize("T", [1, 33, 130, 700, 2100, 9000])
@pytest.mark.parametrize(("shape", "staged"), [("fine gate/up", "gemm_down"), ("fine down", "gemm_gateup")])
def test_one_phase_staged(oracle, shape, staged, T) -> None:
    """More than 16 int8 groups a row in one phase: only that phase leaves the LDS-staged kernel."""
    from uocr_moe import _lib

    moe, other = _pair(oracle, shape, True, group=64)
    x = _x(T, SHAPES[shape][1])
    _lib.timing_begin(16)
    got = n(moe(x))
    names = [name for name, _ in _lib.timing_end(16)]
    assert staged in names and sum(name.startswith("gemm_") for name in names) == 2
    assert bits_equal(got, n(other(x)))


@pytest.mark.parametrize("T", [2048, 2111, 5000])
def test_wide_layers_take_two_launches(oracle, T) -> None:
    """Beyond hidden 2048 each phase has a launch of its own (from 2048 tokens on, the router's limit there)."""
    from uocr_moe import _lib

    moe, other = _pair(oracle, "wide", False)
    x = _x(T, SHAPES["wide"][1])
    _lib.timing_begin(16)
    got = n(moe(x))
    names = [name for name, _ in _lib.timing_end(16)]
    assert [name for name in names if name.startswith("gemm_")] == ["gemm_gateup", "gemm_down"]
    assert bits_equal(got, n(other(x)))
