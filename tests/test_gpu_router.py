"""Router GEMM on the GPU (routing_logits = hidden_bf16 @ gate_weight.T, the linear
layer that produces the operator's routing_logits input, reference
moe/weight_origins_dataflow.md:21, :151-154), and the producer chain
hidden_bf16 -> (router logits, FP8 hidden states + scales) -> operator."""
import numpy as np
import pytest
import torch

import flashinfer_mlsys_amd as fm
from flashinfer_mlsys_amd import workloads as wl
from oracle import cpu_ref, np_ref

from conftest import assert_close_bf16, source_constant

pytestmark = pytest.mark.gpu

N_TERMS, U = 7168, 2.0 ** -24
GAMMA = N_TERMS * U / (1 - N_TERMS * U)  # fp32 summation error bound of a 7168-term dot product


@pytest.fixture(scope="module")
def gate(dev):
    g = wl.gate_weight_bf16()
    return g, g.to(dev)


# token counts on the three kernels (16-token tiles below 576 tokens, 32 x 64 tiles
# with the K steps split over the waves from 576 while they fit on the CUs, 2,048
# tokens on 256 CUs, 128 x 64 tiles beyond) with ragged last tiles and the sizes
# either side of each switch
@pytest.mark.parametrize("T", [1, 5, 16, 17, 64, 100, 575, 576, 1024, 2047, 2048, 2049, 3000, 4100])
def test_router_matches_float64(dev, gate, T):
    print(f"router T={T}", flush=True)
    x = wl.hidden_bf16(T, 900 + T)
    got = fm.router_logits(x.to(dev), gate[1]).cpu().numpy().astype(np.float64)
    ref, mag = np_ref.router_logits_f64(x, gate[0])
    err = np.abs(got - ref)
    assert (err <= GAMMA * mag).all(), f"max error / bound {float((err / (GAMMA * mag)).max()):.3g}"


def test_router_closed_forms(dev, gate):
    """One-hot tokens give exactly one scaled gate column; a gate of unit rows gives
    exactly the selected hidden columns (catches any index or layout mistake)."""
    ks = [0, 127, 128, 3000, 7167]
    x1 = torch.zeros((len(ks), 7168), dtype=torch.bfloat16)
    vals = torch.tensor([1.0, -2.5, 0.0078125, 3.0, -448.0], dtype=torch.bfloat16)
    for i, k in enumerate(ks):
        x1[i, k] = vals[i]
    got = fm.router_logits(x1.to(dev), gate[1]).cpu()
    exp = torch.stack([vals[i].float() * gate[0][:, k].float() for i, k in enumerate(ks)])
    assert torch.equal(got, exp)
    idx = (torch.arange(256) * 28 + 5) % 7168
    gu = torch.zeros((256, 7168), dtype=torch.bfloat16)
    gu[torch.arange(256), idx] = 1.0
    for T in (3, 40, 700, 3100):
        x = wl.hidden_bf16(T, 12)
        assert torch.equal(fm.router_logits(x.to(dev), gu.to(dev)).cpu(), x.float()[:, idx]), T


@pytest.mark.parametrize("T", [8, 2048])
def test_router_deterministic_and_in_place(dev, gate, T):
    x = wl.hidden_bf16(T, 77).to(dev)
    a = fm.router_logits(x, gate[1])
    out = torch.full((T, 256), 5.0, device=dev)
    b = fm.router_logits(x, gate[1], out=out)
    assert b is out and torch.equal(a, b)


def _fused(T, dev):
    """The rule of launch_router_quantize (csrc/moe_router.hip): one kernel, or two in turn."""
    cu = torch.cuda.get_device_properties(dev).multi_processor_count
    return (T < source_constant("moe_router.hip", "RT2_MIN_T") or (T + 31) // 32 * 4 <= cu
            or T >= source_constant("moe_router.hip", "RQ_MIN_TILED_T"))


@pytest.mark.parametrize("T", [1, 5, 16, 17, 64, 100, 575, 576, 1024, 2049, 2999, 3000])
def test_fused_producer_equals_separate_kernels(dev, gate, T):
    """router_logits_and_quantize writes the same logits, e4m3 rows and scales, bit
    for bit, as router_logits and quantize_activations (both kernels' tilings, ragged
    tiles); the rows and scales also equal the CPU oracle's quantiser."""
    assert _fused(T, dev) == (T not in (2049, 2999))  # the two counts at the ends of the other branch
    print(f"fused producer T={T}", flush=True)
    x = wl.hidden_bf16(T, 300 + T)
    xd = x.to(dev)
    lg, q, s = fm.router_logits_and_quantize(xd, gate[1])
    assert torch.equal(lg, fm.router_logits(xd, gate[1]))
    q2, s2 = fm.quantize_activations(xd)
    assert torch.equal(q.view(torch.uint8), q2.view(torch.uint8)) and torch.equal(s, s2)
    if T <= 100:
        qr, sr = cpu_ref.quantize_activations(x)
        assert torch.equal(q.cpu().view(torch.uint8), qr.view(torch.uint8)) and torch.equal(s.cpu(), sr)


@pytest.mark.parametrize("T", [577, 2047, 2048, 3000, 3073, 8191, 17001])
def test_quantiser_waves_equal_the_quantiser_kernel(dev, gate, T):
    """The quantiser waves of the two tiled router kernels (whole and ragged token
    tiles, one and several items per workgroup) against the router and quantiser kernels
    alone, bit for bit, on values that leave the quick path too: zeros of both signs,
    tiny blocks, infinities and NaNs."""
    assert _fused(T, dev)
    x = wl.hidden_bf16(T, 77).to(dev)
    x[0, :128] = 0
    x[1, 128:256] *= 1e-20
    x[T // 2, 5:9] = torch.tensor([-0.0, 3e38, -3e38, 1e-39], dtype=torch.bfloat16, device=dev)
    x[T - 1, 300] = float("inf")
    x[T - 1, 7000] = float("nan")
    lg, q, s = fm.router_logits_and_quantize(x, gate[1])
    q1, s1 = fm.quantize_activations(x)
    assert torch.equal(q.view(torch.uint8), q1.view(torch.uint8))
    assert torch.equal(s.view(torch.int32), s1.view(torch.int32))
    assert torch.equal(lg.view(torch.int32), fm.router_logits(x, gate[1]).view(torch.int32))


@pytest.mark.parametrize("T", [577, 2305, 2433, 3001, 3073])
def test_producer_writes_nothing_past_its_outputs(dev, gate, T):
    """Ragged last token tiles: the outputs are the front of larger buffers (the rows of a
    whole tile and more behind them), whose tails stay as they were. The hidden states are
    the front of a larger buffer too, of NaNs behind the T rows."""
    x = torch.full((T + 160, 7168), float("nan"), dtype=torch.bfloat16, device=dev)
    x[:T] = wl.hidden_bf16(T, 78).to(dev)
    sizes = {"logits": (T * 256 * 4, 160 * 256 * 4), "q": (T * 7168, 160 * 7168), "scale": (56 * T * 4, 56 * 160 * 4)}
    buf = {k: torch.full((n + tail,), 0x5A, dtype=torch.uint8, device=dev) for k, (n, tail) in sizes.items()}
    front = {k: buf[k][:sizes[k][0]] for k in buf}
    out = (front["logits"].view(torch.float32).view(T, 256), front["q"].view(torch.float8_e4m3fn).view(T, 7168),
           front["scale"].view(torch.float32).view(56, T))
    print(f"producer guards T={T}", flush=True)
    fm.router_logits_and_quantize(x[:T], gate[1], out=out)
    for k, b in buf.items():
        assert bool((b[sizes[k][0]:] == 0x5A).all()), k
    q, s = fm.quantize_activations(x[:T])
    assert torch.equal(out[1].view(torch.uint8), q.view(torch.uint8)) and torch.equal(out[2], s)
    assert torch.equal(out[0], fm.router_logits(x[:T], gate[1]))


@pytest.mark.parametrize("T,fused", [(37, True), (700, True), (2500, False), (3073, True)])
def test_producer_graph_replay(dev, gate, T, fused):
    """The producer step (the small kernel, either tiled kernel with quantiser waves, and
    the router and quantiser kernels in turn) captured in a HIP graph: each replay, with
    eager work in between, reproduces the eager result."""
    assert _fused(T, dev) == fused
    x = wl.hidden_bf16(T, 41).to(dev)
    bufs = (torch.empty((T, 256), device=dev), torch.empty((T, 7168), dtype=torch.float8_e4m3fn, device=dev),
            torch.empty((56, T), device=dev))
    fm.router_logits_and_quantize(x, gate[1], out=bufs)
    torch.cuda.synchronize()
    ref = [b.clone() for b in bufs]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fm.router_logits_and_quantize(x, gate[1], out=bufs)
    for i in range(3):
        for b in bufs:
            b.view(torch.uint8).fill_(0x55)
        fm.router_logits(wl.hidden_bf16(16, 6).to(dev), gate[1])  # eager work between replays
        g.replay()
        torch.cuda.synchronize()
        for b, r in zip(bufs, ref):
            assert torch.equal(b.view(torch.uint8), r.view(torch.uint8)), f"replay {i}"


# (T, local_expert_offset, seed): the first seed from 9000 + T whose oracle-chain
# selection margins are at least 256 fp32 ulps (the GPU logits differ from the CPU's
# fp32 matmul by summation order, far below that) and that routes a local pair.
CHAIN = [(4, 0, 9004), (48, 96, 9049), (300, 224, 9302)]


@pytest.mark.parametrize("T,offset,seed", CHAIN)
def test_producer_chain_matches_oracle(weights, dev, gate, T, offset, seed):
    """hidden_bf16 -> router_logits + quantize_activations -> kernel, against the oracle
    chain (cpu router, cpu quantiser, cpu operator)."""
    print(f"producer chain T={T} offset={offset} seed={seed}", flush=True)
    x = wl.hidden_bf16(T, seed)
    bias = wl.make_activations(T, seed, offset)[1]
    lg_ref = cpu_ref.router_logits(x, gate[0])
    g, e = cpu_ref.selection_margins(lg_ref, bias)
    assert min(g, e) >= 256, "the seed must keep the selection far from near-ties"
    hq_ref, hs_ref = cpu_ref.quantize_activations(x)
    ref = cpu_ref.run(lg_ref, bias, hq_ref, hs_ref, *weights[0], offset, 2.5).float().numpy()
    xd = x.to(dev)
    lg = fm.router_logits(xd, gate[1])
    hq, hs = fm.quantize_activations(xd)
    out = fm.run(lg, bias.to(dev), hq, hs, *weights[1], offset, 2.5).float().cpu().numpy()
    ids, _, _ = fm.route(lg, bias.to(dev), 2.5)
    ref_ids = cpu_ref.sorted_selection(cpu_ref.route(lg_ref, bias, 2.5)[0])
    assert torch.equal(ids.cpu().long(), ref_ids)
    assert_close_bf16(out, ref, f"chain T={T}")
