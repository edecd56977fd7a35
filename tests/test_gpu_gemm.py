"""The expert GEMMs at the edges of their tiles: 16-position tiles and blocks
(64 and 128 positions), row tiles past I and H, ragged K, drawn items, and
activations outside fp16's own range.  Reference: the fp64 oracle."""
import numpy as np
import pytest
import torch

import phantom_moe
from oracle import oracle
from phantom_moe import synth
from tests.helpers import to_bf16_tensor

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def run(dev, cfg, xb, L, room=1):
    ex = phantom_moe.MoEWeights.from_q4_0(
        *(torch.from_numpy(a).to(dev) for a in (L.gate, L.up, L.down)), cfg.H, cfg.I, cfg.E,
        shared=None if L.shared is None else tuple(torch.from_numpy(a).to(dev) for a in L.shared))
    y, _, idx = phantom_moe.moe_forward(to_bf16_tensor(xb, dev), torch.from_numpy(L.router_w).to(dev), ex, cfg.k,
                                        cfg.score, return_routing=True)
    ry, ridx, _ = oracle.moe_forward(xb, L.router_w, L.gate, L.up, L.down, cfg.k, cfg.score_mode, None,
                                     shared=L.shared)
    np.testing.assert_array_equal(idx.cpu().numpy(), ridx)
    y = y.cpu().numpy().astype(np.float64)
    assert np.isfinite(y).all()
    # Exact products summed in fp32: every token's error stays within the
    # (H + I) / 32 group sums' and their 32 products' roundings of 2^-24 each,
    # taken as independent with room for the cancellation of the sums
    err = np.linalg.norm(y - ry, axis=1) / np.linalg.norm(ry, axis=1)
    assert err.max() <= room * 8 * np.sqrt((cfg.H + cfg.I) / 32 + 32) * 2.0 ** -24, (cfg.name, err.max())


# (T, H, I, E, k, shared): T * k >= 64 slots per expert, so the GEMMs run
CASES = [
    (64, 128, 32, 1, 1, False),     # one block of four tiles; one row tile pair, the rest past I
    (65, 160, 96, 1, 1, False),     # H: one whole quad and one group; I: half a quad and one group
    (81, 192, 160, 1, 1, False),    # six tiles; two groups past a whole quad
    (112, 224, 128, 1, 1, True),    # seven tiles; three groups past a whole quad
    (128, 96, 224, 1, 1, False),    # a whole gate/up block; K under a quad
    (129, 256, 64, 1, 1, False),    # a last block of one position
    (209, 384, 192, 2, 1, False),   # segments of any length
    (160, 640, 320, 2, 2, True),    # both experts and the shared one see every token
    (1100, 512, 1024, 16, 1, False),  # segments of one or two blocks in down, items dealt
]


@pytest.mark.parametrize("shape", CASES, ids=lambda s: "-".join(str(int(v)) for v in s))
def test_gemm_edges(dev, shape):
    T, H, I, E, k, shared = shape
    cfg = synth.MoEConfig("gemm", H, I, E, k, T, shared=shared)
    run(dev, cfg, synth.activations(T, H, seed=T), synth.host_layer(cfg))


# Launches of four rounds of items or more, whose items are drawn from the
# ranges' counters: gate/up (a ragged last row block of I; H under 1024, where
# the counters lie closer than a 128-byte line) and down (a ragged last row
# block of H, K of three groups), on segments of uneven length
@pytest.mark.parametrize("shape,rows,BM,per_cu", [((1100, 160, 8224, 16, 1, False), "I", 128, 2),
                                                  ((1100, 416, 8224, 7, 1, True), "I", 128, 2),
                                                  ((1100, 16416, 96, 16, 1, False), "H", 64, 3)],
                         ids=["gate_up", "gate_up_shared", "down"])
def test_drawn_items(dev, shape, rows, BM, per_cu):
    T, H, I, E, k, shared = shape
    cfg = synth.MoEConfig("drawn", H, I, E, k, T, shared=shared)
    L, xb = synth.host_layer(cfg), synth.activations(T, H, seed=T)
    idx = oracle.route(xb, L.router_w, k, cfg.score_mode)[0]
    blocks = sum(-(-int(n) // BM) for n in np.bincount(idx.reshape(-1), minlength=E)) + (-(-T // BM) if shared else 0)
    items = blocks * -(-(I if rows == "I" else H) // (64 if rows == "I" else 128))
    # the grid is at most what is resident (expert_gemm.hip: kG2PerCu, kDrawRounds)
    assert items >= 4 * per_cu * torch.cuda.get_device_properties(0).multi_processor_count, items
    run(dev, cfg, xb, L)


# Launches with few position blocks, whose item ranges are cut between row
# blocks unless they are 8 or 16: 1, 3, 6, 7, 9 and 15 blocks in gate/up (with
# the shared expert's); in down also 6 segments of two blocks, which stay whole;
# 17 row blocks of I and 10 of H, the last ones ragged
@pytest.mark.parametrize("shape", [(64, 1184, 1056, 1, 1, False), (192, 1184, 1056, 3, 1, False),
                                   (70, 1184, 1056, 5, 5, True), (64, 1184, 1056, 7, 7, False),
                                   (64, 1184, 1056, 8, 8, False), (64, 1184, 1056, 8, 8, True),
                                   (64, 416, 1056, 15, 15, False), (64, 416, 1056, 16, 16, False)],
                         ids=lambda s: "-".join(str(int(v)) for v in s))
def test_few_blocks(dev, shape):
    T, H, I, E, k, shared = shape
    cfg = synth.MoEConfig("few", H, I, E, k, T, shared=shared)
    run(dev, cfg, synth.activations(T, H, seed=T), synth.host_layer(cfg))


def test_one_block_uses_every_xcd(dev):
    """One position block runs on all eight XCDs: its layer takes well under the
    time of eight such blocks (one per XCD), which is what it took when a range
    held whole blocks only."""
    ms = []
    for E in (1, 8):
        cfg = synth.MoEConfig("spread", 4096, 8192, E, 1, 64 * E)
        dl = synth.device_layer(cfg, dev)
        ex = phantom_moe.MoEWeights.from_q4_0(dl.gate, dl.up, dl.down, cfg.H, cfg.I, cfg.E)
        x = to_bf16_tensor(synth.activations(cfg.T, cfg.H), dev)
        W = torch.zeros_like(dl.router_w)
        W[:, :E] = 1000 * torch.eye(E, device=dev)
        x[:, :E] = torch.eye(E, device=dev, dtype=x.dtype).repeat(64, 1)  # 64 tokens an expert

        def call():
            return phantom_moe.moe_forward(x, W, ex, 1, return_routing=True)

        assert torch.bincount(call()[2].flatten().long(), minlength=E).tolist() == [64] * E
        best = 1e9
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(4):
                call()
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        ms.append(best)
    assert ms[0] < 0.7 * ms[1], ms


# Both sides of the lines between the decode kernels and the GEMMs below 64
# slots per expert: token-tile shapes at 12, 14 and 16 slots per expert and at
# 512, 320 and 160 * 1024 positions x I (by the kernel that would run down),
# shapes whose rows of H are too long for those kernels at 225 * 1024
LINE = [
    ((96, 256, 2048, 16, 2, False), False),
    ((111, 256, 2048, 16, 2, False), False),
    ((96, 256, 2048, 16, 2, True), True),
    ((146, 320, 224, 32, 4, True), False),
    ((147, 320, 224, 32, 4, True), True),
    ((191, 2048, 768, 64, 4, False), False),
    ((192, 2048, 768, 64, 4, False), True),
    ((255, 1024, 480, 64, 4, False), False),
    ((310, 1024, 480, 64, 4, True), True),
    ((79, 384, 2048, 8, 2, False), False),
    ((80, 384, 2048, 8, 2, False), True),
    ((32, 5376, 512, 128, 4, True), False),
    ((112, 5376, 512, 128, 4, False), False),
    ((113, 5376, 512, 128, 4, False), True),
]


@pytest.mark.parametrize("shape,gemm", LINE, ids=lambda v: "-".join(map(str, map(int, v))) if isinstance(v, tuple) else "")
def test_regime_line(dev, shape, gemm):
    from phantom_moe import _lib

    T, H, I, E, k, shared = shape
    names = _lib.load().phantom_moe_expert_kernels(T, H, I, E, k, int(shared)).decode()
    assert ("gemm" in names) == gemm, names
    cfg = synth.MoEConfig("line", H, I, E, k, T, shared=shared)
    # the decode kernels' offset form loses about five times as much
    run(dev, cfg, synth.activations(T, H, seed=T), synth.host_layer(cfg), room=1 if gemm else 8)


@pytest.mark.parametrize("T", [64, 130])  # the one-pass and (E 16) the two-pass router's copy of x
def test_gemm_activation_range(dev, T):
    """Tokens with elements past fp16's range (65504) beside ones down to
    2^-34.  |h| must stay under 65504: with weights of at most 8 * 2^-17 and
    elements spread over 12 octaves below a largest one of at most 2^17.5,
    |g| and |u| stay under about 4 * 16 / 6 * 2^17.5 * 2^-14 = 2^7, and h
    under 2^14."""
    E = 16 if T >= 128 else 1
    k = 8 if T >= 128 else 1
    cfg = synth.MoEConfig("range", 256, 64, E, k, T)
    L = synth.host_layer(cfg)
    for a in (L.gate, L.up):
        a[..., 0:2] = np.full(a.shape[:-1] + (1,), 2.0 ** -17, dtype=np.float16).view(np.uint8)
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, cfg.H)) * np.exp2(rng.uniform(-12, 0, (T, cfg.H)))
    x *= np.exp2(rng.uniform(11, 17.5, (T, 1))) / np.abs(x).max(axis=1, keepdims=True)
    x[:, ::16] *= 2.0 ** -40
    run(dev, cfg, synth.f32_to_bf16_bits(x.astype(np.float32)), L)
