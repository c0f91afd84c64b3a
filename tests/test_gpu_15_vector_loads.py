"""GPU tier: the 16-byte-piece kernels of the reference-dtype block (general.hip) and of the fp32 router
(router.hip), at the sizes where their pieces end: rows that are not whole pieces (element-strided
lanes) or not whole wavefront rounds, one piece, more than one round, every code width across word
boundaries, and bases off 16 bytes (the router's take its element-wise form).

Bars: float32 results within 1e-5 of float64 (scaled by max(1, max|y|); K <= 1096 fp32 sums of
O(1) terms stay below 2e-6), as tests/test_gpu_12_general.py; an unaligned copy of the same data
gives the same bits (same order of sums).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import quant as oq
from quanta_amd import ops
from quanta_amd.moe import MoEConfig, qwen35_moe

pytestmark = pytest.mark.gpu

E, K_TOP = 4, 2


def _ref(x, gate, gu, dn, I):
    logits = x @ gate.T
    p = np.exp(logits - logits.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    y = np.zeros_like(x)
    for t in range(len(x)):
        idx = np.argsort(-p[t], kind="stable")[:K_TOP]
        w = p[t, idx] / p[t, idx].sum()
        for e, we in zip(idx, w):
            g, u = gu[e, :I] @ x[t], gu[e, I:] @ x[t]
            y[t] += we * (dn[e] @ (g / (1 + np.exp(-g)) * u))
    return y


def _off(t: torch.Tensor) -> torch.Tensor:
    """The same contiguous values one element past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    v = buf[1:].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("H,I", [(8, 4), (36, 20), (40, 520), (513, 30), (1096, 24)])
def test_dense_float32_pieces(gpu, H, I):
    rng = np.random.default_rng(H)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    x, gate, gu, dn = f(5, H), f(E, H), f(E, 2 * I, H) / H ** 0.5, f(E, H, I) / I ** 0.5
    cfg = MoEConfig(H, E, K_TOP, I, 0)
    d = lambda v: torch.from_numpy(v).to(gpu)
    p = {"gate": d(gate), "experts_gate_up": d(gu), "experts_down": d(dn)}
    y = qwen35_moe(d(x)[None], p, cfg)[0]
    want = _ref(*(v.astype(np.float64) for v in (x, gate, gu, dn)), I)
    err = np.abs(y.double().cpu().numpy() - want).max() / max(1.0, np.abs(want).max())
    print(f"[parity] dense f32 H={H} I={I}: {err:.2e}", flush=True)
    assert err <= 1e-5
    q = {key: _off(v) for key, v in p.items()}
    assert torch.equal(qwen35_moe(_off(d(x)[None]), q, cfg)[0], y)


@pytest.mark.parametrize("H,I", [(40, 24), (1000, 504), (100, 60)])
def test_dense_bf16_off_alignment(gpu, H, I):
    """bf16 tensors two bytes off give the aligned ones' bits (whole pieces; element-strided lanes)."""
    g = torch.Generator(device="cpu").manual_seed(H)
    r = lambda *s: (torch.randn(*s, generator=g) / s[-1] ** 0.5).to(torch.bfloat16).to(gpu)
    p = {"gate": r(E, H), "experts_gate_up": r(E, 2 * I, H), "experts_down": r(E, H, I)}
    x = r(1, 5, H) * H ** 0.5
    cfg = MoEConfig(H, E, K_TOP, I, 0)
    y = qwen35_moe(x, p, cfg)
    d = lambda t: t.double().cpu().numpy()
    want = _ref(d(x)[0], *(d(p[k]) for k in ("gate", "experts_gate_up", "experts_down")), I)
    # gate, up, h and the down rows each round to bf16 (2^-9 relative), the output once more
    assert np.linalg.norm(d(y)[0] - want) <= 1e-2 * np.linalg.norm(want)
    q = {key: _off(v) for key, v in p.items()}
    assert torch.equal(qwen35_moe(_off(x), q, cfg), y)


@pytest.mark.parametrize("bits,gs,H,I", [(2, 32, 32, 32), (3, 32, 96, 544), (4, 64, 576, 64), (5, 32, 544, 32),
                                         (6, 128, 640, 128), (8, 32, 32, 64)])
def test_packed_float32_pieces(gpu, bits, gs, H, I):
    rng = np.random.default_rng(bits)
    f = lambda *s: rng.standard_normal(s).astype(np.float32)
    x, gate = f(3, H), f(E, H)
    gq = oq.quantize_rtn_f32(f(E, 2 * I, H) / H ** 0.5, bits, gs)
    dq = oq.quantize_rtn_f32(f(E, H, I) / I ** 0.5, bits, gs)
    deq = lambda q, k: np.asarray(oq.dequant_float(q[0], np.float64(q[1]), np.float64(q[2]), k, bits=bits,
                                                   group_size=gs), np.float64)
    d = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(gpu)
    trip = lambda q: {"packed": d(q[0].view(np.int32)), "scale": d(np.float32(q[1])), "bias": d(np.float32(q[2])),
                      "bits": bits, "group_size": gs}
    p = {"gate": d(gate), "experts_gate_up": trip(gq), "experts_down": trip(dq)}
    y = qwen35_moe(d(x)[None], p, MoEConfig(H, E, K_TOP, I, 0))[0]
    want = _ref(x.astype(np.float64), gate.astype(np.float64), deq(gq, H), deq(dq, I), I)
    err = np.abs(y.double().cpu().numpy() - want).max() / max(1.0, np.abs(want).max())
    print(f"[parity] packed f32 int{bits} g{gs} H={H} I={I}: {err:.2e}", flush=True)
    assert err <= 1e-5


@pytest.mark.parametrize("N,H,E_", [(1, 8, 3), (5, 512, 16), (9, 520, 17), (4, 30, 5), (130, 1024, 33)])
def test_router_f32_pieces(gpu, N, H, E_):
    g = torch.Generator(device="cpu").manual_seed(N)
    x = torch.randn(N, H, generator=g).to(torch.bfloat16).to(gpu)
    w, sg = (torch.randn(r, H, generator=g).to(gpu) / H ** 0.5 for r in (E_, 1))
    got = ops.router_logits_f32(x, w, sg.reshape(H))
    want = x.double() @ torch.cat([w, sg]).double().T
    assert (got.double() - want).abs().max() <= 1e-5
    # (the element-wise form sums in another order)
    off = ops.router_logits_f32(x, _off(w), _off(sg.reshape(H)))
    assert (off.double() - want).abs().max() <= 1e-5
