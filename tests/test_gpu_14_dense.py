"""GPU tier: the dense products of batches above the decode sizes (dense.hip `qmm_dense_kernel`: the shared
expert over 64-token x 64-row tiles; prefill.hip `router_logits_kernel`) and the two-chain hybrid
regime around them, against the oracle.

The shapes sit where the kernel's tiling can go wrong: hidden and shared sizes for each number of
wavefronts that cut K (1, 2, 4 and 8, with stages that do not divide evenly), weight-row blocks that
do not fill a workgroup, router rows past the experts, the last token block with 1, 63 and 64 rows,
more tokens than weight rows (the other tile order), and hidden sizes off the large kernel's 256
(no hybrid regime). Shared weights are scaled up so that they carry most of the output. Bars: the
BASELINE gates (tests/_util.assert_close).
"""

from __future__ import annotations

import pytest
import torch

from oracle import moe as om
from quanta_amd import _lib as L
from quanta_amd import ops, synth
from quanta_amd.moe import prepare, qwen35_moe
from quanta_amd.quant import quantize_affine
from tests._util import assert_close, f64, oracle_params_from_torch

pytestmark = pytest.mark.gpu

SHARED = ("shared_gate_proj", "shared_up_proj", "shared_down_proj")


@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("N,H,Is,E", [(257, 256, 128, 8), (319, 384, 640, 16), (320, 512, 1152, 40),
                                      (450, 1024, 256, 64), (321, 2176, 512, 96), (700, 256, 384, 255)])
def test_dense_products_vs_oracle(gpu, N, H, Is, E, bits):
    s = synth.scaled_spec("c1", hidden_size=H, num_experts=E, num_experts_per_tok=2,
                          moe_intermediate_size=128, shared_expert_intermediate_size=Is)
    p = synth.make_layer(s, device=gpu, seed=N)
    for key in SHARED:
        w = (p[key].float() * 8.0).to(torch.bfloat16)
        if bits == 8:
            pk, sc, bi = quantize_affine(w, 8, group_size=64)
            w = {"packed": pk, "scale": sc, "bias": bi, "group_size": 64, "bits": 8}
        p[key] = w
    x = synth.make_inputs(s, N, device=gpu, seed=3 + N)
    y = qwen35_moe(x[None], p, s.cfg)[0]
    _, it = om.moe_forward(f64(x), oracle_params_from_torch(p), k=2, inter=128)
    assert_close(f64(y), it["y_exact"], f"dense N={N} H={H} Is={Is} E={E} int{bits}")


@pytest.mark.parametrize("N,H,E", [(257, 256, 16), (300, 640, 40), (513, 512, 255), (700, 2048, 256), (1000, 768, 64),
                                   (1023, 4096, 512), (1537, 4096, 512)])
def test_router_logits_keep_their_order(gpu, N, H, E):
    """Router logits above the decode sizes are one fp32 sum over all of K in k order, bit for bit the large
    kernel's (hidden sizes off 256: the decode kernel's), so that a prompt's expert ids do not depend on
    the kernel its size takes. 32- and 64-token tiles, last tiles partly filled, fewer superblocks than the
    ring holds, rows with and without the shared gate's past the last block of 16. (The workspace starts with
    the logits.)"""
    s = synth.scaled_spec("c1", hidden_size=H, num_experts=E, num_experts_per_tok=2,
                          moe_intermediate_size=128, shared_expert_intermediate_size=128)
    p = synth.make_layer(s, device=gpu, seed=N)
    pr = prepare(p, s.cfg, topk=2)
    rows = pr.cfg.router_rows
    x = synth.make_inputs(s, N, device=gpu, seed=N)
    ws = torch.zeros(ops.forward_workspace(pr.cfg, N), dtype=torch.uint8, device=gpu)
    ops.forward(pr.cfg, pr.weights, x, ws=ws)
    got = ws[: N * rows * 4].view(torch.float32).view(N, rows)[:, : E + 1]
    want = ops.grouped_qmm(x, K=H, n_rows=rows, weight_format=L.FMT_BF16, codes=pr.router_tiled, sb=None,
                           out_rows=N, epilogue=L.EPI_F32, dense_rows=N,
                           regime=L.REGIME_LARGE if H % 256 == 0 else L.REGIME_SMALL)[:, : E + 1]
    assert torch.equal(got, want)


@pytest.mark.parametrize("E,N", [(64, 300), (32, 400), (8, 300)])
def test_two_chains_repeat_bit_for_bit(gpu, E, N):
    """The hot and cold experts' chains run on two streams over disjoint rows: calls on one stream after
    another, each waited for, give the same bits (mean rows per expert 9, 25 and 75: the cold chain, then the hot
    one on the caller's stream)."""
    s = synth.scaled_spec("c1", hidden_size=512, num_experts=E, num_experts_per_tok=2,
                          moe_intermediate_size=256, shared_expert_intermediate_size=256)
    p = synth.make_layer(s, device=gpu, seed=E)
    x = synth.make_inputs(s, N, device=gpu, seed=N)[None]
    want = qwen35_moe(x, p, s.cfg)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for i in range(6):
        if i % 2:
            with torch.cuda.stream(side):
                y = qwen35_moe(x, p, s.cfg)
            side.synchronize()
        else:
            y = qwen35_moe(x, p, s.cfg)
            torch.cuda.synchronize()
        assert torch.equal(y, want), i


@pytest.mark.parametrize("H,I,E,k,N", [(512, 256, 64, 2, 300), (512, 256, 8, 2, 300), (2048, 512, 256, 8, 391),
                                       (2048, 512, 256, 8, 600), (4096, 1024, 256, 4, 600)])
def test_two_chains_of_concurrent_callers(gpu, H, I, E, k, N):
    """Two callers' streams, other inputs on each and no wait between their calls, share the auxiliary stream and
    its events: every output is the serial call's, bit for bit, and that is the decode kernels' within the gates
    (hot chain on the auxiliary stream, on the caller's, and, from 1e9 weights, in phases)."""
    s = synth.scaled_spec("c1", hidden_size=H, num_experts=E, num_experts_per_tok=k,
                          moe_intermediate_size=I, shared_expert_intermediate_size=256)
    p = synth.make_layer(s, device=gpu, seed=E)
    xs = [synth.make_inputs(s, N, device=gpu, seed=N + i)[None] for i in range(2)]
    want = [qwen35_moe(x, p, s.cfg) for x in xs]
    small = [qwen35_moe(x, p, s.cfg, regime=L.REGIME_SMALL) for x in xs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = []
    for i in range(8):
        with torch.cuda.stream(streams[i % 2]):
            outs.append(qwen35_moe(xs[i % 2], p, s.cfg))
    torch.cuda.synchronize()
    for i, y in enumerate(outs):
        assert torch.equal(y, want[i % 2]), f"call {i}"
    for w, r in zip(want, small):
        assert_close(f64(w[0]), f64(r[0]), f"two chains H={H} E={E} N={N} vs decode kernels", want_rounded=True)
