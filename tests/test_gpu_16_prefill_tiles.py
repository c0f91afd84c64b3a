"""GPU tier: the prefill kernel (prefill.hip `prefill_kernel`) at the ends of its tiles and rings: m-tiles of
1, 16, 17, 32, 33, 64, 65, 96, 97, 127 and 128 rows (1 to 4 m-blocks, rings of two and three slots, the
last wavefront's activations loaded or not) and an expert of two tiles; K of one superblock, of as many
as the ring holds and more; 512-row weight blocks and the 256-row form; int4, int3 and int6; the three
epilogues.

Bar: relative L2 error 2e-3 of the float64 product with the exact weights s q + b, over fp32 outputs
(weights rounded to fp16, 2^-11 relative to each, 3e-4 over a row's sum) and 5e-3 over bf16 ones.
"""

from __future__ import annotations

import pytest
import torch

from quanta_amd import _lib as L
from quanta_amd import ops
from quanta_amd.moe import tile_experts_packed
from quanta_amd.quant import quantize_affine, unpack_affine

pytestmark = pytest.mark.gpu

ROWS = (1, 16, 17, 32, 33, 64, 65, 96, 97, 127, 128, 129)
FMT = {4: L.FMT_INT4_G64, 3: L.FMT_INT3_G64, 6: L.FMT_INT6_G64}


@pytest.mark.parametrize("bits", [4, 3, 6])
@pytest.mark.parametrize("K,n_rows", [(128, 512), (256, 512), (384, 256), (640, 768), (1152, 1024)])
def test_prefill_tiles(gpu, K, n_rows, bits):
    g = torch.Generator(device="cpu").manual_seed(K + bits)
    E = len(ROWS)
    w = (torch.randn(E, n_rows, K, generator=g) * 0.05).to(gpu)
    pk, sc, bi = quantize_affine(w, bits, 64)
    te = tile_experts_packed({"packed": pk, "scale": sc, "bias": bi, "group_size": 64, "bits": bits})
    q = unpack_affine(pk, K, bits).double().reshape(E, n_rows, K // 64, 64)
    w64 = (sc.double()[..., None] * q + bi.double()[..., None]).reshape(E, n_rows, K)
    idx = torch.cat([torch.full((r,), e) for e, r in enumerate(ROWS)])
    idx = idx[torch.randperm(len(idx), generator=g)].to(torch.int32)[:, None].contiguous().to(gpu)
    n = len(idx)
    x = torch.randn(n, K, generator=g).to(torch.bfloat16).to(gpu)
    _, off, toff, srt, _, tmap = ops.permute(idx, E, L.LARGE_M_TILE)
    want = torch.empty(n, n_rows, dtype=torch.float64, device=gpu)
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        want[a:b] = x[srt[a:b].long()].double() @ w64[e].T
    kw = dict(K=K, n_rows=n_rows, weight_format=FMT[bits], codes=te["codes"], sb=te["sb"], out_rows=n,
              regime=L.REGIME_LARGE, slot_of=srt, slot_div=1, n_slots=n, offsets=off, tile_off=toff,
              tile_map=tmap, n_experts=E, row_exp=te["rexp"])
    rel = lambda got, ref: float((got.double() - ref).norm() / ref.norm())
    f32 = rel(ops.grouped_qmm(x, epilogue=L.EPI_F32, **kw), want)
    b16 = rel(ops.grouped_qmm(x, epilogue=L.EPI_BF16, **kw), want)
    gate, up = want[:, : n_rows // 2].to(torch.bfloat16).double(), want[:, n_rows // 2:].to(torch.bfloat16).double()
    glu = rel(ops.grouped_qmm(x, epilogue=L.EPI_SWIGLU, **kw), torch.nn.functional.silu(gate) * up)
    print(f"[parity] prefill int{bits} K={K} rows={n_rows}: f32 {f32:.1e} bf16 {b16:.1e} swiglu {glu:.1e}", flush=True)
    assert f32 <= 2e-3 and b16 <= 5e-3 and glu <= 5e-3
