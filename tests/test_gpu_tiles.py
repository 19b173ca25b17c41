"""The tile choices of the prefill GEMMs: every tile of the dense and the
expert kernels at sizes that leave remainders in rows, columns and K steps,
on both sides of the lines between tiles."""
import pytest
import torch

import test_gpu_projections as projections
from helpers import rel_l2
from litemoe_amd import experts, linear
from oracle import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows,n,k", [
    (1, 64, 64), (16, 4099, 192), (3, 1000, 1536),                     # 16 x 64, 1 to 24 K steps
    (17, 4099, 64), (129, 1000, 128), (256, 4096, 192),                # 64 x 64 (256 tiles)
    (257, 4096, 64), (300, 8190, 256),                                 # 128 x 64, then 64 x 128
    (511, 8192, 64), (512, 8192, 192),                                 # 64 x 128 (512 tiles)
    (513, 8200, 128), (1000, 8190, 64),                                # 128 x 128
    (1600, 5632, 128), (1537, 7000, 64),                               # 192 x 128
    (3000, 5700, 192), (2100, 16001, 64)])                             # 256 x 256
@torch.inference_mode()
def test_linear_dense_tiles_match_fp32_product(rows, n, k):
    """Within one bf16 ulp of the fp32 product (1e-3 where a sum cancels), as
    for the shapes of the model; no row or column past the output written."""
    g = torch.Generator(device=DEV).manual_seed(rows + n + k)
    a = torch.randn(rows, k, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    out = torch.full((rows + 1, n), float("nan"), device=DEV, dtype=torch.bfloat16)
    got = linear.linear_dense(a, w, out=out[:rows])
    assert projections.within_ulp_or_abs(got, (a.float() @ w.float().T).to(torch.bfloat16), 1, 1e-3)
    assert out[rows].isnan().all()
    assert torch.equal(linear.linear_dense(a[:1], w), got[:1])  # the tile changes no bits


@pytest.mark.parametrize("rows,hq,hkv,k,batch,cap", [
    (384, 24, 8, 128, 2, 256), (385, 24, 8, 128, 2, 256),    # 64 x 64 up to 384 rows, then 128 x 64
    (1500, 24, 8, 192, 3, 512),                              # 64 x 128
    (2500, 24, 8, 64, 5, 512), (4001, 24, 8, 64, 8, 512)])   # 128 x 128, 192 x 128
@torch.inference_mode()
def test_linear_rope_kv_tiles(rows, hq, hkv, k, batch, cap):
    projections.test_linear_rope_kv_equals_projection_then_rope_kv_write(rows, hq, hkv, k, batch, cap, cap, True)


@pytest.mark.parametrize("m,h,i,e,k", [
    (599, 128, 128, 50, 8), (600, 128, 128, 50, 8),          # 95.8 and 96 routes per expert
    (1300, 256, 128, 96, 8),                                 # more than 64 experts
    (2000, 384, 128, 16, 4), (4200, 384, 256, 16, 4),        # hidden not a multiple of 256
    (1023, 256, 128, 8, 8), (1024, 256, 128, 8, 8), (2048, 256, 128, 8, 8)])
@torch.inference_mode()
def test_expert_gemm_tiles_match_oracle(m, h, i, e, k):
    """lm_moe_routes on the grouped GEMMs against the oracle's per-route math
    (bf16 intermediates: 1e-2), with unequal experts and some without routes;
    fragment-order weights give the same bits."""
    g = torch.Generator().manual_seed(m + h + e)
    x = torch.randn(m, h, generator=g).to(torch.bfloat16)
    w1 = (torch.randn(e, 2 * i, h, generator=g) * 0.05).to(torch.bfloat16)
    w2 = (torch.randn(e, h, i, generator=g) * 0.05).to(torch.bfloat16)
    p = torch.rand(e, generator=g) + 0.02
    if e > k + 2:
        p[1:3] = 0.0
    ids = torch.stack([torch.multinomial(p, k, generator=g) for _ in range(m)]).int()
    d = [t.to(DEV) for t in (x, w1, w2, ids)]
    y = experts.moe_routes(*d)
    exp = ops.expert_routes(x, ids, w1, w2)
    assert rel_l2(y.cpu(), exp) < 1e-2
    per_row = (y.cpu().float() - exp.float()).norm(dim=1) / exp.float().norm(dim=1).clamp_min(1e-6)
    assert float(per_row.max()) < 5e-2
    assert torch.equal(experts.moe_routes(d[0], *experts.pack_expert_weights(d[1], d[2]), d[3], packed=True), y)
