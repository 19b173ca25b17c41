"""The kernels that prefill calls choose by size: every tile of the dense and the
expert kernels at sizes that leave remainders in rows, columns and K steps,
on both sides of the lines between tiles, the persistent router and the
route permutation at their limits."""
import pytest
import torch

import test_gpu_projections as projections
from helpers import rel_l2
from litemoe_amd import _lib, experts, flash_decode, linear, norm, router
from oracle import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows,n,k", [
    (1, 64, 64), (16, 4099, 192), (3, 1000, 1536),                     # 16 x 64, 1 to 24 K steps
    (17, 4099, 64), (129, 1000, 128), (256, 4096, 192),                # 64 x 64 (256 tiles)
    (257, 4096, 64), (300, 8190, 256),                                 # 128 x 64
    (511, 8192, 64), (512, 8192, 192),                                 # 128 x 64 (512 tiles)
    (1500, 2563, 64), (1400, 2820, 192), (64, 17001, 128),             # 64 x 128
    (513, 8200, 128), (1000, 8190, 64),                                # 128 x 128
    (1600, 5632, 128), (1537, 7000, 64),                               # 192 x 128
    (3000, 5700, 192), (2100, 16001, 64),                              # 192 x 128, two rounds and more
    (3900, 4095, 192), (3841, 4092, 64), (3900, 4088, 128),            # 256 x 256: 2-, 8- and 16-byte stores
    (200, 49155, 64)])                                                 # one row tile of it
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


@pytest.mark.parametrize("m,h,e,k,add", [
    (1024, 1536, 40, 8, True), (1025, 1024, 32, 8, True), (1039, 512, 17, 2, True),
    (4096, 1024, 33, 4, False), (4096 + 16, 1536, 40, 8, True), (9000 + 15, 1536, 64, 8, True),
    (2055, 512, 64, 16, False)])
@torch.inference_mode()
def test_persistent_router_matches_per_token_kernel(m, h, e, k, add):
    """One block per workgroup and several, with and without a tail: x and z
    bitwise the norm kernel's, logits within a bf16 ulp of the per-token
    kernels' (their own in the tail), the selection exact given the logits."""
    g = torch.Generator(device=DEV).manual_seed(m + h)
    x = torch.randn(m, h, generator=g, device=DEV).to(torch.bfloat16)
    a = torch.randn(m, h, generator=g, device=DEV).to(torch.bfloat16) if add else None
    w = (1 + 0.2 * torch.randn(h, generator=g, device=DEV)).to(torch.bfloat16)
    wr = (0.02 * torch.randn(e, h, generator=g, device=DEV)).to(torch.bfloat16)
    x1, x2 = x.clone(), x.clone()
    got, ref = (torch.empty(m, e, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    weights, ids, z = router.add_rmsnorm_route(x1, a, 0.22, w, 1e-6, wr, k, logits_out=got)
    z2 = norm.add_rmsnorm(x2, a, 0.22, w, 1e-6)
    assert torch.equal(x1, x2) and torch.equal(z, z2)
    for i in range(0, m, 1000):
        router.route(z2[i:i + 1000], wr, k, logits_out=ref[i:i + 1000])
    assert projections.within_ulp_or_abs(got, ref, 1, 2e-3)
    tail = m - m % 16
    assert torch.equal(got[tail:], ref[tail:])
    ew, eids = ops.route(got.cpu(), k)
    assert torch.equal(ids.cpu(), eids)
    torch.testing.assert_close(weights.cpu(), ew, rtol=2e-6, atol=1e-7)


@pytest.mark.parametrize("routes", [1, 63, 64, 65, 1024, 1025, 8191, 8192, 8193])
@pytest.mark.parametrize("local,first", [(1, 0), (40, 0), (63, 3), (511, 0)])
@torch.inference_mode()
def test_moe_align_around_its_kernels_limits(routes, local, first):
    g = torch.Generator().manual_seed(routes + local)
    ids = torch.randint(0, local + 2 * first + 1, (routes, 1), generator=g, dtype=torch.int32)
    offsets, order, inverse = experts.moe_align(ids.to(DEV), local, first)
    eo, eord, einv = ops.permutation(ids, local, first)
    assert offsets.cpu().tolist() == eo.tolist()
    assert torch.equal(order.cpu().long(), eord) and torch.equal(inverse.cpu().long(), einv)


@pytest.mark.parametrize("splits", [2, 4, 5, 16, 17, 40])
@torch.inference_mode()
def test_flash_decode_combine_batches(splits):
    """Split counts around the combine's batches (4, 16, several), rows that
    fill one split, some and all: against the oracle (bf16 output and P, 1e-2),
    with NaN in the workspace of the splits that a short row leaves unwritten."""
    g = torch.Generator().manual_seed(splits)
    b, hq, hkv, cap = 4, 8, 4, 2048
    q = torch.randn(b, hq, 1, 64, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(b, hkv, cap, 64, generator=g).to(torch.bfloat16) for _ in range(2))
    used = torch.tensor([1, 200, 1025, cap], dtype=torch.int32)
    flash = flash_decode.FlashDecode(b, hkv, hq // hkv, cap, DEV, num_splits=splits)
    flash.workspace.fill_(0xFF)
    got = flash(q.to(DEV), k.to(DEV), v.to(DEV), None, None, 0.125, used.to(DEV))
    exp = ops.decode_attention(q[:, :, 0], k, v, used, 0.125)
    assert rel_l2(got[:, :, 0].cpu(), exp) < 1e-2 and torch.isfinite(got).all()


@pytest.mark.parametrize("m,h,i,e,k", [(264, 1536, 512, 40, 8), (265, 1536, 512, 40, 8), (511, 384, 128, 7, 5),
                                       (2113, 128, 128, 3, 1)])
@torch.inference_mode()
def test_expert_gemm_line_matches_oracle(m, h, i, e, k):
    """Both sides of the route count from which the grouped GEMMs run."""
    test_expert_gemm_tiles_match_oracle(m, h, i, e, k)


@pytest.mark.parametrize("batch,topk,hidden,rank,remap", [
    (3, 8, 8, 0, False), (5, 3, 1544, 0, True), (4, 8, 4104, 1, False), (700, 8, 1536, 0, False)])
@torch.inference_mode()
def test_finish_in_route_order(batch, topk, hidden, rank, remap):
    """lm_moe_finish without an order (rows in route order), bit-exact against
    the oracle: waves with one column in the row, routes of another rank (NaN
    rows) and a logical map."""
    g = torch.Generator().manual_seed(batch + hidden)
    count = 8
    ids = torch.stack([torch.randperm(2 * count, generator=g)[:topk] for _ in range(batch)]).int()
    y = torch.randn(batch * topk, hidden, generator=g).to(torch.bfloat16)
    y[(ids.flatten() < rank * count) | (ids.flatten() >= (rank + 1) * count)] = float("nan")
    scales = torch.softmax(torch.randn(batch, topk, generator=g), -1)
    logical = torch.randperm(2 * count, generator=g) if remap else None
    out = torch.full((batch + 1, hidden), 7.0, dtype=torch.bfloat16, device=DEV)
    d = [t.to(DEV) for t in (y, ids, scales)]
    lg = None if logical is None else logical.to(DEV)
    _lib.call("lm_moe_finish", d[0].data_ptr(), d[1].data_ptr(), None, d[2].data_ptr(), _lib.ptr(lg), out.data_ptr(),
              batch, hidden, topk, rank, count, None, 0, _lib.stream(out.device))
    assert torch.equal(out[:batch].cpu(), ops.finish(y, ids, scales, rank, count, logical))
    assert (out[batch] == 7).all()


@pytest.mark.parametrize("m,h,i,e,k,hot", [
    (1, 1024, 512, 32, 8, False), (5, 1536, 512, 40, 8, False), (8, 256, 128, 17, 8, True),
    (31, 512, 256, 64, 8, True), (32, 128, 1024, 65, 8, False), (33, 128, 128, 100, 8, True)])
@pytest.mark.parametrize("packed", [False, True])
@torch.inference_mode()
def test_few_routes_equal_block_path(m, h, i, e, k, hot, packed):
    """Calls below four routes per expert, to 256 routes (each wave finds its
    expert's routes) and past them: the bits of the aligned-block path, with
    experts of none, some and more than 16 and 32 routes."""
    g = torch.Generator().manual_seed(m + e)
    x = torch.randn(m, h, generator=g).to(torch.bfloat16).to(DEV)
    w1 = (torch.randn(e, 2 * i, h, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    w2 = (torch.randn(e, h, i, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(m)]).int()
    if hot:
        ids[:, 0] = e - 1  # also as a repeated id
    ids = ids.to(DEV)
    w = experts.pack_expert_weights(w1, w2) if packed else (w1, w2)
    assert torch.equal(experts.moe_routes(x, *w, ids, packed=packed), experts.moe_routes(x, w1, w2, ids, block_rows=16))


@torch.inference_mode()
def test_finish_in_route_order_takes_y_of_the_owned_rows_only():
    """Routes of other ranks have no row behind y: the first tokens hold the
    owned routes, and y ends with the last of them."""
    g = torch.Generator().manual_seed(3)
    batch, topk, hidden, count, rank = 40, 8, 1536, 8, 1
    ids = torch.stack([torch.randperm(count, generator=g)[:topk] for _ in range(batch)]).int()
    ids[:7, ::2] += rank * count
    owned = (ids.flatten() >= count).nonzero().flatten()
    y = torch.randn(batch * topk, hidden, generator=g).to(torch.bfloat16)
    scales = torch.softmax(torch.randn(batch, topk, generator=g), -1)
    d = [t.to(DEV) for t in (y[:int(owned[-1]) + 1], ids, scales)]
    out = torch.full((batch, hidden), 7.0, dtype=torch.bfloat16, device=DEV)
    _lib.call("lm_moe_finish", d[0].data_ptr(), d[1].data_ptr(), None, d[2].data_ptr(), None, out.data_ptr(), batch,
              hidden, topk, rank, count, None, 0, _lib.stream(out.device))
    assert torch.equal(out.cpu(), ops.finish(y, ids, scales, rank, count, None))


@pytest.mark.parametrize("m,h,i,e,k", [(3, 128, 128, 9, 3), (700, 1536, 128, 16, 8), (300, 2048, 128, 16, 8)])
@torch.inference_mode()
def test_fused_experts_combine_drops_ids_of_no_expert(m, h, i, e, k):
    """The combine that loads every row of the library's scratch: ids outside
    every expert add nothing, whatever their rows hold."""
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, h, generator=g).to(torch.bfloat16).to(DEV)
    w1 = (torch.randn(e, 2 * i, h, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    w2 = (torch.randn(e, h, i, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(m)]).int()
    ids[::3, 0] = e
    ids[1::3, -1] = -1
    scales = torch.softmax(torch.randn(m, k, generator=g), -1)
    backend = experts.HipFusedExperts()
    backend.workspace.get(x.device, 1 << 26).fill_(0xFF)  # NaN in every row that is not written
    out = backend.operation(x, w1, w2, scales.to(DEV), ids.to(DEV), global_num_experts=e)
    y = experts.moe_routes(x, w1, w2, ids.to(DEV)).cpu()
    assert torch.equal(out.cpu(), ops.finish(y, ids, scales, 0, e, None))


@pytest.mark.parametrize("m,h,e", [
    (300, 384, 32), (600, 384, 32), (1300, 256, 96), (900, 384, 7), (2049, 256, 8), (1200, 1536, 8), (4100, 384, 16)])
@torch.inference_mode()
def test_expert_stages_equal_fused_routes(m, h, e):
    """lm_moe_gate_up and lm_moe_down on aligned routes (act in route order, the
    route list behind the staged tile or its own) against lm_moe_routes (act in
    sorted order), bit for bit, ids of no expert among them."""
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, h, generator=g).to(torch.bfloat16).to(DEV)
    w1 = (torch.randn(e, 256, h, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    w2 = (torch.randn(e, h, 128, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    ids = torch.stack([torch.randperm(e + 1, generator=g)[:7] for _ in range(m)]).int().to(DEV)
    offsets, order, _ = experts.moe_align(ids, e)
    act = experts.gate_up(x, w1, offsets, order, 7)
    y = experts.down(act, w2, offsets, order)
    expected = torch.zeros_like(y)
    experts.moe_routes(x, w1, w2, ids, y=expected)
    assert torch.equal(y, expected)


@pytest.mark.parametrize("rows,n,k", [
    (513, 1536, 64), (563, 6300, 128), (734, 5271, 64),      # each XCD an eighth of the tiles, by column
    (4955, 2786, 64), (2904, 4523, 1024),                    # by row
    (1317, 1852, 64), (575, 6400, 64)])                      # whole row tiles, fewer row tiles than XCDs
@torch.inference_mode()
def test_linear_dense_tile_orders(rows, n, k):
    test_linear_dense_tiles_match_fp32_product(rows, n, k)


@torch.inference_mode()
def test_linear_rope_kv_tiles_dealt_by_eighths():
    projections.test_linear_rope_kv_equals_projection_then_rope_kv_write(6400, 24, 8, 64, 13, 512, 512, True)


@pytest.mark.parametrize("rows,n,k", [
    (17, 32769, 64), (64, 40003, 192), (33, 53248, 128),     # 64 x 256, three stages
    (64, 53249, 64), (40, 66001, 128),                       # 64 x 128 past them
    (65, 66000, 64), (128, 70001, 128)])                     # 128 x 128, any number of column tiles
@torch.inference_mode()
def test_linear_dense_one_row_tile(rows, n, k):
    test_linear_dense_tiles_match_fp32_product(rows, n, k)


@pytest.mark.parametrize("rows,n,k", [
    (65, 21761, 64), (100, 24001, 192), (128, 32768, 64), (128, 32769, 128),  # 341 to 512 tiles of 128 x 64, and past them
    (257, 6700, 64), (506, 4961, 192), (624, 4076, 64)])
@torch.inference_mode()
def test_linear_dense_narrow_tiles_of_wide_outputs(rows, n, k):
    test_linear_dense_tiles_match_fp32_product(rows, n, k)


@pytest.mark.parametrize("rows,n,k", [
    (193, 35001, 64), (256, 66000, 64),                      # 256 rows where 192 would pad to 384
    (300, 60001, 64), (520, 34000, 128)])                    # and 192 where 256 would pad by a third
@torch.inference_mode()
def test_linear_dense_tile_height_by_padding(rows, n, k):
    test_linear_dense_tiles_match_fp32_product(rows, n, k)


@pytest.mark.parametrize("m,h,i,e,k", [
    (1450, 256, 128, 8, 8), (3000, 256, 256, 16, 8),         # one round of 192 x 128 tiles, more than one
    (6400, 256, 128, 32, 8), (6200, 384, 128, 32, 8)])       # where 256 x 256 ones take one
@torch.inference_mode()
def test_expert_gate_tile_by_rounds(m, h, i, e, k):
    test_expert_gemm_tiles_match_oracle(m, h, i, e, k)
