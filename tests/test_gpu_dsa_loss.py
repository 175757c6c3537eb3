"""DSA indexer KL loss: the HIP kernel against the float64 oracle, and the wrapper's contract
(reference: cppmega_mlx/nn/_tilelang/dsa_splitk_indexer_loss.py:1327-1570).

Tolerance: the kernel accumulates in float32 (dot products, exp, log); against the float64 oracle
on the same (already rounded) inputs the per-position loss agrees to 2e-5 absolute + 2e-4 relative.
"""

import numpy as np
import pytest
import torch

from cppmega_mlx_amd.nn._tilelang.dsa_splitk_indexer_loss import (
    dsa_splitk_indexer_loss_per_position,
    dsa_splitk_indexer_loss_tilelang,
    dsa_splitk_path_c_status,
    tilelang_supports,
)
from oracle import dsa_loss as od

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _case(seed, ASq, AB, AH, AD, Sk, topk, dtype):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn((ASq, AB, AH, AD), generator=g).to(dtype)
    k = torch.randn((Sk, AB, AH, AD), generator=g).to(dtype)
    idx = torch.randn((AB, ASq, Sk), generator=g) * 2.0
    top = torch.stack([torch.stack([torch.randperm(Sk, generator=g)[:topk] for _ in range(ASq)]) for _ in range(AB)])
    return q, k, idx, top


def _want(q, k, idx, top, scale, sparse):
    mask = od.sparse_index_mask(top.numpy(), k.shape[0]) if sparse else None
    return od.dsa_indexer_loss_per_position(idx.numpy(), q.float().numpy(), k.float().numpy(), softmax_scale=scale, index_mask=mask)


def test_cpu_side_checks_need_no_device():
    q = torch.zeros((4, 2, 3, 8)); k = torch.zeros((6, 2, 3, 8)); idx = torch.zeros((2, 4, 6)); top = torch.zeros((2, 4, 2), dtype=torch.int64)
    with pytest.raises(ValueError, match="query/key shape mismatch"):
        dsa_splitk_indexer_loss_tilelang(idx, top, q, k[:, :, :2], 1.0, 1.0, False)
    zero = dsa_splitk_indexer_loss_tilelang(idx[:, :0], top[:, :0], q[:0], k, 1.0, 1.0, True)
    assert zero.shape == () and zero.dtype == torch.float32 and float(zero) == 0.0
    assert float(dsa_splitk_indexer_loss_tilelang(idx[:, :, :0], top, q, k[:0], 1.0, 1.0, False)) == 0.0
    with pytest.raises(ValueError, match="AH > 128"):
        dsa_splitk_indexer_loss_tilelang(torch.zeros((1, 2, 2)), None, torch.zeros((2, 1, 129, 4)), torch.zeros((2, 1, 129, 4)), 1.0, 1.0, False)
    with pytest.raises(TypeError, match="dtypes must match"):
        dsa_splitk_indexer_loss_tilelang(idx, top, q, k.half(), 1.0, 1.0, False)
    with pytest.raises(TypeError, match="unsupported Q/K dtype"):
        dsa_splitk_indexer_loss_tilelang(idx, top, q.double(), k.double(), 1.0, 1.0, False)
    with pytest.raises(ValueError, match="unsupported device type"):
        dsa_splitk_indexer_loss_tilelang(idx, top, q, k, 1.0, 1.0, False)
    assert tilelang_supports(None) is False and tilelang_supports("cpu") is False
    assert isinstance(dsa_splitk_path_c_status().reason, str)


@pytest.mark.gpu
@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", [(5, 1, 2, 8, 5, 3), (33, 2, 4, 64, 33, 7), (17, 3, 3, 20, 40, 9), (40, 1, 8, 128, 24, 24), (300, 1, 2, 32, 300, 64)])
def test_per_position_loss_matches_the_oracle(shape, dt, sparse):
    ASq, AB, AH, AD, Sk, topk = shape
    q, k, idx, top = _case(11 + ASq, ASq, AB, AH, AD, Sk, topk, DTYPES[dt])
    scale = AD ** -0.5
    got = dsa_splitk_indexer_loss_per_position(idx.cuda(), top.cuda(), q.cuda(), k.cuda(), scale, sparse).cpu().numpy()
    want = _want(q, k, idx, top, scale, sparse)
    assert np.isfinite(got).all()
    np.testing.assert_allclose(got, want, atol=2e-5, rtol=2e-4)


@pytest.mark.gpu
def test_closed_forms_on_the_device():
    ASq, AB, AH, AD, Sk = 9, 2, 3, 16, 12
    z = lambda *s: torch.zeros(s, device="cuda")
    got = dsa_splitk_indexer_loss_per_position(z(AB, ASq, Sk), None, z(ASq, AB, AH, AD), z(Sk, AB, AH, AD), 0.5, False).cpu().numpy()
    want = np.log(Sk) - np.log(np.arange(1, ASq + 1))
    np.testing.assert_allclose(got, np.broadcast_to(want, (AB, ASq)), atol=1e-5)


@pytest.mark.gpu
def test_wrapper_contract_on_the_device():
    ASq, AB, AH, AD, Sk, topk = 24, 2, 4, 32, 24, 6
    q, k, idx, top = _case(5, ASq, AB, AH, AD, Sk, topk, torch.bfloat16)
    qd, kd, idxd, topd = q.cuda(), k.cuda(), idx.cuda(), top.cuda()
    for sparse in (False, True):
        got = dsa_splitk_indexer_loss_tilelang(idxd, topd, qd, kd, 0.2, 0.37, sparse)
        assert got.shape == () and got.dtype == torch.float32
        want = _want(q, k, idx, top, 0.2, sparse).mean() * 0.37
        assert abs(float(got) - want) < 2e-5 + 2e-4 * abs(want)
    # int32 lists, non-contiguous inputs and non-float32 index scores are taken as the reference takes them
    a = dsa_splitk_indexer_loss_tilelang(idxd, topd.int(), qd, kd, 0.2, 1.0, True)
    b = dsa_splitk_indexer_loss_tilelang(idxd.double(), topd, qd.transpose(0, 1).contiguous().transpose(0, 1), kd, 0.2, 1.0, True)
    c = dsa_splitk_indexer_loss_tilelang(idxd, topd, qd, kd, 0.2, 1.0, True)
    assert float(a) == float(c) == float(b)
    # duplicates in a list select the key once
    dup = topd.clone(); dup[..., 1] = dup[..., 0]
    want_dup = _want(q, k, idx, dup.cpu(), 0.2, True).mean()
    assert abs(float(dsa_splitk_indexer_loss_tilelang(idxd, dup, qd, kd, 0.2, 1.0, True)) - want_dup) < 1e-4
    with pytest.raises(ValueError, match="out of range"):
        bad = topd.clone(); bad[0, 0, 0] = Sk
        dsa_splitk_indexer_loss_tilelang(idxd, bad, qd, kd, 0.2, 1.0, True)
    with pytest.raises(ValueError, match="out of range"):
        bad = topd.clone(); bad[1, 3, 2] = -1
        dsa_splitk_indexer_loss_tilelang(idxd, bad, qd, kd, 0.2, 1.0, True)
    with pytest.raises(ValueError, match="TOPK"):
        dsa_splitk_indexer_loss_tilelang(idxd, topd[:, :, :0], qd, kd, 0.2, 1.0, True)
    with pytest.raises(ValueError, match="must have shape"):
        dsa_splitk_indexer_loss_tilelang(idxd, topd[:, :-1], qd, kd, 0.2, 1.0, True)
    with pytest.raises(TypeError, match="int32 or int64"):
        dsa_splitk_indexer_loss_tilelang(idxd, topd.float(), qd, kd, 0.2, 1.0, True)
    with pytest.raises(ValueError, match="device"):
        dsa_splitk_indexer_loss_tilelang(idxd, top, qd, kd, 0.2, 1.0, True)
    assert tilelang_supports("cuda") and dsa_splitk_path_c_status().available


@pytest.mark.gpu
def test_long_rows_use_the_large_lds_window():
    ASq, AB, AH, AD, Sk, topk = 6, 1, 2, 64, 9000, 512
    q, k, idx, top = _case(9, ASq, AB, AH, AD, Sk, topk, torch.bfloat16)
    # query positions near the end of a long context: rows see thousands of keys
    qpos = Sk - ASq
    qfull = torch.zeros((Sk, AB, AH, AD), dtype=torch.bfloat16); qfull[qpos:] = q
    idxfull = torch.zeros((AB, Sk, Sk)); idxfull[:, qpos:] = idx
    topfull = torch.zeros((AB, Sk, topk), dtype=torch.int64); topfull[:, qpos:] = top
    got = dsa_splitk_indexer_loss_per_position(idxfull.cuda(), topfull.cuda(), qfull.cuda(), k.cuda(), 0.125, True)[:, qpos:].cpu().numpy()
    mask = od.sparse_index_mask(top.numpy(), Sk)
    want = np.zeros((AB, ASq))
    for i in range(ASq):                       # query position qpos + i sees keys 0 .. qpos + i
        for b in range(AB):
            want[b, i] = od.row_loss(idx.double().numpy()[b, i], q.double().numpy()[i, b], k.double().numpy()[:, b], qpos + i + 1, 0.125, mask[b, i])
    np.testing.assert_allclose(got, want, atol=2e-5, rtol=2e-4)


@pytest.mark.gpu
def test_bench_size_properties():
    """At the size the bench times (4096 positions, 8 heads of 64): the closed form for zero rows and a uniform index,
    and non-negativity / finiteness of the divergence for random rows, dense and sparse."""
    ASq = Sk = 4096
    AB, AH, AD, topk = 1, 8, 64, 1024
    z = lambda *s: torch.zeros(s, device="cuda", dtype=torch.bfloat16)
    got = dsa_splitk_indexer_loss_per_position(torch.zeros((AB, ASq, Sk), device="cuda"), None, z(ASq, AB, AH, AD), z(Sk, AB, AH, AD),
                                               0.125, False).cpu().numpy()
    want = np.log(Sk) - np.log(np.arange(1, ASq + 1))
    np.testing.assert_allclose(got[0], want, atol=2e-5, rtol=2e-4)
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn((ASq, AB, AH, AD), generator=g, device="cuda").to(torch.bfloat16)
    k = torch.randn((Sk, AB, AH, AD), generator=g, device="cuda").to(torch.bfloat16)
    idx = torch.randn((AB, ASq, Sk), generator=g, device="cuda")
    top = torch.topk(idx, topk, dim=-1).indices
    for sparse in (False, True):
        loss = dsa_splitk_indexer_loss_per_position(idx, top, q, k, AD ** -0.5, sparse)
        assert torch.isfinite(loss).all() and (loss >= -1e-4).all()       # a divergence of p against a sub-normalised q
    # a few rows against the float64 oracle row function
    mask = None
    for sq in (0, 17, 2047, 4095):
        w = od.row_loss(idx[0, sq].double().cpu().numpy(), q[sq, 0].double().cpu().numpy(), k[:, 0].double().cpu().numpy(), sq + 1,
                        AD ** -0.5, mask)
        d = float(dsa_splitk_indexer_loss_per_position(idx, top, q, k, AD ** -0.5, False)[0, sq])
        assert abs(d - w) <= 2e-5 + 2e-4 * abs(w), (sq, d, w)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(130, 1, 3, 96, 203, 40), (200, 2, 5, 64, 97, 33), (64, 1, 1, 128, 64, 64), (65, 1, 2, 32, 129, 1), (1, 3, 2, 64, 1, 1),
                                   (130, 1, 2, 32, 345, 20)])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("sparse", [False, True])
def test_tile_edges(shape, dt, sparse):
    """Positions and keys that are not whole tiles of 64 x 128, more positions than keys and the other way round, rows of
    index scores that are not whole 16-byte loads."""
    ASq, AB, AH, AD, Sk, topk = shape
    q, k, idx, top = _case(ASq + Sk, ASq, AB, AH, AD, Sk, topk, DTYPES[dt])
    got = dsa_splitk_indexer_loss_per_position(idx.cuda(), top.cuda(), q.cuda(), k.cuda(), AD ** -0.5, sparse).cpu().numpy()
    np.testing.assert_allclose(got, _want(q, k, idx, top, AD ** -0.5, sparse), atol=2e-5, rtol=2e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(4096, 1, 64, 32, 4096, 0), (389, 2, 4, 64, 389, 50)])
def test_tiled_kernels_agree_with_the_kernel_without_a_workspace(shape):
    """Several slabs of positions (64 heads x 4096 positions), and an additive mask with masked rows."""
    import ctypes as C

    from cppmega_mlx_amd import _lib, ops
    ASq, AB, AH, AD, Sk, topk = shape
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k = (torch.randn((n, AB, AH, AD), generator=g, device="cuda").to(torch.bfloat16) for n in (ASq, Sk))
    idx = torch.randn((AB, ASq, Sk), generator=g, device="cuda")
    mask = None
    if topk:
        mask = torch.where(torch.rand((AB, ASq, Sk), generator=g, device="cuda") < 0.3, float("-inf"), torch.randn((AB, ASq, Sk), generator=g, device="cuda"))
        mask[:, 7] = float("-inf")
    got, want = (torch.empty((AB, ASq), device="cuda") for _ in range(2))
    ops.dsa_indexer_loss(q, k, idx, softmax_scale=AD ** -0.5, out=got, index_mask=mask)
    a = _lib.DsaLossArgs()
    a.struct_size, a.in_dtype, a.softmax_scale = _lib.DsaLossArgs.workspace.offset, _lib.BF16, AD ** -0.5
    a.query, a.key, a.index_scores, a.index_mask, a.loss = q.data_ptr(), k.data_ptr(), idx.data_ptr(), _lib.ptr(mask), want.data_ptr()
    a.seq_q, a.batch, a.heads, a.head_dim, a.seq_k = ASq, AB, AH, AD, Sk
    assert _lib.load().cppmega_mi355_dsa_indexer_loss(C.byref(a), a.struct_size, _lib.current_stream(q.device)) == 0
    torch.testing.assert_close(got, want, atol=2e-5, rtol=2e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["list", "mask", "dense"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_key_rows_that_do_not_count_may_hold_anything(form, bad, dt):
    """Keys that no position attends to (behind the last position, on no list, masked) and keys that only the positions in
    front of them name are not finite; the tiles they share with keys that count give what finite rows give."""
    from cppmega_mlx_amd import ops
    ASq, AB, AH, AD, Sk, topk = 150, 1, 2, 64 if form == "list" else 96, 203, 40       # (short dense rows of 64 take another kernel)
    q, k, idx, top = _case(77, ASq, AB, AH, AD, Sk, topk, DTYPES[dt])
    broken = torch.zeros(Sk, dtype=torch.bool)
    broken[ASq:] = True                                   # behind the last position
    if form != "dense":
        broken[[3, 70, 100]] = True                       # masked where a position could see them
    mask = None
    if form == "list":
        visible = torch.arange(Sk)[None, :] <= torch.arange(ASq)[:, None]
        top[0] = (torch.rand((ASq, Sk), generator=torch.Generator().manual_seed(1)) - 2.0 * (visible & broken)).topk(topk, dim=-1).indices
    elif form == "mask":
        mask = torch.randn((AB, ASq, Sk), generator=torch.Generator().manual_seed(2))
        mask[:, :, broken] = float("-inf")
    kb = k.clone()
    kb[broken] = bad
    out = torch.empty((AB, ASq), device="cuda")
    ops.dsa_indexer_loss(q.cuda(), kb.cuda(), idx.cuda(), softmax_scale=AD ** -0.5, out=out, index_mask=None if mask is None else mask.cuda(),
                         topk_indices=top.cuda() if form == "list" else None)
    if mask is None:
        want = _want(q, k, idx, top, AD ** -0.5, form == "list")
    else:
        want = od.dsa_indexer_loss_per_position(idx.numpy(), q.float().numpy(), k.float().numpy(), softmax_scale=AD ** -0.5, index_mask=mask.numpy())
    np.testing.assert_allclose(out.cpu().numpy(), want, atol=2e-5, rtol=2e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("at", [(0, 0), (1, 149), (1, 70)])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_lists_out_of_range_leave_the_output_as_it_was(dt, at):
    q, k, idx, top = (t.cuda() for t in _case(8, 150, 2, 4, 64, 150, 20, DTYPES[dt]))
    out = torch.full((2, 150), 5.0, device="cuda")
    bad = top.clone()
    bad[at[0], at[1], 3] = 150
    with pytest.raises(ValueError, match="out of range"):
        dsa_splitk_indexer_loss_per_position(idx, bad, q, k, 0.125, True, out=out)
    torch.cuda.synchronize()
    assert (out == 5.0).all()
    dsa_splitk_indexer_loss_per_position(idx, top, q, k, 0.125, True, out=out)       # (and the next call is not held up)
    assert not (out == 5.0).any()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(150, 1, 3, 64, 170, 40), (330, 2, 6, 128, 330, 50), (340, 1, 5, 64, 340, 30), (70, 1, 2, 128, 70, 9), (1100, 3, 5, 96, 1100, 64)])
@pytest.mark.parametrize("sparse", [False, True])
def test_scores_far_from_zero(shape, sparse):
    """Tiles whose exponentials leave float32 without a maximum taken off beside tiles where they do not; heads that are not
    whole groups of two or four.  Scores of up to 250 in base 2 are good to 250 * 2^-23 = 3e-5, and so are the shares."""
    ASq, AB, AH, AD, Sk, topk = shape
    q, k, idx, top = _case(ASq + AH, ASq, AB, AH, AD, Sk, topk, torch.bfloat16)
    q[ASq // 3:] *= 32
    got = dsa_splitk_indexer_loss_per_position(idx.cuda(), top.cuda(), q.cuda(), k.cuda(), AD ** -0.5, sparse).cpu().numpy()
    np.testing.assert_allclose(got, _want(q, k, idx, top, AD ** -0.5, sparse), atol=2e-5, rtol=2e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(420, 1, 8, 64, 420, 100), (420, 1, 8, 128, 420, 100)])
@pytest.mark.parametrize("sparse", [False, True])
def test_scores_on_a_common_level_lose_no_digits(shape, sparse):
    """Scores around 25 in base 2.  A head's log2 of its denominator, in [32, 64), is rounded to float32 once: off by up to
    2^-19, its share by that times ln 2, 7.6e-7 rms; the mean of 8 heads by 2.7e-7, and a loss of about one by up to twice
    that.  (3.1e-7 .. 4.3e-7 measured; 1.2e-6 .. 1.8e-6 where the scores themselves are rounded before a maximum is taken off.)"""
    ASq, AB, AH, AD, Sk, topk = shape
    q, k, idx, top = _case(5, ASq, AB, AH, AD, Sk, topk, torch.bfloat16)
    scale = AD ** -0.5
    q[..., 0], k[..., 0] = 25 / 1.4427 / scale / 4, 4.0
    got = dsa_splitk_indexer_loss_per_position(idx.cuda(), top.cuda(), q.cuda(), k.cuda(), scale, sparse).cpu().numpy()
    want = _want(q, k, idx, top, scale, sparse)
    assert np.sqrt(np.mean(((got - want) / np.maximum(1.0, np.abs(want))) ** 2)) <= 8e-7


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(128, 1, 16, 64, 128, 1), (128, 1, 17, 64, 128, 1), (192, 2, 12, 64, 192, 1), (193, 1, 24, 32, 193, 1), (320, 1, 5, 64, 320, 1), (321, 1, 5, 64, 321, 1), (40, 1, 128, 32, 128, 1)])
def test_short_dense_losses_on_both_sides_of_the_one_launch_rule(shape):
    ASq, AB, AH, AD, Sk, topk = shape
    q, k, idx, top = _case(ASq + AH, ASq, AB, AH, AD, Sk, topk, torch.bfloat16)
    got = dsa_splitk_indexer_loss_per_position(idx.cuda(), None, q.cuda(), k.cuda(), AD ** -0.5, False).cpu().numpy()
    np.testing.assert_allclose(got, _want(q, k, idx, top, AD ** -0.5, False), atol=2e-5, rtol=2e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(330, 2, 6, 64, 330, 50), (330, 1, 16, 64, 341, 50), (330, 1, 3, 128, 330, 50), (2750, 1, 2, 64, 2750, 60)],
                         ids=["split", "statistics_in_the_first_pass", "large_heads", "whole_tiles"])
@pytest.mark.parametrize("sparse", [False, True])
def test_index_scores_that_are_not_finite(shape, sparse):
    """Scores that count and are -inf or NaN carry no probability; scores that no list names may be anything."""
    ASq, AB, AH, AD, Sk, topk = shape
    q, k, idx, top = _case(ASq + AH, ASq, AB, AH, AD, Sk, topk, torch.bfloat16)
    member = torch.ones(idx.shape, dtype=torch.bool)
    if sparse:
        member = torch.zeros(idx.shape, dtype=torch.bool).scatter_(2, top, True)
    draw = torch.rand(idx.shape, generator=torch.Generator().manual_seed(5))
    gone = member & (draw < 0.05)
    gone[..., 0] = False
    bad = torch.where(gone, torch.where(draw < 0.02, float("nan"), float("-inf")), idx)
    for i, value in enumerate((float("nan"), float("inf"), float("-inf"))):
        bad[~member & (draw > 0.9 + 0.03 * i) & (draw <= 0.93 + 0.03 * i)] = value
    got = dsa_splitk_indexer_loss_per_position(bad.cuda(), top.cuda(), q.cuda(), k.cuda(), AD ** -0.5, sparse).cpu().numpy()
    clean = torch.where(gone, float("-inf"), idx)
    np.testing.assert_allclose(got, _want(q, k, clean, top, AD ** -0.5, sparse), atol=2e-5, rtol=2e-4)


def test_scores_of_eight_million_keys_take_the_tiled_path():
    """The size query is the same function of the positions on both sides of where 64 rows of scores leave 31 bits of offset."""
    import ctypes as C

    from cppmega_mlx_amd import _lib
    sizes = []
    for Sk in ((1 << 23) - 1, 1 << 23, (1 << 24) + 1, (1 << 30) + 1):
        a = _lib.DsaLossArgs()
        a.struct_size, a.in_dtype = C.sizeof(a), _lib.BF16
        a.seq_q, a.batch, a.heads, a.head_dim, a.seq_k = 130, 1, 8, 32, Sk
        need = C.c_size_t(0)
        assert _lib.load().cppmega_mi355_dsa_indexer_loss_workspace_bytes(C.byref(a), C.sizeof(a), C.byref(need)) == _lib.OK
        sizes.append(need.value)
    assert sizes[0] > 0 and sizes == sizes[:1] * 4


@pytest.mark.gpu
@pytest.mark.parametrize("AH,AD,scale", [(2, 32, 0.2), (4, 64, 0.1), (4, 64, -0.1), (3, 128, 0.1)],
                         ids=["split_in_two", "split_in_four", "masks_behind_the_products", "large_heads"])
@pytest.mark.parametrize("Sk", [(1 << 23) + 5, (1 << 24) + 2])
def test_scores_of_eight_million_keys(AH, AD, scale, Sk):
    """64 rows of scores are 2 and 4 GB: the tolerance of the other shapes, with the softmax over all keys in float64."""
    ASq = 130
    g = torch.Generator(device="cuda").manual_seed(AH + AD)
    q = torch.randn((ASq, 1, AH, AD), generator=g, device="cuda").to(torch.bfloat16)
    k = torch.zeros((Sk, 1, AH, AD), dtype=torch.bfloat16, device="cuda")
    k[:ASq] = torch.randn((ASq, 1, AH, AD), generator=g, device="cuda").to(torch.bfloat16)
    scores = torch.randn((1, ASq, Sk), generator=g, device="cuda")
    scores[..., :ASq] += 12.0                            # (the visible keys hold a share that the logarithm's offset does not hide)
    got = dsa_splitk_indexer_loss_per_position(scores, None, q, k, scale, False).double().cpu().numpy()
    log_sum = torch.stack([torch.logsumexp(scores[0, i].double(), 0) for i in range(ASq)])
    index = torch.exp(scores[0, :, :ASq].double() - log_sum[:, None])
    hidden = torch.ones((ASq, ASq), dtype=torch.bool, device="cuda").triu(1)
    p = torch.zeros((ASq, ASq), dtype=torch.float64, device="cuda")
    for h in range(AH):
        s = q[:, 0, h].double() @ k[:ASq, 0, h].double().T * scale
        p += torch.softmax(s.masked_fill(hidden, float("-inf")), -1) / AH
    want = (p * (torch.log(p + od.EPS) - torch.log(index + od.EPS))).masked_fill(hidden, 0.0).sum(-1).cpu().numpy()
    np.testing.assert_allclose(got[0], want, atol=2e-5, rtol=2e-4)
