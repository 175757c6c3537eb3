"""The native launch path against the Python launch helpers it stands in front of: the same results, and a refusal
(None) without a launch for what is not the plain case."""

import pytest
import torch

from cppmega_mlx_amd import ops
from cppmega_mlx_amd.inference.engine import SparseFP8KVCache, SparseFP8KVCacheConfig
from cppmega_mlx_amd.nn import mla_absorb, sparse_mla
from cppmega_mlx_amd.nn._tilelang import fp8_vecmat_path_c as vm
from cppmega_mlx_amd.nn._tilelang import sparse_mla_blockscaled_path_c as bs
from cppmega_mlx_amd.nn._tilelang import sparse_mla_fp8_path_c as f8
from cppmega_mlx_amd.nn._tilelang.dsa_splitk_indexer_loss import dsa_splitk_indexer_loss_per_position
from cppmega_mlx_amd.nn._tilelang.fused_fp8_gemm import fused_fp8_gemm
from cppmega_mlx_amd.nn._tilelang.sparse_mla_path_c import sparse_mla_bwd_path_c
from cppmega_mlx_amd.nn._tilelang.topk_selector import topk_selector, topk_selector_tilelang_direct
from cppmega_mlx_amd.nn.lightning_indexer import indexer_scores_topk


class _Declines:
    """Stands in for the extension: nothing is the plain case."""

    def __getattr__(self, name):
        return getattr(_HOST, name) if "workspace" in name else (lambda *args: None)


_HOST = ops.host


def _calls(device):
    g = torch.Generator(device=device).manual_seed(4)
    normal = lambda *s: torch.randn(s, generator=g, device=device)
    codes = lambda *s: normal(*s).to(torch.float8_e4m3fn).view(torch.uint8)
    B, S, H, T, k = 2, 3, 64, 200, 64
    q, idx = normal(B, S, H, 576).bfloat16(), torch.randint(-1, T, (B, S, 1, k), generator=g, device=device, dtype=torch.int32)
    cfg = SparseFP8KVCacheConfig(num_layers=1, batch_size=B, num_kv_heads=1, head_dim=512, max_seq_len=256, rope_dim=64, scale_block=128)
    lat, rope = normal(B, T, 1, 512).bfloat16(), normal(B, T, 1, 64).bfloat16()
    out, lse = torch.empty((B, S, H, 512), dtype=torch.bfloat16, device=device), torch.empty((B, S, H), device=device)

    def latent():
        views = SparseFP8KVCache(cfg, device).append_latent(0, lat, rope)                      # views with a batch pitch
        return views, bs.sparse_mla_blockscaled_path_c_apply_direct(q, None, views[0], views[1], idx, sm_scale=0.04, out=out.clone(), lse=lse.clone(),
                                                                    d_v=512, kv_rope=views[2])

    qc, kc, qs, ks = codes(B, S, H, 576), codes(B, T, 1, 576), normal(B, S, H).abs(), normal(B, T, 1).abs()
    sinks = normal(H)
    x, w = normal(3, 256).bfloat16(), codes(130, 256)
    scores, ends = normal(5, 300), torch.randint(1, 300, (5,), generator=g, device=device, dtype=torch.int32)
    iq, ik, iw = normal(B, S, 8, 64).bfloat16(), normal(B, T, 64).bfloat16(), normal(B, S, 8).bfloat16()
    w_uk = normal(4, 512, 128).bfloat16()
    return {
        "latent": latent,
        "per_token": lambda: f8.sparse_mla_fp8_path_c_apply_direct(qc, qs, kc, ks, idx, sm_scale=0.04, out=out.clone(), lse=lse.clone(), d_v=512, sinks=sinks),
        "float": lambda: sparse_mla.sparse_mla_attention(q, kc[..., :576].to(torch.bfloat16), idx, d_v=512, return_lse=True),
        "topk": lambda: topk_selector(scores, 20, ends=ends),
        "topk_by_value": lambda: topk_selector_tilelang_direct(scores, 20, out=torch.empty((5, 20), dtype=torch.int32, device=device), starts=ends // 2),
        "indexer": lambda: indexer_scores_topk(iq, ik, iw, sm_scale=0.1, index_topk=32),
        "fused_gemm": lambda: fused_fp8_gemm(w, torch.ones((2, 2), device=device), x.view(1, 3, 256)),
        "vecmat": lambda: vm.fp8_scaled_vecmat_path_c_direct(x, w, scale_x=None, scale_w=torch.ones((130, 2), device=device),
                                                             out=torch.empty((3, 130), dtype=torch.float32, device=device)),
        "head_gemm": lambda: ops.head_gemm(normal(3, 4, 128).bfloat16() * 0 + 1, w_uk, out=torch.empty((3, 4, 512), dtype=torch.float32, device=device)),
        "absorb": lambda: mla_absorb.absorb_query(q[..., :128].reshape(B, S, H, 128)[:, :, :4].contiguous(), w_uk.transpose(1, 2),
                                                  out=torch.empty((B, S, 4, 576), dtype=torch.bfloat16, device=device)[..., :512]),
    }


def _flat(v):
    return [t for x in v for t in _flat(x)] if isinstance(v, (tuple, list)) else [v]


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["latent", "per_token", "float", "topk", "topk_by_value", "indexer", "fused_gemm", "vecmat", "head_gemm", "absorb"])
def test_same_results_as_the_python_helpers(device, monkeypatch, name):
    call = _calls(device)[name]
    native = _flat(call())
    monkeypatch.setattr(ops, "host", _Declines())
    for a, b in zip(native, _flat(call()), strict=True):
        assert a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.gpu
def test_declines_what_is_not_the_plain_case(device):
    h, d = ops.host, device
    i32 = lambda *s: torch.zeros(s, dtype=torch.int32, device=d)
    scores = torch.zeros((4, 64), device=d)
    assert h.topk(scores, 8, None, None, None, False, False) is not None
    for bad in ((scores.cpu(), 8, None, None, None), (scores, 65, None, None, None), (scores, 0, None, None, None), (scores.T, 8, None, None, None),
                (scores.double(), 8, None, None, None), (scores, 8, None, i32(3), None), (scores, 8, None, i32(4).cpu(), None),
                (scores, 8, None, None, i32(4, 9)), (scores, 8.0, None, None, None), (scores[:0], 8, None, None, None)):
        assert h.topk(*bad, False, False) is None
    q, kv, idx = torch.zeros((1, 2, 4, 64), device=d), torch.zeros((1, 8, 1, 64), device=d), i32(1, 2, 1, 4)
    call = lambda q, kv, idx, d_v: h.sparse_mla(q, None, kv, None, None, idx, None, None, None, d_v, 1.0, ops.RULES_FLOAT, 0, False)
    assert call(q, kv, idx, 32) is not None
    for bad in ((q, kv, idx, 65), (q, kv, idx, 0), (q[..., :32], kv, idx, 32), (q, kv.cpu(), idx, 32), (q, kv, idx.float(), 32), (q, kv, idx[:, :1], 32),
                (q, kv[:, ::2], idx, 32), (q.to(torch.int32), kv, idx, 32), (q, kv, idx, 10 ** 30)):
        assert call(*bad) is None


def test_cpu_tensors_are_declined():
    x = torch.zeros((4, 8))
    assert ops.host.topk(x, 2, None, None, None, False, False) is None
    assert ops.host.fused_gemm(x, x, x, None) is None and ops.host.topk() is None


def _training_calls(device):
    g = torch.Generator(device=device).manual_seed(9)
    normal = lambda *s: torch.randn(s, generator=g, device=device)
    B, S, H, T, k = 2, 5, 16, 90, 24
    q, kv, d_out = normal(B, S, H, 576).half(), normal(B, T, 1, 576).half(), normal(B, S, H, 512).half()
    idx = torch.randint(-1, T, (B, S, 1, k), generator=g, device=device, dtype=torch.int32)
    query, key, scores = normal(300, B, 4, 64).bfloat16(), normal(300, B, 4, 64).bfloat16(), normal(B, 300, 300)
    lists = scores.topk(40, dim=-1).indices
    per_position = dsa_splitk_indexer_loss_per_position
    return {
        "backward": lambda: sparse_mla_bwd_path_c(q, kv, d_out, idx, d_v=512),
        "backward_scaled": lambda: sparse_mla_bwd_path_c(q.float(), kv.float(), d_out.float(), idx.long(), sm_scale=0.03, d_v=512),
        "loss": lambda: per_position(scores, None, query, key, 0.125, False),
        "loss_lists": lambda: per_position(scores, lists, query, key, 0.125, True, out=torch.empty((B, 300), device=device)),
        "loss_lists_int32": lambda: per_position(scores, lists.int(), query.float(), key.float(), 0.125, True),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["backward", "backward_scaled", "loss", "loss_lists", "loss_lists_int32"])
def test_training_calls_give_the_results_of_the_python_helpers(device, monkeypatch, name):
    call = _training_calls(device)[name]
    native = _flat(call())
    monkeypatch.setattr(ops, "host", _Declines())
    for a, b in zip(native, _flat(call()), strict=True):
        assert a.dtype == b.dtype and a.stride() == b.stride()
        # (float32 rows of the backward are added with atomics: no order, sums of up to 2 x 5 x 16 terms)
        assert torch.equal(a, b) if name != "backward_scaled" else torch.allclose(a, b, rtol=1e-4, atol=1e-4 * b.abs().max().item())


@pytest.mark.gpu
def test_training_calls_decline_what_is_not_the_plain_case(device):
    host = _HOST
    q, kv, d_out = (torch.zeros(s, device=device, dtype=torch.bfloat16) for s in ((1, 2, 16, 576), (1, 9, 1, 576), (1, 2, 16, 512)))
    idx = torch.zeros((1, 2, 1, 4), device=device, dtype=torch.int32)
    assert host.mla_backward(q, kv, d_out, idx, None, 512) is not None
    for args in ((q.cpu(), kv, d_out, idx, None, 512), (q, kv.half(), d_out, idx, None, 512), (q, kv, d_out[..., :500], idx, None, 500),
                 (q, kv, d_out, idx, 1, 512), (q, kv, d_out, idx, None, 577), (q, kv, d_out, idx.float(), None, 512), (q[:, :0], kv, d_out[:, :0], idx[:, :0], None, 512)):
        assert host.mla_backward(*args) is None
    query, scores = torch.zeros((300, 1, 4, 64), device=device, dtype=torch.bfloat16), torch.zeros((1, 300, 300), device=device)
    lists = torch.zeros((1, 300, 8), device=device, dtype=torch.int32)
    watch = ops._range_watch(scores.device)
    good = (scores, lists, query, query, 0.1, None, watch.flag_address, watch.event_handle)
    assert host.indexer_loss(*good) is not None
    for i, bad in ((0, scores.half()), (0, scores[:, :, :299]), (1, lists[:, :, :0]), (1, lists[:, :299]), (2, query.float()), (4, 1), (5, scores), (6, 0), (7, 0)):
        assert host.indexer_loss(*good[:i], bad, *good[i + 1:]) is None
    out = torch.full((1, 300), 7.0, device=device)
    lists[0, 5, 3] = 300
    assert host.indexer_loss(*good[:5], out, *good[6:]) is False and (out == 7.0).all()
    assert host.indexer_loss(*good) is False
    lists[0, 5, 3] = 0
    assert host.indexer_loss(*good) is not None          # (the report is of one call)
