"""Performance cases of the sparse-attention path, called the way a user's program calls them.

Each case is a dict of plain values; its "kind" names the entry point:

  attn_float   ``sparse_mla_attention`` over unquantised 16-bit rows
  attn_latent  ``sparse_mla_blockscaled_path_c_apply_direct`` over the FP8 latent cache (prefill and decode)
  attn_fp8     the prepared-buffer FP8 forwards (per-token float32 scales, or E8M0 bytes per 32 channels)
  layer        one decode step of an attention layer: cache append, indexer, absorbed query, attention,
               per-head value projection, FP8 output projection
  proj         an FP8 block-scaled linear layer, from one decode token to a prefill chunk
  topk         the selector on its own
  indexer      ``indexer_scores_topk``
  backward     ``sparse_mla_bwd_path_c``
  loss         the indexer's KL loss
"""

import math

import torch

from cppmega_mlx_amd import ops
from cppmega_mlx_amd.inference.engine import SparseFP8KVCache, SparseFP8KVCacheConfig
from cppmega_mlx_amd.nn._tilelang import fp8_vecmat_path_c as vecmat
from cppmega_mlx_amd.nn._tilelang import sparse_mla_blockscaled_path_c as blockscaled
from cppmega_mlx_amd.nn._tilelang import sparse_mla_fp8_path_c as fp8_path
from cppmega_mlx_amd.nn._tilelang.dsa_splitk_indexer_loss import dsa_splitk_indexer_loss_per_position
from cppmega_mlx_amd.nn._tilelang.fused_fp8_gemm import fused_fp8_gemm
from cppmega_mlx_amd.nn._tilelang.sparse_mla_path_c import sparse_mla_bwd_path_c
from cppmega_mlx_amd.nn._tilelang.topk_selector import topk_selector, topk_selector_tilelang_direct
from cppmega_mlx_amd.nn.lightning_indexer import indexer_scores_topk
from cppmega_mlx_amd.nn.mla_absorb import absorb_query
from cppmega_mlx_amd.nn.sparse_mla import sparse_mla_attention

LATENT, ROPE, D_V = 512, 64, 512
D_QK = LATENT + ROPE
SM_SCALE = D_QK ** -0.5
HALF = {"bf16": torch.bfloat16, "f16": torch.float16}
FLOP_PER_PAIR = 2 * (D_QK + D_V)            # one query head against one selected key

# The decode layer: 128 heads of 128 + 64 query channels, 7168 model channels, an indexer of 64 heads of 128.
L_HEADS, L_DK, L_DV, L_MODEL = 128, 128, 128, 7168
I_HEADS, I_DIM = 64, 128


def listed():
    return [
        # the smallest call: a toy-sized forward, all launch and host time
        {"name": "attn_small_bf16", "kind": "attn_float", "dtype": "bf16", "batch": 1, "queries": 64, "heads": 16, "keys": 256, "topk": 64},
        # the attention of one decode step of 32 sequences with 64k tokens each
        {"name": "decode_b32_64k", "kind": "attn_latent", "batch": 32, "queries": 1, "heads": 128, "keys": 65536, "topk": 2048},
        # the attention of a whole causal prefill
        {"name": "prefill_8k", "kind": "attn_latent", "batch": 1, "queries": 8192, "heads": 128, "keys": 8192, "topk": 2048},
        # a ragged chunk behind a past, on the prepared per-token FP8 buffers
        {"name": "prefill_fp8_rows", "kind": "attn_fp8", "scales": "token", "batch": 1, "queries": 999, "heads": 128, "keys": 4099, "topk": 2048},
        # everything that one attention layer runs for one new token of a few sequences
        {"name": "decode_layer_b4", "kind": "layer", "batch": 4, "keys": 8191, "topk": 2048},
        # output projection of one token, of a small batch, and an up-projection of a prefill chunk
        {"name": "proj_m1", "kind": "proj", "dtype": "bf16", "scales": "row", "m": 1, "n": 7168, "k": 16384},
        {"name": "proj_m16", "kind": "proj", "dtype": "bf16", "scales": "grid", "m": 16, "n": 7168, "k": 16384},
        {"name": "proj_prefill", "kind": "proj", "dtype": "bf16", "scales": "grid", "m": 2048, "n": 8192, "k": 1536},
        # selection for a batch of prefill chunks, causal bounds, tied scores
        {"name": "topk_prefill", "kind": "topk", "order": "index", "rows": 4096, "width": 8192, "topk": 2048},
        # scores and selection of one decode step over long caches
        {"name": "indexer_decode", "kind": "indexer", "batch": 32, "queries": 1, "keys": 65536, "topk": 2048},
        # training: gradients of the attention, and the indexer's loss
        {"name": "attn_backward", "kind": "backward", "dtype": "bf16", "batch": 1, "queries": 1024, "heads": 16, "keys": 4096, "topk": 256},
        {"name": "indexer_loss", "kind": "loss", "dtype": "bf16", "batch": 1, "positions": 4096, "heads": 8, "dim": 64, "topk": 1024},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, uniform in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attn_float", "attn_latent", "attn_latent", "attn_fp8", "layer", "proj", "proj", "topk", "indexer", "backward", "loss"])
    if kind == "attn_float":
        keys = _log(rng, 128, 8192)
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16"]), "batch": rng.randint(1, 2), "queries": _log(rng, 1, min(keys, 1024)),
                "heads": rng.choice([16, 64, 128]), "keys": keys, "topk": min(keys, _log(rng, 64, 2048))}
    if kind == "attn_latent":
        heads, topk = rng.choice([16, 64, 128]), rng.choice([512, 1024, 2048])
        if rng.random() < 0.5:                                   # decode
            batch = _log(rng, 1, 32)
            return {"kind": kind, "batch": batch, "queries": 1, "heads": heads, "keys": _log(rng, topk, 65536), "topk": topk}
        queries = _log(rng, 16, 6000)                            # a prefill chunk, with or without a past
        past = rng.choice([0, _log(rng, 64, 8192)])
        return {"kind": kind, "batch": 1, "queries": queries, "heads": heads, "keys": max(topk, queries + past), "topk": topk}
    if kind == "attn_fp8":
        keys = _log(rng, 512, 16384)
        return {"kind": kind, "scales": rng.choice(["token", "token", "e8m0"]), "batch": 1, "queries": _log(rng, 1, min(keys, 2048)),
                "heads": rng.choice([16, 64, 128]), "keys": keys, "topk": min(keys, _log(rng, 256, 2048))}
    if kind == "layer":
        keys = _log(rng, 2048, 32768)
        return {"kind": kind, "batch": _log(rng, 1, 32), "keys": keys, "topk": rng.choice([1024, 2048])}
    if kind == "proj":
        n, k = _log(rng, 256, 16384), 128 * _log(rng, 4, 128)
        m = _log(rng, 1, min(4096, int(2e11 / (n * k))))
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "bf16", "f16"]), "scales": rng.choice(["grid", "row"]), "m": m, "n": n, "k": k}
    if kind == "topk":
        width = _log(rng, 512, 65536)
        return {"kind": kind, "order": rng.choice(["index", "index", "value"]), "rows": _log(rng, 1, min(4096, (1 << 25) // width)),
                "width": width, "topk": min(width, _log(rng, 64, 2048))}
    if kind == "indexer":
        if rng.random() < 0.5:
            return {"kind": kind, "batch": _log(rng, 1, 32), "queries": 1, "keys": _log(rng, 2048, 65536), "topk": 2048}
        queries = _log(rng, 64, 4096)
        return {"kind": kind, "batch": 1, "queries": queries, "keys": queries + _log(rng, 64, 8192), "topk": rng.choice([1024, 2048])}
    if kind == "backward":
        keys = _log(rng, 512, 8192)
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16"]), "batch": 1, "queries": _log(rng, 64, min(keys, 1024)),
                "heads": rng.choice([8, 16, 32, 64]), "keys": keys, "topk": _log(rng, 64, 512)}
    positions = _log(rng, 256, 4096)
    return {"kind": kind, "dtype": rng.choice(["bf16", "f16"]), "batch": rng.randint(1, 2), "positions": positions,
            "heads": rng.choice([8, 16]), "dim": rng.choice([64, 128]), "topk": rng.choice([0, max(64, positions // 4)])}


# --------------------------------------------------------------------------- inputs

class _Maker:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32):
        return torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32).to(dtype)

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda")

    def codes(self, x, block):
        """e4m3 bytes of x [..., K] and amax / 448 per ``block`` channels."""
        blocks = x.reshape(*x.shape[:-1], x.shape[-1] // block, block)
        scale = (blocks.abs().amax(-1) / 448.0).clamp_min(1e-12)
        return (blocks / scale[..., None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8).reshape(x.shape).contiguous(), scale.contiguous()

    def selection(self, batch, queries, keys, topk):
        """What an indexer hands over: the query at position keys - queries + s attends to topk of the keys up to
        its own, ascending, with -1 behind them where fewer are visible."""
        out = torch.empty((batch, queries, 1, topk), dtype=torch.int32, device="cuda")
        col = torch.arange(keys, device="cuda")
        for b in range(batch):
            for s in range(0, queries, 2048):
                e = min(queries, s + 2048)
                last = torch.arange(s, e, device="cuda") + (keys - queries)
                r = self.uniform(e - s, keys) - 2.0 * (col[None, :] > last[:, None])
                idx = torch.where(r >= 0, col[None, :], keys).gather(1, r.topk(topk, dim=-1).indices).sort(-1).values
                out[b, s:e, 0] = torch.where(idx < keys, idx, -1).to(torch.int32)
        return out

    def latent_cache(self, batch, keys):
        kv = torch.empty((batch, keys, 1, LATENT), dtype=torch.uint8, device="cuda")
        scale = torch.empty((batch, keys, 1, LATENT // 128), dtype=torch.float32, device="cuda")
        rope = torch.empty((batch, keys, 1, ROPE), dtype=torch.bfloat16, device="cuda")
        for b in range(batch):
            kv[b], scale[b] = self.codes(self.normal(keys, 1, LATENT), 128)
            rope[b] = self.normal(keys, 1, ROPE)
        return kv, scale, rope

    def weight(self, n, k, scales):
        w = self.normal(n, k) * k ** -0.5
        if scales == "row":
            return self.codes(w, 128)
        n_pad = -n % 128
        tiles = torch.nn.functional.pad(w, (0, 0, 0, n_pad)).reshape((n + n_pad) // 128, 128, k // 128, 128)
        scale = (tiles.abs().amax(dim=(1, 3)) / 448.0).contiguous()
        codes = (tiles / scale[:, None, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
        return codes.reshape(n + n_pad, k)[:n].contiguous(), scale


def prepare(case, seed):
    make, c = _Maker(seed), case
    kind = c["kind"]
    s = {"case": c}
    if kind == "attn_float":
        dt = HALF[c["dtype"]]
        s["q"] = make.normal(c["batch"], c["queries"], c["heads"], D_QK, dtype=dt)
        s["kv"] = make.normal(c["batch"], c["keys"], 1, D_QK, dtype=dt)
        s["indices"] = make.selection(c["batch"], c["queries"], c["keys"], c["topk"])
    elif kind == "attn_latent":
        s["q"] = make.normal(c["batch"], c["queries"], c["heads"], D_QK, dtype=torch.bfloat16)
        s["kv"], s["scale"], s["rope"] = make.latent_cache(c["batch"], c["keys"])
        s["indices"] = make.selection(c["batch"], c["queries"], c["keys"], c["topk"])
        s["out"] = torch.empty((c["batch"], c["queries"], c["heads"], D_V), dtype=torch.bfloat16, device="cuda")
        s["lse"] = torch.empty((c["batch"], c["queries"], c["heads"]), dtype=torch.float32, device="cuda")
    elif kind == "attn_fp8":
        q, kv = make.normal(c["batch"], c["queries"], c["heads"], D_QK), make.normal(c["batch"], c["keys"], 1, D_QK)
        if c["scales"] == "token":
            s["q"], q_scale = make.codes(q, D_QK)
            s["kv"], kv_scale = make.codes(kv, D_QK)
            s["q_scale"], s["kv_scale"] = q_scale[..., 0].contiguous(), kv_scale[..., 0].contiguous()
        else:                                                    # power-of-two scales, one byte per 32 channels
            for name, x in (("q", q), ("kv", kv)):
                blocks = x.reshape(*x.shape[:-1], D_QK // 32, 32)
                e = torch.ceil(torch.log2(blocks.abs().amax(-1) / 448.0))
                s[name] = (blocks * torch.exp2(-e)[..., None]).to(torch.float8_e4m3fn).view(torch.uint8).reshape(x.shape).contiguous()
                s[name + "_scale"] = (e + 127).to(torch.uint8).contiguous()
        s["indices"] = make.selection(c["batch"], c["queries"], c["keys"], c["topk"])
        s["out"] = torch.empty((c["batch"], c["queries"], c["heads"], D_V), dtype=torch.bfloat16, device="cuda")
        s["lse"] = torch.empty((c["batch"], c["queries"], c["heads"]), dtype=torch.float32, device="cuda")
    elif kind == "layer":
        B, T = c["batch"], c["keys"]
        s["cache"] = SparseFP8KVCache(SparseFP8KVCacheConfig(num_layers=1, batch_size=B, num_kv_heads=1, head_dim=LATENT, max_seq_len=T + 64,
                                                             rope_dim=ROPE, scale_block=128))
        s["cache"].append_latent(0, make.normal(B, T - 1, 1, LATENT, dtype=torch.bfloat16), make.normal(B, T - 1, 1, ROPE, dtype=torch.bfloat16))
        s["latent"], s["rope"] = make.normal(B, 1, 1, LATENT, dtype=torch.bfloat16), make.normal(B, 1, 1, ROPE, dtype=torch.bfloat16)
        s["index_q"] = make.normal(B, 1, I_HEADS, I_DIM, dtype=torch.bfloat16)
        s["index_k"] = make.normal(B, T, I_DIM, dtype=torch.bfloat16)
        s["index_w"] = (make.normal(B, 1, I_HEADS) * I_HEADS ** -0.5).to(torch.bfloat16)
        s["q_nope"] = make.normal(B, 1, L_HEADS, L_DK, dtype=torch.bfloat16)
        s["q_rope"] = make.normal(B, 1, L_HEADS, ROPE, dtype=torch.bfloat16)
        s["q"] = torch.empty((B, 1, L_HEADS, D_QK), dtype=torch.bfloat16, device="cuda")
        s["w_uk"] = (make.normal(L_HEADS, LATENT, L_DK) * L_DK ** -0.5).to(torch.bfloat16).transpose(1, 2)
        s["w_uv"] = (make.normal(L_HEADS, L_DV, LATENT) * LATENT ** -0.5).to(torch.bfloat16)
        s["w_o"], s["w_o_scale"] = make.weight(L_MODEL, L_HEADS * L_DV, "grid")
        s["attended"] = torch.empty((B, 1, L_HEADS, D_V), dtype=torch.bfloat16, device="cuda")
        s["lse"] = torch.empty((B, 1, L_HEADS), dtype=torch.float32, device="cuda")
        s["heads"] = torch.empty((B, L_HEADS, L_DV), dtype=torch.bfloat16, device="cuda")
    elif kind == "proj":
        s["w"], s["w_scale"] = make.weight(c["n"], c["k"], c["scales"])
        s["x"] = make.normal(c["m"], c["k"], dtype=HALF[c["dtype"]])
        s["out"] = torch.empty((c["m"], c["n"]), dtype=HALF[c["dtype"]], device="cuda")
    elif kind == "topk":
        rows, width = c["rows"], c["width"]
        x = make.normal(rows, width)
        s["scores"] = torch.where(make.uniform(rows, width) < 0.05, x.roll(1, dims=1), x)       # a twentieth are copies of their neighbour
        chunk = min(rows, max(1, width // 8))                    # causal: the queries of a chunk see one key more each
        s["ends"] = (width - chunk + 1 + torch.arange(rows, device="cuda") % chunk).to(torch.int32)
        s["out"] = torch.empty((rows, c["topk"]), dtype=torch.int32, device="cuda")
    elif kind == "indexer":
        B, S, T = c["batch"], c["queries"], c["keys"]
        s["q"] = make.normal(B, S, I_HEADS, I_DIM, dtype=torch.bfloat16)
        s["k"] = make.normal(B, T, I_DIM, dtype=torch.bfloat16)
        s["w"] = (make.normal(B, S, I_HEADS) * I_HEADS ** -0.5).to(torch.bfloat16)
        s["ends"] = (torch.arange(1, S + 1, device="cuda") + (T - S)).repeat(B).to(torch.int32)
    elif kind == "backward":
        dt = HALF[c["dtype"]]
        s["q"] = make.normal(c["batch"], c["queries"], c["heads"], D_QK, dtype=dt)
        s["kv"] = make.normal(c["batch"], c["keys"], 1, D_QK, dtype=dt)
        s["d_out"] = make.normal(c["batch"], c["queries"], c["heads"], D_V, dtype=dt)
        s["indices"] = make.selection(c["batch"], c["queries"], c["keys"], c["topk"])
    else:
        B, T, dt = c["batch"], c["positions"], HALF[c["dtype"]]
        s["query"], s["key"] = (make.normal(T, B, c["heads"], c["dim"], dtype=dt) for _ in range(2))
        s["scores"] = make.normal(B, T, T)
        s["indices"] = None
        if c["topk"]:                                            # keys behind the query's own come last in its list
            pos = torch.arange(T, device="cuda")
            s["indices"] = (s["scores"] - 20.0 * (pos[None, :] > pos[:, None])).topk(c["topk"], dim=-1).indices.to(torch.int32)
    return s


# --------------------------------------------------------------------------- one pass

def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "attn_float":
        return sparse_mla_attention(s["q"], s["kv"], s["indices"], d_v=D_V, return_lse=True)
    if kind == "attn_latent":
        return blockscaled.sparse_mla_blockscaled_path_c_apply_direct(s["q"], None, s["kv"], s["scale"], s["indices"], sm_scale=SM_SCALE,
                                                                      out=s["out"], lse=s["lse"], d_v=D_V, kv_rope=s["rope"])
    if kind == "attn_fp8":
        apply = (fp8_path.sparse_mla_fp8_path_c_apply_direct if c["scales"] == "token"
                 else blockscaled.sparse_mla_blockscaled_path_c_apply_direct)
        return apply(s["q"], s["q_scale"], s["kv"], s["kv_scale"], s["indices"], sm_scale=SM_SCALE, out=s["out"], lse=s["lse"], d_v=D_V)
    if kind == "layer":
        return _decode_step(s)
    if kind == "proj":
        if c["m"] == 1 and c["scales"] == "row":
            return vecmat.fp8_scaled_vecmat_path_c_direct(s["x"], s["w"], scale_x=None, scale_w=s["w_scale"], out=s["out"])
        return fused_fp8_gemm(s["w"], s["w_scale"], s["x"])
    if kind == "topk":
        if c["order"] == "index":
            return topk_selector(s["scores"], c["topk"], ends=s["ends"])
        return topk_selector_tilelang_direct(s["scores"], c["topk"], out=s["out"], ends=s["ends"])
    if kind == "indexer":
        return indexer_scores_topk(s["q"], s["k"], s["w"], sm_scale=I_DIM ** -0.5, index_topk=c["topk"], ends=s["ends"])
    if kind == "backward":
        return sparse_mla_bwd_path_c(s["q"], s["kv"], s["d_out"], s["indices"], d_v=D_V)
    return dsa_splitk_indexer_loss_per_position(s["scores"], s["indices"], s["query"], s["key"], c["dim"] ** -0.5, bool(c["topk"]))


def _decode_step(s):
    batch = s["case"]["batch"]
    kv, scale, rope = s["cache"].append_latent(0, s["latent"], s["rope"])
    indices = indexer_scores_topk(s["index_q"], s["index_k"], s["index_w"], sm_scale=I_DIM ** -0.5, index_topk=s["case"]["topk"])
    s["q"][..., LATENT:] = s["q_rope"]
    absorb_query(s["q_nope"], s["w_uk"], out=s["q"][..., :LATENT])
    blockscaled.sparse_mla_blockscaled_path_c_apply_direct(s["q"], None, kv, scale, indices.unsqueeze(2), sm_scale=(L_DK + ROPE) ** -0.5,
                                                           out=s["attended"], lse=s["lse"], d_v=D_V, kv_rope=rope)
    ops.head_gemm(s["attended"].view(batch, L_HEADS, LATENT), s["w_uv"], out=s["heads"])
    y = fused_fp8_gemm(s["w_o"], s["w_o_scale"], s["heads"].view(batch, L_HEADS * L_DV))
    row = kv.shape[1] - 1
    s["cache"].trim(1)                                           # the next pass writes the same position again
    return {"y": y, "indices": indices, "kv": kv[:, row:], "scale": scale[:, row:], "rope": rope[:, row:]}


# --------------------------------------------------------------------------- what a pass cannot do without

def _pairs(c):
    """Selected (query, key) pairs of a causal selection."""
    queries, keys, topk = c["queries"], c["keys"], c["topk"]
    first = keys - queries + 1                                   # keys the first query sees
    short = max(0, min(queries, topk - first))
    pairs = short * first + short * (short - 1) // 2 + (queries - short) * topk
    return c["batch"] * pairs


def _attention(c, row_bytes, q_bytes, out_bytes):
    pairs, rows = _pairs(c), c["batch"] * c["queries"] * c["heads"]
    nbytes = (min(pairs, c["batch"] * c["keys"]) * row_bytes + c["batch"] * c["queries"] * c["topk"] * 4
              + rows * (q_bytes + D_V * out_bytes + 4))
    return {"bytes": nbytes, "flops": pairs * c["heads"] * FLOP_PER_PAIR}


def work(case):
    c = case
    kind = c["kind"]
    if kind == "attn_float":
        return _attention(c, 2 * D_QK, 2 * D_QK, 2)
    if kind == "attn_latent":
        return _attention(c, LATENT + 4 * (LATENT // 128) + 2 * ROPE, 2 * D_QK, 2)
    if kind == "attn_fp8":
        side = D_QK + (4 if c["scales"] == "token" else D_QK // 32)
        return _attention(c, side, side, 2)
    if kind == "layer":
        B, T = c["batch"], c["keys"]
        attn = _attention(dict(c, queries=1, heads=L_HEADS), LATENT + 16 + 2 * ROPE, 0, 0)
        weights = L_HEADS * LATENT * (L_DK + L_DV)
        out_w = L_MODEL * L_HEADS * L_DV
        return {"bytes": attn["bytes"] + 2 * weights + out_w + B * (T * I_DIM * 2 + I_HEADS * I_DIM * 2 + L_HEADS * (L_DK + ROPE) * 2 + L_MODEL * 2
                                                                   + 2 * D_QK + 656),
                "flops": attn["flops"] + 2 * B * (weights + out_w + T * I_DIM + I_HEADS * I_DIM)}
    if kind == "proj":
        m, n, k = c["m"], c["n"], c["k"]
        n_scale = (n if c["scales"] == "row" else (n + 127) // 128) * (k // 128)
        return {"bytes": n * k + 4 * n_scale + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "topk":
        return {"bytes": 4 * c["rows"] * (c["width"] + c["topk"] + 1), "flops": 0}
    if kind == "indexer":
        B, S, T = c["batch"], c["queries"], c["keys"]
        visible = B * S * (T - (S - 1) / 2)
        topk = min(c["topk"], T)
        return {"bytes": 2 * B * (S * I_HEADS * I_DIM + T * I_DIM + S * I_HEADS) + 4 * B * S * (topk + 1),
                "flops": 2 * (B * S * I_HEADS * I_DIM + visible * I_DIM)}
    if kind == "backward":
        rows, pairs = c["batch"] * c["queries"] * c["heads"], _pairs(c)
        return {"bytes": rows * 2 * (2 * D_QK + D_V) + c["batch"] * c["keys"] * D_QK * (2 + 4) + c["batch"] * c["queries"] * c["topk"] * 4,
                "flops": 2 * pairs * c["heads"] * (3 * D_QK + 2 * D_V)}
    B, T, H, D = c["batch"], c["positions"], c["heads"], c["dim"]
    return {"bytes": 2 * 2 * B * T * H * D + 4 * B * T * ((T + 1) // 2 if not c["topk"] else c["topk"]) + 4 * B * T * (c["topk"] + 1),
            "flops": 2 * B * H * D * T * (T + 1) // 2}


def tolerance(case):
    kind = case["kind"]
    if kind == "topk":
        return "exact"
    if kind == "indexer":                                        # scores closer than float32 sums resolve may change places
        return {"rel": 0.0, "differ": 0.01}
    if kind == "layer":
        return {"rel": 1e-2, "max": 0.1, "differ": 0.01}
    if kind == "loss":                                           # float32 sums over 16-bit products, logarithms of small shares
        return {"rel": 5e-5, "max": 1e-3}
    if kind == "backward":                                       # dq is rounded to 16 bits
        return {"rel": 5e-3, "max": 0.05}
    return {"rel": 1e-2, "max": 0.1}
