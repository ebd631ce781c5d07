"""Timing cases of the sparse-attention inference path: what a serving program asks of it.

Each case is a dict of plain values; ``kind`` names the path:

* ``decode``  one token per row through ``SparseDecodeLayer``'s captured graph (emission, indexer,
  top-k, split attention and merge), rows at their own positions as under continuous batching,
  so a share of them completes a group;
* ``attend``  ``csa2_attn.fwd`` over a prompt: the sliding window and each query's selected entries;
* ``index``   the prompt's selection: query quantization, indexer scores against the published
  keys and the top-k (a later chunk of a long prompt starts at ``start``);
* ``reindex`` the two-level selection of a decode step: a source layer's dense scores, block
  list and top-k, then a following layer's scores and top-k over those candidates only;
* ``ingest``  a prompt's compressed entries: pooling and norm, RoPE, and the packed caches;
* ``module``  ``DeepseekV41Attention.forward``: a whole prompt without a cache, or a prompt and
  then single tokens through ``DeepseekV41CSACache``.

Sizes are those of ``bench.py``'s configurations and of the tests, plus small and ragged ones.
``exact`` restates each path in plain torch in 64 bits, with the roundings that define it
(quantized caches and operands, the bfloat16 tensors between its stages).
"""

import math

import torch

from mzoo_amd import cache as mcache
from mzoo_amd import csa2_attn, indexer, owlet1, quant
from mzoo_amd.decode import CompressorWeights, DecodeConfig, SparseDecodeLayer

DEV = "cuda"
THETA, COMPRESS_THETA = 10000.0, 160000.0
EPS = 1e-6


# ---- the cases ----------------------------------------------------------------------------

def listed():
    return [
        # one user's chat turn: a single row at a short context, where launches and latency count
        dict(name="decode b1 4k", kind="decode", batch=1, ctx=4096, heads=128, index_heads=64, fmt="fp8", topk=1024,
             coarse=0, nsplit=16),
        # the headline serving step: a full batch at 32k context
        dict(name="decode b32 32k", kind="decode", batch=32, ctx=32768, heads=128, index_heads=64, fmt="fp8",
             topk=2048, coarse=0, nsplit=4),
        # long documents, the 4-bit index
        dict(name="decode b8 128k mxfp4", kind="decode", batch=8, ctx=131072, heads=128, index_heads=64, fmt="mxfp4",
             topk=2048, coarse=0, nsplit=14),
        # the hierarchical form: a dense coarse branch beside the selected entries
        dict(name="decode b4 512k coarse", kind="decode", batch=4, ctx=524288, heads=128, index_heads=64, fmt="mxfp4",
             topk=2048, coarse=128, nsplit=32),
        # a long prompt's attention, every head of the latent
        dict(name="attend s8192 h128", kind="attend", batch=1, seq=8192, heads=128, dim=576, topk=2048, window=128),
        # a short ragged prompt of a smaller model: narrow latent, few heads, a real selection
        dict(name="attend s1001 h16 d160", kind="attend", batch=2, seq=1001, heads=16, dim=160, topk=128, window=64),
        # the long prompt's selection, 8-bit index
        dict(name="index s8192 fp8", kind="index", batch=1, seq=8192, start=0, heads=64, dim=128, fmt="fp8", topk=2048),
        # a later ragged chunk of a longer prompt, the 4-bit index
        dict(name="index s1021+15000 mxfp4", kind="index", batch=1, seq=1021, start=15000, heads=32, dim=128,
             fmt="mxfp4", topk=512),
        # two layers' selection at a long context: the candidate source and a layer that reuses it
        dict(name="reindex b4 512k", kind="reindex", batch=4, groups=131072, heads=64, fmt="mxfp4", topk=2048,
             blocks=2048),
        # a prompt's compressed entries into the packed caches
        dict(name="ingest s8192", kind="ingest", batch=1, seq=8192, fmt="fp8", ratio=4),
        # a small fp32 model's layer over a prompt
        dict(name="module s1024 fp32", kind="module", batch=1, seq=1024, steps=0, dtype="float32", hidden=512, heads=8,
             dim=160, rope=32, q_rank=256, o_groups=2, o_rank=128, index_heads=4, index_dim=64, topk=128, window=64),
        # a bf16 layer generating: a ragged prompt, then tokens one by one through the cache
        dict(name="module s509+8 bf16", kind="module", batch=4, seq=509, steps=8, dtype="bfloat16", hidden=4096,
             heads=128, dim=576, rope=64, q_rank=1536, o_groups=16, o_rank=1024, index_heads=64, index_dim=128,
             topk=2048, window=128),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "attend", "attend", "index", "index", "reindex", "ingest", "module"])
    if kind == "decode":
        fmt = rng.choice(["fp8", "mxfp4"])
        batch = _log(rng, 1, 32)
        ctx = _log(rng, 1500, min(524288, (1 << 20 if fmt == "fp8" else 1 << 21) // batch))
        heads = rng.choice([32, 64, 128, 128])
        nsplit = max(1, min(32, 256 // (batch * -(-heads // 64))))
        coarse = 128 if ctx >= 65536 and rng.random() < 0.4 else 0
        return dict(kind=kind, batch=batch, ctx=ctx, heads=heads, index_heads=rng.choice([32, 64, 64]), fmt=fmt,
                    topk=rng.choice([512, 1000, 2048]), coarse=coarse, nsplit=nsplit)
    if kind == "attend":
        dim = rng.choice([128, 160, 256, 576, 576])
        heads = rng.choice([8, 16, 64, 128])
        batch = rng.choice([1, 1, 2, 3])
        return dict(kind=kind, batch=batch, seq=_log(rng, 60, 8000 // batch), heads=heads, dim=dim,
                    topk=rng.choice([100, 128, 512, 2048]), window=rng.choice([64, 128]))
    if kind == "index":
        fmt = rng.choice(["fp8", "mxfp4", "bf16"])
        seq = _log(rng, 50, 8000)
        return dict(kind=kind, batch=1, seq=seq, start=rng.choice([0, 0, _log(rng, 100, 12000)]),
                    heads=rng.choice([4, 32, 64]), dim=128 if fmt != "bf16" else rng.choice([64, 128]), fmt=fmt,
                    topk=rng.choice([128, 512, 2048]))
    if kind == "reindex":
        batch = _log(rng, 1, 32)
        fmt = rng.choice(["fp8", "mxfp4"])
        return dict(kind=kind, batch=batch, groups=_log(rng, 16500, min(131072, (1 << 19) // batch)),
                    heads=rng.choice([32, 64]), fmt=fmt, topk=rng.choice([512, 2048]), blocks=rng.choice([1024, 2048]))
    if kind == "ingest":
        batch = rng.choice([1, 2, 4])
        return dict(kind=kind, batch=batch, seq=_log(rng, 130, 16000 // batch), fmt=rng.choice(["fp8", "mxfp4"]),
                    ratio=rng.choice([2, 4, 4, 128]))
    seq = _log(rng, 70, 1500)
    return dict(kind="module", batch=rng.choice([1, 2]), seq=seq, steps=rng.choice([0, 0, 5]),
                dtype=rng.choice(["float32", "bfloat16"]), hidden=512, heads=rng.choice([8, 32]), dim=160, rope=32,
                q_rank=256, o_groups=2, o_rank=128, index_heads=rng.choice([4, 32]), index_dim=64,
                topk=rng.choice([128, 512]), window=rng.choice([64, 128]))


# ---- inputs -------------------------------------------------------------------------------

def _rnd(seed):
    gen = torch.Generator(device=DEV).manual_seed(seed * 7919 + 11)
    return lambda *shape: torch.randn(*shape, generator=gen, device=DEV)


def _positions(batch, ctx, seed):
    """Rows somewhere in the second half of the context, each at its own position."""
    gen = torch.Generator().manual_seed(seed * 31 + 5)
    return torch.randint(ctx // 2, ctx, (batch,), generator=gen)


def _decode_inputs(c, seed):
    rnd = _rnd(seed)
    b, h, d, hi, w = c["batch"], c["heads"], 576, c["index_heads"], 128
    g = c["ctx"] // 4
    x = dict(pos=_positions(b, 4 * g, seed), sinks=rnd(h), kv_w=(1 + 0.1 * rnd(d)).bfloat16(),
             norm_w=(1 + 0.1 * rnd(d)).bfloat16(), wk=(0.04 * rnd(128, d)).bfloat16(),
             k_norm=(1 + 0.1 * rnd(128)).bfloat16(), win=rnd(b, w, d).bfloat16(), main=rnd(b, g, d).bfloat16(),
             keys=rnd(b, g, 128).bfloat16(), q=rnd(b, h, d).bfloat16(), kv=rnd(b, d).bfloat16(),
             q_idx=rnd(b, hi, 128).bfloat16(), w=rnd(b, hi) * hi ** -0.5, carry=(rnd(b, 3, d), rnd(b, 3, d)),
             comp=(rnd(b, d), rnd(b, d)))
    if c["coarse"]:
        r = c["coarse"]
        x.update(coarse_w=(1 + 0.1 * rnd(d)).bfloat16(), coarse=rnd(b, c["ctx"] // r, d).bfloat16(),
                 c_carry=(rnd(b, r - 1, d), rnd(b, r - 1, d)), c_comp=(rnd(b, d), rnd(b, d)))
    return x


def _causal_lists(rnd, b, s, groups, topk, ratio=4, start=0):
    """What the indexer gives: each query's best visible groups, ascending, then -1."""
    n = max(min(topk, groups), 1)
    out = torch.full((b, s, topk), -1, dtype=torch.int32, device=DEV)
    vis = (start + torch.arange(s, device=DEV) + 1) // ratio
    cols = torch.arange(groups, device=DEV)
    for i in range(b):
        for s0 in range(0, s, 1024):
            v = vis[s0:s0 + 1024, None]
            sc = rnd(v.shape[0], groups).masked_fill_(cols >= v, float("-inf"))
            val, idx = sc.topk(n, -1)
            idx = idx.masked_fill(val == float("-inf"), groups).sort(-1).values
            out[i, s0:s0 + 1024, :n] = idx.masked_fill(idx == groups, -1).int()
    return out


def _attend_inputs(c, seed):
    rnd = _rnd(seed)
    b, s, h, d = c["batch"], c["seq"], c["heads"], c["dim"]
    g = s // 4
    return dict(q=rnd(b, s, h, d).bfloat16(), kv=rnd(b, s, 1, d).bfloat16(), main=rnd(b, g, 1, d).bfloat16(),
                idx=_causal_lists(rnd, b, s, g, c["topk"]), sinks=rnd(h))


def _index_inputs(c, seed):
    rnd = _rnd(seed)
    b, s, hi, di = c["batch"], c["seq"], c["heads"], c["dim"]
    g = (c["start"] + s) // 4
    return dict(q=rnd(b, s, hi, di).bfloat16(), keys=rnd(b, g, di).bfloat16(), w=rnd(b, s, hi) * hi ** -0.5,
                pos=(c["start"] + torch.arange(s, device=DEV)).expand(b, s).contiguous())


def _reindex_inputs(c, seed):
    rnd = _rnd(seed)
    b, hi, g = c["batch"], c["heads"], c["groups"]
    return dict(q=[rnd(b, 1, hi, 128).bfloat16() for _ in range(2)], w=[rnd(b, 1, hi) * hi ** -0.5 for _ in range(2)],
                keys=[rnd(b, g, 128).bfloat16() for _ in range(2)], pos=_positions(b, 4 * g, seed).to(DEV).view(b, 1))


def _ingest_inputs(c, seed):
    rnd = _rnd(seed)
    b, t, d, r = c["batch"], c["seq"], 576, c["ratio"]
    n = t // r
    inv = 1.0 / (COMPRESS_THETA ** (torch.arange(0, 64, 2, device=DEV).float() / 64))
    ang = (r * torch.arange(n, device=DEV)).float()[None, :, None] * inv
    return dict(kv=rnd(b, t, d), gate=rnd(b, t, d), norm_w=(1 + 0.1 * rnd(d)).bfloat16(),
                cos=ang.cos().bfloat16().expand(b, -1, -1).contiguous(),
                sin=ang.sin().bfloat16().expand(b, -1, -1).contiguous(), keys=rnd(b, n, 128).bfloat16(),
                win=rnd(b, 128, d).bfloat16())


def _module_config(c):
    return owlet1.AttentionConfig(
        hidden_size=c["hidden"], num_attention_heads=c["heads"], head_dim=c["dim"], qk_rope_head_dim=c["rope"],
        q_lora_rank=c["q_rank"], o_groups=c["o_groups"], o_lora_rank=c["o_rank"], rope_theta=THETA,
        compress_rope_theta=COMPRESS_THETA, sliding_window=c["window"], compress_ratios=[4], kv_source_layer_ids=[0],
        index_source_layer_ids=[0], candidate_source_layer_id=-1, index_n_heads=c["index_heads"],
        index_head_dim=c["index_dim"], index_topk=c["topk"], rms_norm_eps=1e-20)


def _module_inputs(c, seed):
    """(weights by name, hidden states [B, S + steps, hidden]) in the model's type."""
    rnd = _rnd(seed)
    dt = getattr(torch, c["dtype"])
    h, d, hid, ql = c["heads"], c["dim"], c["hidden"], c["q_rank"]
    hi, di, og, orank = c["index_heads"], c["index_dim"], c["o_groups"], c["o_rank"]
    shapes = {"wq_a.weight": (ql, hid), "wq_b.weight": (h * d, ql), "wkv.weight": (d, hid),
              "wo_a.weight": (og * orank, h * d // og), "wo_b.weight": (hid, og * orank), "attn_sink": (h,),
              "compressor.wkv.weight": (d, hid), "compressor.wgate.weight": (d, hid),
              "indexer.wq_b.weight": (hi * di, ql), "indexer.weights_proj.weight": (hi, hid),
              "indexer.wk.weight": (di, d)}
    par = {k: (0.02 * rnd(*v)).to(dt) for k, v in sorted(shapes.items())}
    for k, n in (("q_norm", ql), ("kv_norm", d), ("compressor.norm", d), ("indexer.k_norm", di)):
        par[k + ".weight"] = torch.ones(n, device=DEV, dtype=dt)
    return par, rnd(c["batch"], c["seq"] + c["steps"], hid).to(dt)


# ---- prepare and run ----------------------------------------------------------------------

def prepare(case, seed):
    c = case
    if c["kind"] == "decode":
        x = _decode_inputs(c, seed)
        b, g, d = c["batch"], c["ctx"] // 4, 576
        cfg = DecodeConfig(batch=b, heads=c["heads"], index_heads=c["index_heads"], topk=c["topk"], max_groups=g,
                           index_format=c["fmt"], coarse_ratio=c["coarse"],
                           coarse_groups=c["ctx"] // c["coarse"] if c["coarse"] else 0, nsplit=c["nsplit"])
        cw = CompressorWeights(norm_weight=x["norm_w"], wk=x["wk"], k_norm_weight=x["k_norm"],
                               coarse_norm_weight=x.get("coarse_w"), rope_theta=COMPRESS_THETA)
        layer = SparseDecodeLayer(cfg, DEV, sinks=x["sinks"], kv_norm_weight=x["kv_w"], compressor=cw,
                                  max_position=4 * g)
        layer.fill_window(x["win"], cfg.window - 1)
        step = max(1, (1 << 26) // (b * d))
        for g0 in range(0, g, step):
            layer.append_groups(g0, x["main"][:, g0:g0 + step], x["keys"][:, g0:g0 + step])
        layer.set_carry(*x["carry"])
        comp = x["comp"]
        if c["coarse"]:
            layer.fill_coarse(x["coarse"])
            layer.set_carry(*x["c_carry"], coarse=True)
            comp = comp + x["c_comp"]
        layer.set_positions(x["pos"])
        layer.capture(x["q"], x["kv"], x["q_idx"], x["w"], rope="table", compress=comp)
        return dict(case=c, layer=layer)
    if c["kind"] == "attend":
        return dict(case=c, **_attend_inputs(c, seed))
    if c["kind"] == "index":
        x = _index_inputs(c, seed)
        keys = x.pop("keys")
        if c["fmt"] == "fp8":
            kc, ks = quant.quant_fp8_block(keys, c["dim"])
            x["keys"] = (kc, ks[..., 0].contiguous())
        else:
            x["keys"] = quant.quant_mxfp4(keys) if c["fmt"] == "mxfp4" else keys
        return dict(case=c, **x)
    if c["kind"] == "reindex":
        x = _reindex_inputs(c, seed)
        fp8 = c["fmt"] == "fp8"

        def packed(t, block):
            if not fp8:
                return quant.quant_mxfp4(t)
            codes, scales = quant.quant_fp8_block(t, block)
            return codes, scales[..., 0].contiguous()

        return dict(case=c, q=[packed(t, 128) for t in x["q"]], keys=[packed(t, 128) for t in x["keys"]], w=x["w"],
                    pos=x["pos"], lens=((x["pos"] + 1) // 4).unsqueeze(-1))
    if c["kind"] == "ingest":
        x = _ingest_inputs(c, seed)
        cfg = DecodeConfig(batch=c["batch"], max_groups=c["seq"] // c["ratio"], index_format=c["fmt"], ratio=c["ratio"],
                           nsplit=1)
        return dict(case=c, layer=SparseDecodeLayer(cfg, DEV), **x)
    par, x = _module_inputs(c, seed)
    with torch.device("meta"):
        mod = owlet1.DeepseekV41Attention(_module_config(c), 0)
    mod.load_state_dict(par, strict=True, assign=True)
    rot = owlet1.DeepseekV41RotaryEmbedding(mod.config).to(DEV)
    mod.indexer.rotary_emb, mod.compress_rotary = rot, rot  # buffers of their own, made on the GPU
    return dict(case=c, mod=mod.eval(), rot=rot, x=x)


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "decode":
        layer = s["layer"]
        out = layer.replay()
        got = dict(out=out, lse=layer.lse, win=layer.win, main=layer.main, carry_kv=layer.carry_kv,
                   carry_gate=layer.carry_gate)
        got["keys"] = (layer.k_codes, layer.k_scales) if c["fmt"] == "fp8" else (layer.k_packed, layer.k_e8m0)
        if c["coarse"]:
            got.update(coarse=layer.coarse)
        return got
    if c["kind"] == "attend":
        return csa2_attn.fwd(s["q"], s["kv"], s["main"], s["idx"], window=c["window"], compress_ratio=4,
                             sinks=s["sinks"])
    if c["kind"] == "index":
        kw = dict(compress_ratio=4, positions=s["pos"])
        if c["fmt"] == "fp8":
            qc, qs = quant.quant_fp8_block(s["q"], c["dim"])
            scores = indexer.scores_fp8(qc, qs[..., 0], s["w"], *s["keys"], **kw)
        elif c["fmt"] == "mxfp4":
            scores = indexer.scores_mxfp4(*quant.quant_mxfp4(s["q"]), s["w"], *s["keys"], **kw)
        else:
            scores = indexer.fwd(s["q"], s["keys"], s["w"], **kw)
        return scores, indexer.topk(scores, c["topk"])
    if c["kind"] == "reindex":
        fp8 = c["fmt"] == "fp8"
        dense = indexer.scores_fp8 if fp8 else indexer.scores_mxfp4
        gather = indexer.candidate_scores_fp8 if fp8 else indexer.candidate_scores_mxfp4
        kw = dict(compress_ratio=4, positions=s["pos"])
        scores = dense(*s["q"][0], s["w"][0], *s["keys"][0], **kw)
        blocks = indexer.candidate_block_list(scores, s["lens"], c["blocks"], 8)
        first = indexer.topk(scores, c["topk"])
        cand = gather(*s["q"][1], s["w"][1], *s["keys"][1], blocks, block_size=8, **kw)
        return scores, blocks, first, cand, indexer.candidate_topk(cand, blocks, 8, c["topk"])
    if c["kind"] == "ingest":
        layer = s["layer"]
        latent = mcache.compress(s["kv"], s["gate"], c["ratio"], s["norm_w"], EPS, torch.bfloat16)
        layer.append_groups(0, mcache.apply_rotary_pos_emb(latent, s["cos"], s["sin"]), s["keys"])
        layer.fill_window(s["win"], c["seq"] - 1)
        keys = (layer.k_codes, layer.k_scales) if c["fmt"] == "fp8" else (layer.k_packed, layer.k_e8m0)
        return latent, layer.main, keys, layer.win
    from transformers.cache_utils import Cache
    mod, rot, x, n = s["mod"], s["rot"], s["x"], c["seq"]
    cache = Cache(layers=[owlet1.DeepseekV41CSACache(mod.config)]) if c["steps"] else None
    outs = []
    with torch.no_grad():
        for a, e in [(0, n)] + [(n + i, n + i + 1) for i in range(c["steps"])]:
            pos = torch.arange(a, e, device=DEV).expand(c["batch"], -1)
            part = x[:, a:e]
            pe = {k: rot(part, pos, k) for k in ("main", "compress")}
            outs.append(mod(part, position_embeddings=pe, attention_mask=None, past_key_values=cache,
                            shared=owlet1.SharedState(), position_ids=pos)[0])
    if cache is None:
        return outs
    kept = cache.layers[0]
    return outs, [kept.compressed_kv["compressor"], kept.compressed_kv["indexer"], kept.keys]


# ---- what a pass cannot do without --------------------------------------------------------

KEY = {"fp8": 132, "mxfp4": 68, "bf16": 256}


def work(case):
    c = case
    if c["kind"] == "decode":
        b, h, d, hi, g = c["batch"], c["heads"], 576, c["index_heads"], c["ctx"] // 4
        vis = 0.75 * g  # rows lie in the second half of the context
        entries = 128 + min(c["topk"], vis) + (0.75 * (c["ctx"] // c["coarse"]) if c["coarse"] else 0)
        nbytes = b * (vis * KEY[c["fmt"]] + entries * 656 + 4 * h * d + 2 * hi * 128 + 18 * d)
        return dict(bytes=int(nbytes), flops=int(b * (4 * d * h * entries + 2 * hi * 128 * vis)))
    if c["kind"] == "attend":
        b, s, h, d = c["batch"], c["seq"], c["heads"], c["dim"]
        pairs = sum(min(t + 1, c["window"]) + min((t + 1) // 4, c["topk"]) for t in range(s))
        return dict(bytes=b * (4 * s * h * d + 2 * s * d + 2 * (s // 4) * d + 4 * s * min(c["topk"], s // 4) + 4 * s * h),
                    flops=4 * b * pairs * h * d)
    if c["kind"] == "index":
        b, s, hi, di, g = c["batch"], c["seq"], c["heads"], c["dim"], (c["start"] + c["seq"]) // 4
        pairs = sum((c["start"] + t + 1) // 4 for t in range(s))
        nbytes = b * (2 * s * hi * di + 4 * s * hi + g * KEY[c["fmt"]] * di // 128 + 4 * s * g + 4 * s * c["topk"])
        return dict(bytes=nbytes, flops=2 * b * pairs * hi * di)
    if c["kind"] == "reindex":
        b, hi, g, n = c["batch"], c["heads"], c["groups"], c["blocks"] * 8
        vis, cand = 0.75 * g, min(n, 0.75 * g)
        nbytes = b * ((vis + cand) * KEY[c["fmt"]] + 4 * (g + n) + 4 * c["blocks"] + 8 * c["topk"] + 4 * hi * 128)
        return dict(bytes=int(nbytes), flops=int(2 * b * hi * 128 * (vis + cand)))
    if c["kind"] == "ingest":
        b, t, d, n = c["batch"], c["seq"], 576, c["seq"] // c["ratio"]
        return dict(bytes=b * (8 * t * d + n * (2 * d + 656 + 256 + KEY[c["fmt"]]) + 128 * (2 * d + 656)),
                    flops=b * 6 * t * d)
    b, s, h, d, hid = c["batch"], c["seq"] + c["steps"], c["heads"], c["dim"], c["hidden"]
    hi, di = c["index_heads"], c["index_dim"]
    size = 4 if c["dtype"] == "float32" else 2
    weights = (c["q_rank"] * (hid + h * d + hi * di) + 3 * d * hid + c["o_rank"] * (h * d + c["o_groups"] * hid)
               + hi * hid + di * d)
    pairs = sum(min(t + 1, c["window"]) + min((t + 1) // 4, c["topk"]) for t in range(s))
    return dict(bytes=size * (weights * (1 + c["steps"]) + 2 * b * s * hid),
                flops=2 * b * s * weights + b * (4 * pairs * h * d + 2 * hi * di * sum((t + 1) // 4 for t in range(s))))


def tolerance(case):
    kind = case["kind"]
    if kind in ("decode", "attend"):  # bf16 outputs and probabilities: 0.0021 - 0.0026 off the exact ones
        return {"rel": 1e-2}
    if kind in ("index", "reindex"):
        # the matrix units' own sums: 1.5e-5 off the exact ones over e4m3 operands, 9e-8 over the
        # others; a near-tie at the boundary shifts the rest of a row's ascending list
        return {"rel": 6e-5 if case["fmt"] == "fp8" else 1e-6, "differ": 2e-2 if kind == "index" else 2e-1}
    if kind == "ingest":  # the pooling's order is fixed, the rest is elementwise
        return "exact"
    # a rounding that falls the other way flips a 4- or 8-bit code downstream: 0.034 off the exact
    # outputs in bf16, 0.0023 in fp32
    return {"rel": 6e-2 if case["dtype"] == "bfloat16" else 1e-2}


# ---- the same in 64 bits ------------------------------------------------------------------

def _bf(x):
    return x.to(torch.bfloat16).double()


def _pow2_ceil(x):
    m, e = torch.frexp(x)
    return torch.ldexp(torch.ones_like(x), torch.where(m == 0.5, e - 1, e))


def _e4m3(x):
    return x.float().to(torch.float8_e4m3fn).double()


def _q8(x, block):
    """_fake_quant_fp8_block: e4m3 codes times a power-of-two scale per block."""
    v = x.unflatten(-1, (-1, block))
    s = _pow2_ceil(v.abs().amax(-1, keepdim=True).clamp_min(1e-4) / 448)
    return (_e4m3((v / s).clamp(-448, 448)) * s).flatten(-2)


def _q4(x, block, e4m3=False):
    """_fake_quant_fp4_block: e2m1 codes times a power-of-two (or e4m3) scale per block."""
    v = x.unflatten(-1, (-1, block))
    a = v.abs().amax(-1, keepdim=True)
    s = _e4m3(a.clamp_min(6 * 2.0 ** -9) / 6) if e4m3 else _pow2_ceil(a.clamp_min(6 * 2.0 ** -126) / 6)
    u = (v / s).clamp(-6, 6)
    m = u.abs()
    step = torch.where(m < 2, 0.5, torch.where(m < 4, 1.0, 2.0)).to(m)
    return (torch.copysign(torch.round(m / step) * step, u) * s).flatten(-2)


def _latent(x):
    """What an FP8 latent entry holds of [..., 576]."""
    return torch.cat([_q8(x[..., :512], 128), _bf(x[..., 512:])], -1)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rms_bf(x, w, eps):
    return _bf(_bf(x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)) * w.double())


def _rope(x, cos, sin):
    n = 2 * cos.shape[-1]
    a, b = x[..., -n::2], x[..., x.shape[-1] - n + 1::2]
    r = torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)
    return torch.cat([x[..., :-n], r], -1)


def _table(pos, theta, dim, dtype):
    """cos / sin [..., dim/2] of integer positions as the model's tables hold them."""
    inv = (1.0 / (theta ** (torch.arange(0, dim, 2).float() / dim))).to(DEV)
    f = pos.to(DEV).float()[..., None] * inv
    return f.cos().to(dtype).double(), f.sin().to(dtype).double()


def _attention(q, entries, ok, sinks):
    """q [R, H, D] over entries [R, N, D] where ok [R, N]; (out [R, H, D], lse [R, H])."""
    s = torch.bmm(q, entries.transpose(1, 2).contiguous()) * q.shape[-1] ** -0.5
    s = s.masked_fill(~ok[:, None, :], float("-inf"))
    lse = torch.logsumexp(torch.cat([s, sinks.double().expand(q.shape[0], -1)[..., None]], -1), -1)
    return torch.bmm(torch.exp(s - lse[..., None]), entries), lse


def _relu_scores(q, w, k, vis):
    """q [R, Hi, Di], w [R, Hi], k [G, Di], vis [R] -> [R, G]."""
    out = torch.empty(q.shape[0], k.shape[0], dtype=torch.float64, device=DEV)
    kt = k.t().contiguous()
    step = max(1, (1 << 27) // (q.shape[1] * k.shape[0]))
    for r in range(0, q.shape[0], step):
        d = torch.matmul(q[r:r + step].flatten(0, 1), kt).relu_().unflatten(0, (-1, q.shape[1]))
        out[r:r + step] = (d * w[r:r + step, :, None].double()).sum(1) * q.shape[-1] ** -0.5
    return out.masked_fill_(torch.arange(k.shape[0], device=DEV) >= vis[:, None], float("-inf"))


def _exact_decode(c, seed):
    x = _decode_inputs(c, seed)
    b, g = c["batch"], c["ctx"] // 4
    pos = x["pos"].to(DEV)
    cos, sin = _table(pos, COMPRESS_THETA, 64, torch.bfloat16)
    rows = torch.arange(b, device=DEV)

    def emit(ratio, carry, comp, norm_w):
        slot = (pos % ratio)[:, None, None]
        at = torch.arange(ratio, device=DEV)[None, :, None]
        kv, gate = (torch.where(at == slot, new[:, None], torch.cat([old, new[:, None]], 1)).double()
                    for old, new in zip(carry, comp))
        lat = _rms_bf(_bf((kv * gate.softmax(1)).sum(1)), norm_w, EPS)
        gc, gs = _table(pos // ratio * ratio, COMPRESS_THETA, 64, torch.bfloat16)
        return lat, gc, gs, (pos + 1) % ratio == 0

    lat, gc, gs, done = emit(4, x["carry"], x["comp"], x["norm_w"])
    key = _rope(_rms_bf(_bf(lat @ x["wk"].double().t()), x["k_norm"], EPS), gc, gs)
    quantize = (lambda t: _q8(t, 128)) if c["fmt"] == "fp8" else (lambda t: _q4(t, 32))
    kq, entry = quantize(_bf(key)), _latent(_rope(lat, gc, gs))
    win = _latent(x["win"].double())
    win[rows, pos % 128] = _latent(_rope(_rms_bf(x["kv"].double(), x["kv_w"], EPS), cos, sin))
    qi = quantize(_bf(_rope(x["q_idx"].double(), cos[:, None], sin[:, None])))
    q = _rope(x["q"].double(), cos[:, None], sin[:, None])
    q = torch.cat([q[..., :512], _bf(q[..., 512:])], -1)
    vis, cur = (pos + 1) // 4, pos // 4
    outs, lses = [], []
    for i in range(b):
        k = quantize(x["keys"][i].double())
        if done[i]:
            k[cur[i]] = kq[i]
        sc = _relu_scores(qi[i:i + 1], x["w"][i:i + 1], k, vis[i:i + 1])[0]
        val, idx = sc.topk(min(c["topk"], g))
        idx = idx[val > float("-inf")]
        e = _latent(x["main"][i][idx].double())
        if done[i]:
            e[idx == cur[i]] = entry[i]
        parts = [win[i], e]
        if c["coarse"]:
            n = int((pos[i] + 1) // c["coarse"])
            co = _latent(x["coarse"][i, :n].double())
            if i == 0:
                clat, cc, cs, cdone = emit(c["coarse"], x["c_carry"], x["c_comp"], x["coarse_w"])
            if cdone[i]:
                co[n - 1] = _latent(_rope(clat[i], cc[i], cs[i]))
            parts.append(co)
        e = torch.cat(parts)[None]
        ok = torch.ones(1, e.shape[1], dtype=torch.bool, device=DEV)
        if pos[i] < 127:
            ok[0, :128] = torch.arange(128, device=DEV) <= pos[i]
        o, lse = _attention(q[i:i + 1], e, ok, x["sinks"])
        outs.append(o)
        lses.append(lse)
    out = _rope(torch.cat(outs), cos[:, None], -sin[:, None])
    return dict(out=out, lse=torch.cat(lses))


def _exact_prompt_attention(q, win, main, idx, window, sinks):
    """q [S, H, D], win [S, D], main [G, D], idx [S, k] (-1: none) in 64 bits, causal."""
    s, h, d = q.shape
    g = main.shape[0]
    out, lses = torch.empty(s, h, d, dtype=torch.float64, device=DEV), torch.empty(h, s, dtype=torch.float64, device=DEV)
    step = max(16, (1 << 27) // (h * (g + window + 256)))
    for r in range(0, s, step):
        e = min(s, r + step)
        w0 = max(0, r - window + 1)
        t, cols = torch.arange(r, e, device=DEV)[:, None], torch.arange(w0, e, device=DEV)[None]
        sel = torch.zeros(e - r, g + 1, dtype=torch.bool, device=DEV)
        sel.scatter_(1, idx[r:e].long().masked_fill(idx[r:e] < 0, g), True)
        ok = torch.cat([(cols <= t) & (cols > t - window), sel[:, :g]], 1)
        kv = torch.cat([win[w0:e], main])
        sc = (q[r:e].flatten(0, 1) @ kv.t().contiguous()).mul_(d ** -0.5).unflatten(0, (-1, h))
        sc = sc.masked_fill_(~ok[:, None, :], float("-inf"))
        lse = torch.logaddexp(torch.logsumexp(sc, -1), sinks.double()[None, :])
        out[r:e] = (sc.sub_(lse[..., None]).exp_().flatten(0, 1) @ kv).unflatten(0, (-1, h))
        lses[:, r:e] = lse.t()
    return out, lses


def _exact_module(c, seed):
    par, x = _module_inputs(c, seed)
    dt = x.dtype
    p = {k: v.double() for k, v in par.items()}
    x = x.double()
    b, s, _ = x.shape
    h, d, hi, di, eps = c["heads"], c["dim"], c["index_heads"], c["index_dim"], 1e-20
    pos, g = torch.arange(s), s // 4
    cos, sin = _table(pos, COMPRESS_THETA, c["rope"], dt)
    gcos, gsin = _table(4 * torch.arange(g), COMPRESS_THETA, c["rope"], dt)
    lin = lambda t, k: t @ p[k + ".weight"].t()  # noqa: E731
    qr = _rms(lin(x, "wq_a"), p["q_norm.weight"], eps)
    q = _rope(lin(qr, "wq_b").unflatten(-1, (h, d)), cos[:, None], sin[:, None])
    kv = _q8(_rope(_rms(lin(x, "wkv"), p["kv_norm.weight"], eps), cos, sin), 32)
    ck, cg = (lin(x[:, :4 * g], "compressor." + k).unflatten(1, (g, 4)) for k in ("wkv", "wgate"))
    lat = _rms((ck * cg.softmax(2)).sum(2), p["compressor.norm.weight"], eps)
    key = _q4(_rope(_rms(lin(lat, "indexer.wk"), p["indexer.k_norm.weight"], eps), gcos, gsin), 32)
    qi = _q4(_rope(lin(qr, "indexer.wq_b").unflatten(-1, (hi, di)), cos[:, None], sin[:, None]), 32)
    w = lin(x, "indexer.weights_proj") * hi ** -0.5
    comp = _q4(_rope(lat, gcos, gsin), 16, e4m3=True)
    vis = ((pos + 1) // 4).to(DEV)
    outs = []
    for i in range(b):
        val, idx = _relu_scores(qi[i], w[i], key[i], vis).topk(min(c["topk"], g), -1)
        o, _ = _exact_prompt_attention(q[i], kv[i], comp[i], idx.masked_fill(val == float("-inf"), -1), c["window"],
                                       p["attn_sink"])
        o = _rope(o, cos[:, None], -sin[:, None]).reshape(s, c["o_groups"], -1)
        wa = p["wo_a.weight"].unflatten(0, (c["o_groups"], -1))
        o = torch.stack([o[:, j] @ wa[j].t() for j in range(c["o_groups"])], 1)
        outs.append(lin(o.flatten(1), "wo_b"))
    out = torch.stack(outs)
    n = c["seq"]
    outs = [out[:, :n]] + [out[:, n + i:n + i + 1] for i in range(c["steps"])]
    return (outs, [None, None, None]) if c["steps"] else outs


def exact(case, seed):
    c = case
    if c["kind"] == "decode":
        got = _exact_decode(c, seed)
        got.update(win=None, main=None, carry_kv=None, carry_gate=None, keys=(None, None))
        if c["coarse"]:
            got.update(coarse=None)
        return got
    if c["kind"] == "attend":
        x = _attend_inputs(c, seed)
        pairs = [_exact_prompt_attention(x["q"][i].double(), x["kv"][i, :, 0].double(), x["main"][i, :, 0].double(),
                                         x["idx"][i], c["window"], x["sinks"]) for i in range(c["batch"])]
        return torch.stack([o for o, _ in pairs]), torch.stack([v for _, v in pairs])
    quantize = (lambda t: _q8(t, 128)) if c.get("fmt") == "fp8" else (lambda t: _q4(t, 32))
    if c["kind"] == "index":
        x = _index_inputs(c, seed)
        f = (lambda t: t) if c["fmt"] == "bf16" else quantize
        q, k = f(x["q"].double()), f(x["keys"].double())
        return torch.stack([_relu_scores(q[i], x["w"][i], k[i], (x["pos"][i] + 1) // 4)
                            for i in range(c["batch"])]), None
    if c["kind"] == "reindex":
        x = _reindex_inputs(c, seed)
        vis = (x["pos"][:, 0] + 1) // 4
        sc = torch.stack([_relu_scores(quantize(x["q"][0][i].double()), x["w"][0][i], quantize(x["keys"][0][i].double()),
                                       vis[i:i + 1]) for i in range(c["batch"])])
        return sc, None, None, None, None
    if c["kind"] == "ingest":
        x = _ingest_inputs(c, seed)
        n, r = c["seq"] // c["ratio"], c["ratio"]
        kv, gate = (x[k][:, :n * r].double().unflatten(1, (n, r)) for k in ("kv", "gate"))
        lat = _rms((kv * gate.softmax(2)).sum(2), x["norm_w"].double(), EPS)
        return lat, None, (None, None), None
    return _exact_module(c, seed)
