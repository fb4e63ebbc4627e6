"""Timed workloads of the fused DeepSeek-Sparse-Attention path, through its public entry points.

Five kinds of work, over the sizes the path meets in use:

  decode   one step of a serving loop: a few tokens for each of several sequences, against caches of latent keys and of
           quantised indexer keys that the server keeps (absorbed query -> indexer -> top-k -> sparse attention ->
           value projection)
  prefill  one chunk of a prompt behind the part of it that is cached already, forward only
  train    the attention module of a training step, forward and backward, with the indexer's KL loss
  csa      the same over a sliding window plus compressed keys, with attention sinks, forward and backward
  rope     the rotary kernels around the attention, forward and backward

A case is a dict of plain values.  Inputs are standard normal as in the benchmark and the tests (scores of the selected
keys then spread over a few units), lengths of sequences and documents are uneven and follow from the case alone.
"""
import math
from types import SimpleNamespace

import torch

from loongforge_amd import dsa_fused, ops
from loongforge_amd import dsa_fused_kernels as K
from loongforge_amd.csa_kernels import CSAIndexerKernel, get_window_topk_idxs
from loongforge_amd.megatron_compat import AttnMaskType, ModuleSpec, PackedSeqParams

BF = torch.bfloat16
D_QK, D_V, D_ROPE, D_NOPE = 576, 512, 64, 128
SCALE = 192.0 ** -0.5
HIDDEN, Q_LORA = 1024, 512          # widths of the indexer's projections in the training module
WINDOW = 128                        # sliding window of the compressed-key attention


def listed():
    return [
        # one user, one token, a short conversation: every launch shows
        dict(name="decode_one", kind="decode", seqs=1, draft=1, context=4096, heads=128, index_heads=64, topk=2048),
        # a serving batch, conversations of uneven length, all heads on one GPU
        dict(name="decode_ragged_48", kind="decode", seqs=48, draft=1, context=7001, heads=128, index_heads=64, topk=2048),
        # a large batch of short conversations on a 32-head shard, four tokens each (one plus three drafted ones)
        dict(name="decode_draft_shard", kind="decode", seqs=50, draft=4, context=2500, heads=32, index_heads=32, topk=512),
        # a user's follow-up question behind a long cached document
        dict(name="extend_61", kind="prefill", tokens=61, cached=20000, heads=64, index_heads=64, topk=1024),
        # an ordinary prompt chunk
        dict(name="prefill_1500", kind="prefill", tokens=1500, cached=6692, heads=128, index_heads=64, topk=2048),
        # a whole prompt of 8k tokens
        dict(name="prefill_8192", kind="prefill", tokens=8192, cached=0, heads=128, index_heads=64, topk=2048),
        # the tiny configuration: 16 heads, indexer 4 x 64, top-k 256
        dict(name="train_tiny", kind="train", tokens=1024, docs=1, heads=16, index_heads=4, index_dim=64, topk=256),
        # a small packed batch with odd lengths
        dict(name="train_packed_2077", kind="train", tokens=2077, docs=3, heads=64, index_heads=32, index_dim=128, topk=512),
        # the benchmark's sequence
        dict(name="train_8192", kind="train", tokens=8192, docs=1, heads=128, index_heads=64, index_dim=128, topk=2048),
        # the largest configuration: 32k packed tokens in four documents
        dict(name="train_packed_32768", kind="train", tokens=32768, docs=4, heads=128, index_heads=64, index_dim=128, topk=2048),
        # compressed-key attention: window 128 + 512 compressed keys, ratio 4
        dict(name="csa_3072", kind="csa", tokens=3072, ratio=4, heads=64, index_heads=64, topk=512),
        # rotary kernels of the reference's call sequence
        dict(name="rope_4096", kind="rope", tokens=4096, heads=128, interleaved=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "train", "train", "csa", "rope"])
    heads = rng.choice([32, 64, 128, 128])
    topk = rng.choice([256, 512, 1024, 2048, 2048])
    if kind == "decode":
        seqs = _log(rng, 1, 200)
        context = _log(rng, 300, min(32768, 500000 // seqs))
        return dict(kind=kind, seqs=seqs, draft=rng.choice([1, 1, 2, 4]), context=context, heads=heads,
                    index_heads=rng.choice([32, 64]), topk=topk)
    if kind == "prefill":
        tokens = _log(rng, 20, 8192)
        return dict(kind=kind, tokens=tokens, cached=rng.choice([0, _log(rng, 100, 24000)]), heads=heads,
                    index_heads=rng.choice([32, 64]), topk=topk)
    if kind == "train":
        return dict(kind=kind, tokens=_log(rng, 300, 12000), docs=rng.choice([1, 1, 2, 3, 5]),
                    heads=rng.choice([16, 32, 64, 128, 128]), index_heads=rng.choice([32, 64]), index_dim=128, topk=topk)
    if kind == "csa":
        return dict(kind=kind, tokens=_log(rng, 500, 8192), ratio=4, heads=heads, index_heads=64, topk=rng.choice([256, 512]))
    return dict(kind=kind, tokens=_log(rng, 16, 8192), heads=heads, interleaved=rng.random() < 0.5)


# ---------------------------------------------------------------------------------------------------
# lengths
# ---------------------------------------------------------------------------------------------------
def _lengths(total, parts):
    """`parts` uneven lengths that sum to `total` (weights 0.4 .. 1.6, spread by the golden ratio)."""
    w = [0.4 + 1.2 * ((0.5 + 0.6180339887 * i) % 1.0) for i in range(parts)]
    edges, run = [0], 0.0
    for x in w:
        run += x
        edges.append(int(round(total * run / sum(w))))
    edges[-1] = total
    return [b - a for a, b in zip(edges, edges[1:])]


def _contexts(case):
    """Tokens in each sequence's cache, the step's own among them."""
    return [max(n, case["draft"]) for n in _lengths(case["seqs"] * case["context"], case["seqs"])]


def _visible(first, last, most=None):
    """Sum over i in first .. last of min(i, most)."""
    tri = lambda n: n * (n + 1) // 2                                             # noqa: E731
    if most is None or last <= most:
        return tri(last) - tri(first - 1)
    low = tri(most) - tri(first - 1) if first <= most else 0
    return low + most * (last - max(most, first - 1))


# ---------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------
def _tables(positions, dev):
    freq = 10000.0 ** (-torch.arange(0, D_ROPE, 2, device=dev, dtype=torch.float32) / D_ROPE)
    ang = positions.float()[:, None] * freq
    ang = torch.cat([ang, ang], -1)
    return ang.cos().to(BF).view(-1, 1, 1, D_ROPE).contiguous(), ang.sin().to(BF).view(-1, 1, 1, D_ROPE).contiguous()


def _config(**kw):
    base = dict(qk_pos_emb_head_dim=D_ROPE, v_head_dim=128, kv_lora_rank=D_V, apply_rope_fusion=True, kv_channels=192,
                num_layers=1, hidden_size=HIDDEN, q_lora_rank=Q_LORA, dsa_indexer_loss_coeff=1.0, rope_type="rope",
                rotary_percent=1.0, rotary_base=10000, init_method=None, layernorm_epsilon=1e-5,
                dsa_indexer_rotate_activation=True, enable_chunkpipe=False)
    base.update(kw)
    return SimpleNamespace(**base)


class _Linear(torch.nn.Module):
    """A projection as the trainer hands it to the module: bf16 weight, returns (output, bias)."""

    def __init__(self, n_in, n_out, **_):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.empty(n_out, n_in, dtype=BF))

    def forward(self, x):
        return torch.nn.functional.linear(x, self.weight), None


class _Norm(torch.nn.LayerNorm):
    def __init__(self, config=None, hidden_size=None, eps=1e-5):
        super().__init__(hidden_size, eps=eps)

    def forward(self, x):
        return super().forward(x.float()).to(x.dtype)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    rnd = lambda *shape, std=1.0: torch.randn(*shape, generator=g, device=dev, dtype=BF).mul_(std)    # noqa: E731
    return _PREPARE[case["kind"]](case, rnd, dev)


def _prepare_decode(case, rnd, dev):
    n, h, hi = case["draft"], case["heads"], case["index_heads"]
    ctx = torch.tensor(_contexts(case), dtype=torch.int64)
    start = torch.cumsum(ctx, 0) - ctx
    rows = case["seqs"] * n
    pos = (ctx[:, None] - n + torch.arange(n)[None]).reshape(-1)                 # position of each token in its sequence
    first = start.repeat_interleave(n)
    cos, sin = _tables(pos.to(dev), dev)
    k8, k_scale = ops.rotate_quant_e4m3(rnd(int(ctx.sum()), 128))
    return dict(kind="decode", topk=case["topk"], q_up=rnd(rows, h, D_NOPE + D_ROPE), w_uk_t=rnd(h, D_V, D_NOPE, std=D_NOPE ** -0.5),
                w_uv=rnd(h, 128, D_V, std=D_V ** -0.5), cos=cos, sin=sin, index_q=rnd(rows, hi, 128), weights=rnd(rows, hi, std=0.1).float(),
                kv=rnd(int(ctx.sum()), D_QK), k8=k8, k_scale=k_scale, window_start=first.int().to(dev),
                window_end=(first + pos + 1).int().to(dev), all_keys=int(ctx.sum()))


def _prepare_prefill(case, rnd, dev):
    s, c, h, hi = case["tokens"], case["cached"], case["heads"], case["index_heads"]
    cos, sin = _tables(torch.arange(c, c + s, device=dev), dev)
    return dict(kind="prefill", topk=case["topk"], cached=c, q_up=rnd(s, 1, h, D_NOPE + D_ROPE),
                w_uk_t=rnd(h, D_V, D_NOPE, std=D_NOPE ** -0.5), w_uv=rnd(h, 128, D_V, std=D_V ** -0.5), cos=cos, sin=sin,
                latent=rnd(s, 1, 1, D_V), k_pe=rnd(s, 1, 1, D_ROPE), index_q=rnd(s, hi, 128), index_k=rnd(c + s, 128),
                weights=rnd(s, hi, std=0.1).float(), kv=rnd(c + s, D_QK), indexer=K.DSAIndexerKernel(),
                attention=K.DSADotProductAttention(_config(num_attention_heads=h), softmax_scale=SCALE))


def _prepare_train(case, rnd, dev):
    s, h = case["tokens"], case["heads"]
    cfg = _config(num_attention_heads=h, dsa_indexer_n_heads=case["index_heads"], dsa_indexer_head_dim=case["index_dim"],
                  dsa_indexer_topk=case["topk"], apply_rope_fusion=case["index_dim"] == 128)
    sub = dsa_fused.DSAttentionFusedSubmodules(indexer=ModuleSpec(
        module=dsa_fused.DSAIndexerFused,
        submodules=dsa_fused.DSAIndexerFusedSubmodules(linear_wq_b=_Linear, linear_wk=_Linear, k_norm=_Norm,
                                                       linear_weights_proj=_Linear)))
    mod = dsa_fused.DSAttentionFused(cfg, sub, layer_number=1, attn_mask_type=AttnMaskType.causal, attention_type="self",
                                     k_channels=192).to(dev).train()
    with torch.no_grad():
        for p in mod.parameters():
            if p.ndim == 2:
                p.copy_(rnd(*p.shape, std=p.shape[1] ** -0.5))
    packed, lead = None, (s, 1)
    if case["docs"] > 1:
        lens = _lengths(s, case["docs"])
        cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device=dev)
        packed = PackedSeqParams(qkv_format="thd", cu_seqlens_q=cu, cu_seqlens_kv=cu, max_seqlen_q=max(lens), max_seqlen_kv=max(lens))
        lead = (s,)
    return dict(kind="train", module=mod, packed=packed, query=rnd(*lead, h, D_QK).requires_grad_(True),
                key=rnd(*lead, D_QK).requires_grad_(True), x=rnd(*lead, HIDDEN), qr=rnd(*lead, Q_LORA),
                dout=rnd(*((s,) if packed is not None else (1, s)), h, D_V), params=list(mod.parameters()))


def _prepare_csa(case, rnd, dev):
    s, h, hi = case["tokens"], case["heads"], case["index_heads"]
    n_c = s // case["ratio"]
    return dict(kind="csa", topk=case["topk"], tokens=s, query=rnd(s, 1, h, D_QK).requires_grad_(True),
                kv=rnd(s + n_c, 1, D_QK).requires_grad_(True), index_q=rnd(s, 1, hi, 128).requires_grad_(True),
                index_k=rnd(n_c, 1, 128).requires_grad_(True), weights=rnd(s, 1, hi, std=0.1).requires_grad_(True),
                sink=rnd(h).float(), dout=rnd(1, s, h, D_V), dloss=torch.full((), 1.0 / s, device=dev),
                indexer=CSAIndexerKernel(case["ratio"]),
                attention=K.DSADotProductAttention(_config(num_attention_heads=h), softmax_scale=SCALE))


def _prepare_rope(case, rnd, dev):
    s, h = case["tokens"], case["heads"]
    cos, sin = _tables(torch.arange(s, device=dev), dev)
    return dict(kind="rope", interleaved=case["interleaved"], content=rnd(h, s, D_V).requires_grad_(True),
                q_pe=rnd(s, 1, h, D_ROPE).requires_grad_(True), latent=rnd(s, 1, 1, D_V).requires_grad_(True),
                k_pe=rnd(s, 1, 1, D_ROPE).requires_grad_(True), cos=cos, sin=sin, d_query=rnd(s, 1, h, D_QK),
                d_key=rnd(s, 1, 1, D_QK))


_PREPARE = dict(decode=_prepare_decode, prefill=_prepare_prefill, train=_prepare_train, csa=_prepare_csa, rope=_prepare_rope)


# ---------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------
def run(state):
    return _RUN[state["kind"]](state)


@torch.no_grad()
def _run_decode(t):
    query = K.fused_absorb_rope_query(t["q_up"], t["w_uk_t"], t["cos"], t["sin"])
    q8, _, w = ops.quant_rowwise_e4m3_weights(t["index_q"], t["weights"], 128 ** -0.5, rotate=True)
    scores, ids = ops.indexer_topk(q8, w, t["k8"], t["k_scale"], t["window_start"], t["window_end"], t["topk"])
    # the windows have made the ids causal already: a start beyond the last key switches the position test off
    out, lse, _ = ops.sparse_mla_fwd(query, t["kv"], ids, t["all_keys"], SCALE)
    return dict(scores=scores, ids=ids, lse=lse, y=K.absorb_attention_output(out, t["w_uv"]))


@torch.no_grad()
def _run_prefill(t):
    s, c = t["q_up"].shape[0], t["cached"]
    query = K.fused_absorb_rope_query(t["q_up"], t["w_uk_t"], t["cos"], t["sin"])
    key = K.fused_apply_mla_rope_for_absorb_kv(t["latent"], t["k_pe"], t["cos"], t["sin"], D_ROPE, D_V)
    t["kv"][c:] = key.view(s, D_QK)                                              # the chunk joins the cache
    scores, ids = t["indexer"](t["index_q"], t["index_k"], t["weights"], t["topk"], c, None, rotate=True)
    out = t["attention"](query, t["kv"].unsqueeze(1), ids.unsqueeze(0), c)
    return dict(scores=scores, ids=ids, y=K.absorb_attention_output(out, t["w_uv"]))


def _run_train(t):
    out = t["module"](t["query"], t["key"], None, None, x=t["x"], qr=t["qr"], attn_mask_type=AttnMaskType.causal,
                      packed_seq_params=t["packed"])
    grads = torch.autograd.grad(out, [t["query"], t["key"]] + t["params"], t["dout"])
    return dict(out=out.detach(), grads=list(grads))


def _run_csa(t):
    s = t["tokens"]
    scores, ids = t["indexer"](t["index_q"], t["index_k"], t["weights"], t["topk"])
    window = get_window_topk_idxs(WINDOW, 1, s, ids.device)[0].int()
    ids = torch.cat([window, torch.where(ids >= 0, ids + s, ids)], -1)
    out, p_out = t["attention"](t["query"], t["kv"], ids.unsqueeze(0), t["kv"].shape[0], attn_sink=t["sink"],
                                window_size=WINDOW, return_p_out=True)
    target = K.triton_attn_dist(p_out, SCALE)[:, :scores.shape[1]]
    loss = ops.indexer_kl_loss(scores, target)
    grads = torch.autograd.grad([out, loss], [t["query"], t["kv"], t["index_q"], t["index_k"], t["weights"]],
                                [t["dout"], t["dloss"]])
    return dict(out=out.detach(), loss=loss.detach(), grads=list(grads))


def _run_rope(t):
    query = K.fused_rope_permute_cat(t["content"], t["q_pe"], t["cos"], t["sin"], rotary_interleaved=t["interleaved"])
    key = K.fused_apply_mla_rope_for_absorb_kv(t["latent"], t["k_pe"], t["cos"], t["sin"], D_ROPE, D_V,
                                               rotary_interleaved=t["interleaved"])
    grads = torch.autograd.grad([query, key], [t["content"], t["q_pe"], t["latent"], t["k_pe"]], [t["d_query"], t["d_key"]])
    return dict(query=query.detach(), key=key.detach(), grads=list(grads))


_RUN = dict(decode=_run_decode, prefill=_run_prefill, train=_run_train, csa=_run_csa, rope=_run_rope)


# ---------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------
def _indexer_work(rows, keys, vis, hi, di, topk, key_bytes):
    return rows * hi * (2 * di + 4) + keys * key_bytes + rows * topk * 8, 2.0 * hi * di * vis


def work(case):
    kind, h = case["kind"], case["heads"]
    pair_fwd, pair_bwd = 2.0 * h * (D_QK + D_V), 2.0 * h * (3 * D_QK + 2 * D_V)
    if kind == "decode":
        n, k = case["draft"], case["topk"]
        rows, keys = case["seqs"] * n, 0
        vis = pairs = used = 0
        for c in _contexts(case):
            keys += c
            vis += _visible(c - n + 1, c)
            pairs += _visible(c - n + 1, c, k)
            used += min(c, k)                                                    # rows that one of its tokens needs at least
        b, f = _indexer_work(rows, keys, vis, case["index_heads"], 128, k, 132)
        b += 2 * 2 * h * D_V * D_NOPE + rows * h * (2 * (D_NOPE + D_ROPE) + 4 + 2 * 128) + used * 2 * D_QK
        return dict(bytes=b, flops=f + pair_fwd * pairs + 2 * 2.0 * rows * h * D_NOPE * D_V)
    if kind == "prefill":
        s, c, k = case["tokens"], case["cached"], case["topk"]
        vis, pairs = _visible(c + 1, c + s), _visible(c + 1, c + s, k)
        b, f = _indexer_work(s, c + s, vis, case["index_heads"], 128, k, 256)
        b += 2 * 2 * h * D_V * D_NOPE + s * h * (2 * (D_NOPE + D_ROPE) + 2 * 128) + (c + 2 * s) * 2 * D_QK
        return dict(bytes=b, flops=f + pair_fwd * pairs + 2 * 2.0 * s * h * D_NOPE * D_V)
    if kind == "rope":
        s = case["tokens"]
        return dict(bytes=2 * 2 * 2 * s * (h + 1) * D_QK, flops=2 * 3.0 * s * (h + 1) * D_ROPE)
    s, k, hi = case["tokens"], case["topk"], case["index_heads"]
    if kind == "csa":
        r, n_c = case["ratio"], s // case["ratio"]
        vis = sum(max((i + 1) // r, 1) for i in range(s))
        sel = sum(min(max((i + 1) // r, 1), k) for i in range(s))
        pairs = sel + _visible(1, s, WINDOW)
        di, keys, kv = 128, n_c, s + n_c
        proj = 0.0
        b = 2 * s * hi * 2 * di + 2 * n_c * 2 * di + 2 * s * hi * 2                # indexer inputs and their gradients
    else:
        lens = _lengths(s, case["docs"])
        vis = sum(_visible(1, n) for n in lens)
        sel = pairs = sum(_visible(1, n, k) for n in lens)
        di, kv = case["index_dim"], s
        proj = 2 * 2.0 * s * (Q_LORA * hi * di + HIDDEN * (di + hi))             # projections and their weight gradients
        b = 2 * s * (HIDDEN + Q_LORA) + 2 * 2 * (Q_LORA * hi * di + HIDDEN * (di + hi))
    b += 2 * kv * 2 * D_QK + 2 * s * h * 2 * (D_QK + D_V)                          # q, kv, dout in; out, dq, dkv out
    f = 2.0 * hi * di * (vis + 3 * sel) + (pair_fwd + pair_bwd) * pairs + proj
    return dict(bytes=b, flops=f)


def tolerance(case):
    if case["kind"] == "rope":
        return dict(rel=4e-3)                       # one rounding to bf16
    # bf16 results; neighbouring scores of the sorted selection that agree to the last bits may trade places
    return dict(rel=1e-2, differ=2e-3)
