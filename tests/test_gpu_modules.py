"""GPU parity of the module-level drop-in interface: DSADotProductAttention layouts, the
sparse_mla_bwd_interface function and the fused attention module with the KL indexer loss."""
from types import SimpleNamespace

import pytest
import torch

from oracle import dsa_oracle as O
from tests.gpu_util import assert_close, assert_mla_grads

pytestmark = pytest.mark.gpu


def _cfg(**kw):
    base = dict(qk_pos_emb_head_dim=64, v_head_dim=128, kv_lora_rank=512, apply_rope_fusion=False,
                num_attention_heads=128, kv_channels=192, num_layers=2)
    base.update(kw)
    return SimpleNamespace(**base)


def test_dot_product_attention_layouts_and_autograd(gpu):
    from loongforge_amd.dsa_fused_kernels import DSADotProductAttention
    from loongforge_amd.megatron_compat import AttnMaskType, PackedSeqParams

    inp = O.make_mla_inputs(150, 128, 100, seed=1)               # top-k 100 is padded to 128 inside
    attn = DSADotProductAttention(_cfg(), softmax_scale=inp.sm_scale)
    q = inp.q.to(gpu).requires_grad_(True)
    kv = inp.kv.to(gpu).requires_grad_(True)
    ids = inp.idx.to(gpu)
    # sbhd: query [sq, b=1, h, d], kv [skv, b=1, d], ids [b=1, sq, topk]
    out, p_out = attn(q.unsqueeze(1), kv.unsqueeze(1), ids.unsqueeze(0), 0, AttnMaskType.causal, return_p_out=True)
    assert out.shape == (1, 150, 128, 512) and p_out.shape == (150, 128, 128)
    ro, _, rp = O.sparse_mla_fwd(inp.q, inp.kv, inp.idx, 0, inp.sm_scale, 512)
    assert_close(out[0], ro, "out")
    assert torch.isinf(p_out[:, :, 100:]).all()
    out.backward(inp.dout.to(gpu).unsqueeze(0))
    assert_mla_grads(q.grad, kv.grad, inp.q, inp.kv, inp.idx, inp.dout, 0, inp.sm_scale, out=out[0])
    # thd: query [t, h, d], kv [t, d], ids handed as [1, t, topk]
    psp = PackedSeqParams(qkv_format="thd")
    out2 = attn(inp.q.to(gpu), inp.kv.to(gpu), ids.unsqueeze(0), 0, None, packed_seq_params=psp)
    assert out2.shape == (150, 128, 512)
    assert torch.equal(out2, out[0].detach())
    with pytest.raises(AssertionError):
        attn(q.unsqueeze(1), kv.unsqueeze(1), ids.unsqueeze(0), 0, AttnMaskType.no_mask)
    with pytest.raises(NotImplementedError):
        attn(q.unsqueeze(1), kv.unsqueeze(1), ids.unsqueeze(0), 0, None, window_size=4, return_p_out=True)
    with pytest.raises(ValueError):
        attn(q.unsqueeze(1), kv.unsqueeze(1), ids.unsqueeze(0), 0, None, window_size=64)
    # window_size: p_out leaves out the leading (window) slots, the output is unchanged
    out4, p4 = attn(q.unsqueeze(1), kv.unsqueeze(1), ids.unsqueeze(0), 0, None, window_size=64, return_p_out=True)
    assert p4.shape == (150, 128, 64) and torch.equal(p4, p_out[:, :, 64:]) and torch.equal(out4, out)
    # topk_length keeps a prefix of each query's slots; attn_sink ([h] or a divisor of it) joins the denominator
    tl = torch.randint(0, 101, (150,), generator=torch.Generator().manual_seed(4), dtype=torch.int32)
    sink = torch.linspace(-2, 2, 64)
    q.grad = kv.grad = None
    out3 = attn(q.unsqueeze(1), kv.unsqueeze(1), ids.unsqueeze(0), 0, None, topk_length=tl.to(gpu), attn_sink=sink.to(gpu))
    cut = torch.where(torch.arange(inp.idx.shape[1])[None, :] < tl[:, None], inp.idx, torch.full_like(inp.idx, -1))
    sink_h = sink.repeat_interleave(2)
    ro3, _, _ = O.sparse_mla_fwd(inp.q, inp.kv, cut, 0, inp.sm_scale, 512, attn_sink=sink_h)
    assert_close(out3[0], ro3, "out with topk_length and sink")
    out3.backward(inp.dout.to(gpu).unsqueeze(0))
    from loongforge_amd import ops
    cut_pad = torch.nn.functional.pad(cut, (0, 28), value=-1).to(gpu)          # the module pads top-k 100 to 128
    _, lse3, _ = ops.sparse_mla_fwd(q.detach(), kv.detach(), cut_pad, 0, inp.sm_scale, attn_sink=sink_h.to(gpu))
    assert_mla_grads(q.grad, kv.grad, inp.q, inp.kv, cut, inp.dout, 0, inp.sm_scale, "topk_length and sink:", attn_sink=sink_h,
                     out=out3[0], lse=lse3)


def test_sparse_mla_bwd_interface_signature(gpu):
    from loongforge_amd import ops
    from loongforge_amd.sparse_mla_bwd import sparse_mla_bwd_interface

    inp = O.make_mla_inputs(128, 128, 64, seed=2, q_start=30, skv=200)
    q, kv, idx, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, 30, inp.sm_scale)
    offsets = torch.tensor([0, 128], dtype=torch.int32, device=gpu)
    dq, dkv = sparse_mla_bwd_interface(q, kv.unsqueeze(1), out, do, idx.unsqueeze(1), lse, offsets, chunk_offset=30,
                                       sm_scale=inp.sm_scale)
    assert dq.shape == q.shape and dkv.shape == (200, 1, 576)
    assert_mla_grads(dq, dkv[:, 0], inp.q, inp.kv, inp.idx, inp.dout, 30, inp.sm_scale, out=out, lse=lse)


class _Linear(torch.nn.Module):
    """Column-parallel-linear stand-in: returns (output, bias) like the Megatron layers."""

    def __init__(self, n_in, n_out, **_):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.empty(n_out, n_in))

    def forward(self, x):
        return torch.nn.functional.linear(x, self.weight.to(x.dtype)), None


class _Norm(torch.nn.LayerNorm):
    def __init__(self, config=None, hidden_size=None, eps=1e-5):
        super().__init__(hidden_size, eps=eps)

    def forward(self, x):
        return super().forward(x.float()).to(x.dtype)


def test_fused_attention_module_matches_oracle_pipeline(gpu):
    """The reference's tiny configuration (16 query heads, indexer 4 x 64, top-k 256, uniform head
    weights) through DSAttentionFused: indexer -> top-k -> sparse attention -> KL loss -> backward."""
    from loongforge_amd import dsa_fused
    from loongforge_amd.megatron_compat import AttnMaskType, ModuleSpec

    S, H, Hi, Di, K, hid, qlr = 512, 16, 4, 64, 256, 96, 48
    cfg = _cfg(num_attention_heads=H, hidden_size=hid, q_lora_rank=qlr, dsa_indexer_n_heads=Hi,
               dsa_indexer_head_dim=Di, dsa_indexer_topk=K, dsa_indexer_loss_coeff=1.0, rope_type="rope",
               rotary_percent=1.0, rotary_base=10000, init_method=None, layernorm_epsilon=1e-5,
               dsa_indexer_rotate_activation=True, enable_chunkpipe=False)
    sub = dsa_fused.DSAttentionFusedSubmodules(indexer=ModuleSpec(
        module=dsa_fused.DSAIndexerFused,
        submodules=dsa_fused.DSAIndexerFusedSubmodules(linear_wq_b=_Linear, linear_wk=_Linear, k_norm=_Norm,
                                                       linear_weights_proj=_Linear)))
    torch.manual_seed(0)
    mod = dsa_fused.DSAttentionFused(cfg, sub, layer_number=1, attn_mask_type=AttnMaskType.causal,
                                     attention_type="self", k_channels=192)
    for p in mod.parameters():
        if p.ndim == 2:
            torch.nn.init.normal_(p, std=p.shape[1] ** -0.5)
    mod = mod.to(gpu).train()
    g = torch.Generator().manual_seed(0)
    query = torch.randn(S, 1, H, 576, generator=g).to(torch.bfloat16).to(gpu).requires_grad_(True)
    key = torch.randn(S, 1, 576, generator=g).to(torch.bfloat16).to(gpu).requires_grad_(True)
    x = torch.randn(S, 1, hid, generator=g).to(torch.bfloat16).to(gpu)
    qr = torch.randn(S, 1, qlr, generator=g).to(torch.bfloat16).to(gpu)
    out = mod(query, key, None, None, x=x, qr=qr, attn_mask_type=AttnMaskType.causal)
    assert out.shape == (1, S, H, 512)
    loss_logged = dsa_fused.DSAIndexerLossLoggingHelperFused.tracker[1]

    # oracle pipeline on the module's own indexer output (the selection itself is checked against
    # the oracle in test_gpu_indexer.py; re-using the ids keeps this test free of boundary noise)
    with torch.no_grad():
        sc_gpu, ids_gpu = mod.indexer(x, qr)
    ids_c, sc_c = ids_gpu.cpu(), sc_gpu.cpu()
    ro, _, rp = O.sparse_mla_fwd(query.detach().cpu()[:, 0], key.detach().cpu()[:, 0], ids_c, 0, mod.softmax_scale, 512)
    target = O.attn_dist(rp[:, :H], mod.softmax_scale)
    ref = dict(out=ro, idx=ids_c, loss=O.indexer_kl_loss(sc_c, target, 1.0, S))
    assert_close(out[0], ref["out"], "out")
    assert abs(loss_logged.item() - ref["loss"].item()) <= 2e-2 * abs(ref["loss"].item()) + 1e-3

    dout = torch.randn(1, S, H, 512, generator=g).to(torch.bfloat16).to(gpu)
    out.backward(dout)
    assert_mla_grads(query.grad[:, 0], key.grad[:, 0], query.detach().cpu()[:, 0], key.detach().cpu()[:, 0], ref["idx"],
                     dout[0].cpu(), 0, mod.softmax_scale, out=out[0])
    # the indexer loss reached the indexer's weights and only those
    grads = {n: p.grad for n, p in mod.named_parameters()}
    assert all(gv is not None and torch.isfinite(gv).all() and gv.abs().max() > 0 for n, gv in grads.items()
               if "indexer" in n and "k_norm.bias" not in n)


def test_indexer_front_end_with_fused_rope_matches_the_torch_rope(gpu):
    """config.apply_rope_fusion routes the indexer's RoPE through the in-place HIP kernel
    (dsa_fused.py:435-451 of the reference); q and k must agree with the torch-op path to bf16 rounding,
    for one sequence and for a packed batch, and gradients must reach the projection weights."""
    import copy

    from loongforge_amd import dsa_fused
    from loongforge_amd.megatron_compat import PackedSeqParams

    S, Hi, Di, hid, qlr = 300, 4, 128, 96, 48
    cfg = _cfg(num_attention_heads=16, hidden_size=hid, q_lora_rank=qlr, dsa_indexer_n_heads=Hi, dsa_indexer_head_dim=Di,
               dsa_indexer_topk=64, dsa_indexer_loss_coeff=1.0, rope_type="rope", rotary_percent=1.0, rotary_base=10000,
               init_method=None, layernorm_epsilon=1e-5, dsa_indexer_rotate_activation=True, enable_chunkpipe=False)
    sub = dsa_fused.DSAIndexerFusedSubmodules(linear_wq_b=_Linear, linear_wk=_Linear, k_norm=_Norm, linear_weights_proj=_Linear)
    torch.manual_seed(1)
    plain = dsa_fused.DSAIndexerFused(cfg, sub)
    for p in plain.parameters():
        if p.ndim == 2:
            torch.nn.init.normal_(p, std=p.shape[1] ** -0.5)
    plain = plain.to(gpu)
    fused = copy.deepcopy(plain)
    fused.config = copy.copy(cfg)
    fused.config.apply_rope_fusion = True
    g = torch.Generator().manual_seed(2)
    for packed in (False, True):
        shape = (S, hid) if packed else (S, 1, hid)
        x = torch.randn(*shape, generator=g).to(torch.bfloat16).to(gpu)
        qr = torch.randn(*shape[:-1], qlr, generator=g).to(torch.bfloat16).to(gpu)
        psp = None
        if packed:
            cu = torch.tensor([0, 100, 101, 300], dtype=torch.int32, device=gpu)
            psp = PackedSeqParams(qkv_format="thd", cu_seqlens_q=cu, cu_seqlens_kv=cu, max_seqlen_q=199, max_seqlen_kv=199)
        q0, k0, w0 = plain.get_query_key_weight_tensors(x, qr, psp, defer_rotation=True)
        q1, k1, w1 = fused.get_query_key_weight_tensors(x, qr, psp, defer_rotation=True)
        assert q1.shape == q0.shape and k1.shape == k0.shape and torch.equal(w0, w1)
        for a, b in ((q1, q0), (k1, k0)):
            err = (a.float() - b.float()).abs()
            # the torch path rounds every product and the sum to bf16, the kernel once: a few units in the last
            # place of the larger of the result and its two terms (inputs here stay below 8 in magnitude)
            assert (err <= 2.0 ** -6 * (b.float().abs() + 2.0)).all()
            assert torch.equal(a[..., 64:], b[..., 64:])                      # the non-rotary half is untouched
        (q1.float().square().sum() + k1.float().square().sum()).backward()
        assert all(p.grad is not None and torch.isfinite(p.grad).all() and p.grad.abs().max() > 0
                   for n, p in fused.named_parameters() if "weights_proj" not in n and "k_norm.bias" not in n)
        fused.zero_grad()


@pytest.mark.parametrize("patched,training", [(False, True), (False, False), (True, True)])
def test_packed_sequences_that_do_not_hold_every_query_are_refused_by_the_module(gpu, patched, training):
    """The check that is left to the device is waited for behind the attention, and still before the module returns, counts a loss
    or publishes ids; an indexer whose forward is not the module's own waits itself."""
    from loongforge_amd import dsa_fused
    from loongforge_amd.megatron_compat import AttnMaskType, ModuleSpec, PackedSeqParams

    S, H, Hi, Di, K, hid, qlr = 200, 32, 32, 128, 64, 96, 48
    cfg = _cfg(num_attention_heads=H, hidden_size=hid, q_lora_rank=qlr, dsa_indexer_n_heads=Hi,
               dsa_indexer_head_dim=Di, dsa_indexer_topk=K, dsa_indexer_loss_coeff=1.0, rope_type="rope",
               rotary_percent=1.0, rotary_base=10000, init_method=None, layernorm_epsilon=1e-5,
               dsa_indexer_rotate_activation=True, enable_chunkpipe=False, dsa_indexer_topk_freq=2,
               dsa_indexer_skip_topk_offset=0, num_layers=2)
    sub = dsa_fused.DSAttentionFusedSubmodules(indexer=ModuleSpec(
        module=dsa_fused.DSAIndexerFused,
        submodules=dsa_fused.DSAIndexerFusedSubmodules(linear_wq_b=_Linear, linear_wk=_Linear, k_norm=_Norm,
                                                       linear_weights_proj=_Linear)))
    torch.manual_seed(5)
    mod = dsa_fused.DSAttentionFused(cfg, sub, layer_number=1, attn_mask_type=AttnMaskType.causal, attention_type="self",
                                     k_channels=192)
    for p in mod.parameters():
        if p.ndim == 2:
            torch.nn.init.normal_(p, std=p.shape[1] ** -0.5)
    mod = mod.to(gpu).train(training)
    if patched:
        own = mod.indexer.forward
        mod.indexer.forward = lambda x, qr, packed_seq_params=None: own(x, qr, packed_seq_params)
    q, k = (torch.randn(*s, device=gpu, dtype=torch.bfloat16) for s in ((S, H, 576), (S, 576)))
    x, qr = (torch.randn(S, n, device=gpu, dtype=torch.bfloat16) for n in (hid, qlr))

    def call(ends):
        cu = torch.tensor([0] + ends, dtype=torch.int32, device=gpu)
        packed = PackedSeqParams(qkv_format="thd", cu_seqlens_q=cu, cu_seqlens_kv=cu, max_seqlen_q=S, max_seqlen_kv=S)
        return mod(q, k, None, None, x=x, qr=qr, attn_mask_type=AttnMaskType.causal, packed_seq_params=packed, index_share_carrier=carrier)

    tracker = dsa_fused.DSAIndexerLossLoggingHelperFused.tracker
    carrier = SimpleNamespace()
    tracker.clear()
    with pytest.raises(ValueError, match="inconsistent shapes"):
        call([90, S - 1])
    assert not tracker and not getattr(carrier, "dsa_topk_holder", {})
    carrier = SimpleNamespace()
    assert torch.isfinite(call([90, S]).float()).all() and set(carrier.dsa_topk_holder) == {1}


def test_index_share_second_layer_reuses_the_first_layers_topk(gpu):
    """dsa_indexer_topk_freq = 2 (dsa_fused.py:752-778, :839-878 of the reference): layer 1 owns an indexer
    and publishes its top-k ids in the carrier, layer 2 owns none and attends over layer 1's ids; only
    the computing layer contributes an indexer loss."""
    from loongforge_amd import dsa_fused, ops
    from loongforge_amd.megatron_compat import AttnMaskType, ModuleSpec

    S, H, Hi, Di, K, hid, qlr = 320, 16, 4, 64, 64, 96, 48
    cfg = _cfg(num_attention_heads=H, hidden_size=hid, q_lora_rank=qlr, dsa_indexer_n_heads=Hi,
               dsa_indexer_head_dim=Di, dsa_indexer_topk=K, dsa_indexer_loss_coeff=1.0, rope_type="rope",
               rotary_percent=1.0, rotary_base=10000, init_method=None, layernorm_epsilon=1e-5,
               dsa_indexer_rotate_activation=True, enable_chunkpipe=False, dsa_indexer_topk_freq=2,
               dsa_indexer_skip_topk_offset=0, num_layers=2)
    sub = dsa_fused.DSAttentionFusedSubmodules(indexer=ModuleSpec(
        module=dsa_fused.DSAIndexerFused,
        submodules=dsa_fused.DSAIndexerFusedSubmodules(linear_wq_b=_Linear, linear_wk=_Linear, k_norm=_Norm,
                                                       linear_weights_proj=_Linear)))
    torch.manual_seed(3)
    layers = [dsa_fused.DSAttentionFused(cfg, sub, layer_number=n, attn_mask_type=AttnMaskType.causal,
                                         attention_type="self", k_channels=192) for n in (1, 2)]
    assert layers[0].indexer is not None and not layers[0].skip_topk
    assert layers[1].indexer is None and layers[1].skip_topk and layers[1].source_layer == 1
    for p in layers[0].parameters():
        if p.ndim == 2:
            torch.nn.init.normal_(p, std=p.shape[1] ** -0.5)
    layers = [m.to(gpu).train() for m in layers]
    g = torch.Generator().manual_seed(4)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(torch.bfloat16).to(gpu)

    x, qr = rnd(S, 1, hid), rnd(S, 1, qlr)
    carrier = SimpleNamespace()
    dsa_fused.DSAIndexerLossLoggingHelperFused.tracker.clear()
    # the skipping layer cannot run before its source layer has
    with pytest.raises(RuntimeError, match="did not run before"):
        layers[1](rnd(S, 1, H, 576), rnd(S, 1, 576), None, None, x=x, qr=qr, attn_mask_type=AttnMaskType.causal,
                  index_share_carrier=SimpleNamespace())
    q1, k1 = rnd(S, 1, H, 576).requires_grad_(True), rnd(S, 1, 576).requires_grad_(True)
    out1 = layers[0](q1, k1, None, None, x=x, qr=qr, attn_mask_type=AttnMaskType.causal, index_share_carrier=carrier)
    ids = carrier.dsa_topk_holder[1]
    assert ids.shape == (S, K) and set(carrier.dsa_topk_holder) == {1}
    q2, k2 = rnd(S, 1, H, 576).requires_grad_(True), rnd(S, 1, 576).requires_grad_(True)
    out2 = layers[1](q2, k2, None, None, x=x, qr=qr, attn_mask_type=AttnMaskType.causal, index_share_carrier=carrier)
    assert set(carrier.dsa_topk_holder) == {1}                       # the skipping layer publishes nothing
    assert set(dsa_fused.DSAIndexerLossLoggingHelperFused.tracker) == {1}      # ... and adds no indexer loss
    # layer 2 attended over layer 1's ids: the same kernel on the same ids gives the same bits
    qp = torch.nn.functional.pad(q2.detach()[:, 0], (0, 0, 0, 128 - H))
    ref2, _, _ = ops.sparse_mla_fwd(qp, k2.detach()[:, 0], ids.int(), 0, layers[1].softmax_scale)
    assert torch.equal(out2[0], ref2[:, :H])
    ro, _, _ = O.sparse_mla_fwd(q2.detach().cpu()[:, 0], k2.detach().cpu()[:, 0], ids.cpu(), 0, layers[1].softmax_scale, 512)
    assert_close(out2[0], ro, "out of the sharing layer")
    dout = rnd(1, S, H, 512)
    (out1 * dout).sum().backward()
    (out2 * dout).sum().backward()
    assert_mla_grads(q2.grad[:, 0], k2.grad[:, 0], q2.detach().cpu()[:, 0], k2.detach().cpu()[:, 0], ids.cpu(),
                     dout[0].cpu(), 0, layers[1].softmax_scale, "sharing layer:", out=out2[0])
    assert all(p.grad is not None for n, p in layers[0].named_parameters() if "indexer" in n and "k_norm.bias" not in n)


def test_chunkpipe_chunks_through_the_kernels_match_the_whole_sequence(gpu):
    """Chunkpipe (dsa_fused.py:234-421, :674-690, :897-901 of the reference) on the HIP path: every chunk of
    a sequence, given the latent keys of the sequence so far, selects the same keys as the whole sequence in
    one call (the indexer scores chunk queries against [cached keys | own keys] at their global positions) and
    produces the same attention rows bit for bit; the indexer's weight gradients, with the chunks' backward
    passes run last chunk first, agree with the whole-sequence ones."""
    import copy

    from loongforge_amd import dsa_fused
    from loongforge_amd.megatron_compat import AttnMaskType, ModuleSpec

    C, cs, H, Hi, Di, K, hid, qlr = 3, 128, 16, 4, 128, 64, 96, 48
    S = C * cs
    base = dict(num_attention_heads=H, hidden_size=hid, q_lora_rank=qlr, dsa_indexer_n_heads=Hi,
                dsa_indexer_head_dim=Di, dsa_indexer_topk=K, dsa_indexer_loss_coeff=1.0, rope_type="rope",
                rotary_percent=1.0, rotary_base=10000, init_method=None, layernorm_epsilon=1e-5,
                dsa_indexer_rotate_activation=True)
    cfg_w = _cfg(enable_chunkpipe=False, **base)
    cfg_c = _cfg(enable_chunkpipe=True, chunk_num_per_seq=C, chunksize=cs, micro_batch_size=1, chunkpipe_forward=True,
                 chunkpipe_forward_microbatch=0, chunkpipe_backward_microbatch=0, keep_activations_chunks=C,
                 virtual_pipeline_model_parallel_size=None, **base)
    sub = dsa_fused.DSAttentionFusedSubmodules(indexer=ModuleSpec(
        module=dsa_fused.DSAIndexerFused,
        submodules=dsa_fused.DSAIndexerFusedSubmodules(linear_wq_b=_Linear, linear_wk=_Linear, k_norm=_Norm,
                                                       linear_weights_proj=_Linear)))
    torch.manual_seed(7)
    whole = dsa_fused.DSAttentionFused(cfg_w, sub, layer_number=1, attn_mask_type=AttnMaskType.causal,
                                       attention_type="self", k_channels=192)
    for p in whole.parameters():
        if p.ndim == 2:
            torch.nn.init.normal_(p, std=p.shape[1] ** -0.5)
    whole = whole.to(gpu).train()
    chunked = dsa_fused.DSAttentionFused(cfg_c, sub, layer_number=1, attn_mask_type=AttnMaskType.causal,
                                         attention_type="self", k_channels=192).to(gpu).train()
    chunked.load_state_dict(whole.state_dict())
    g = torch.Generator().manual_seed(8)

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(torch.bfloat16).to(gpu)

    query, key, x, qr, dout = rnd(S, 1, H, 576), rnd(S, 1, 576), rnd(S, 1, hid), rnd(S, 1, qlr), rnd(1, S, H, 512)
    out_w = whole(query, key, None, None, x=x, qr=qr, attn_mask_type=AttnMaskType.causal)
    with torch.no_grad():
        _, ids_w = whole.indexer(x, qr)
    (out_w * dout).sum().backward()

    outs = []
    for c in range(C):
        cfg_c.chunkpipe_forward_microbatch = c
        rows = slice(c * cs, (c + 1) * cs)
        outs.append(chunked(query[rows], key[: (c + 1) * cs], None, None, x=x[rows], qr=qr[rows],
                            attn_mask_type=AttnMaskType.causal))
        assert torch.equal(outs[-1], out_w[:, rows])
    for c in reversed(range(C)):
        (outs[c] * dout[:, c * cs:(c + 1) * cs]).sum().backward()
    assert not chunked.indexer.indexer_key_cache_grad
    for (n, pw), pc in zip(whole.named_parameters(), chunked.parameters()):
        if "k_norm.bias" in n and pw.grad is None:
            continue
        # each chunk's loss is normalised by the chunk's length (loss / sq, dsa_fused.py:940), the whole
        # sequence's by S: C times the gradient.  The key gradient reaches the projections as a sum of bf16
        # pieces, one per chunk, instead of one bf16 value.
        scale = pw.grad.abs().max().item()
        err = (pc.grad / C - pw.grad).abs().max().item()
        assert err <= 2e-2 * scale, "%s: %.3e against %.3e" % (n, err, scale)


@pytest.mark.parametrize("case", ["rotate", "plain", "packed", "packed_host", "front"])
def test_indexer_forward_in_one_call_is_that_of_the_separate_calls(gpu, case, monkeypatch):
    """Quantisers, key windows and selection issued by one native call: the same bits, saved tensors and gradients as step by step,
    with gradients recorded and without."""
    from loongforge_amd import dsa_fused_kernels as K, ops
    from loongforge_amd.megatron_compat import PackedSeqParams

    S, off = 70, 0 if case.startswith("packed") else 130
    Sk = S + off
    g = torch.Generator().manual_seed(3)
    q, k, w = (torch.randn(*s, generator=g).to(gpu, torch.bfloat16) for s in ((S, 32, 128), (Sk, 128), (S, 32)))
    packed, front, ln = None, None, (None, None)
    if case.startswith("packed"):
        cu = torch.tensor([0, 9, 9, 41, 70], dtype=torch.int32, device="cpu" if case == "packed_host" else gpu)
        packed = PackedSeqParams(qkv_format="thd", cu_seqlens_q=cu, cu_seqlens_kv=cu, max_seqlen_q=32, max_seqlen_kv=32)
    if case == "front":
        ang = torch.rand(Sk, 64, generator=g).to(gpu)
        ln = (torch.rand(128, generator=g).to(gpu), torch.rand(128, generator=g).to(gpu))
        front = K.IndexerFrontEnd(cos=ang.cos(), sin=ang.sin(), pairing=ops.ROPE_SPLIT)
    kern, rotate = K.DSAIndexerKernel(), case != "plain"

    def both(record):
        leaves = [t.clone().requires_grad_(record) for t in (q, k, w) + tuple(x for x in ln if x is not None)]
        with torch.set_grad_enabled(record):
            s, i = kern(leaves[0], leaves[1], leaves[2], 64, off, packed, rotate, front, *(leaves[3:] or (None, None)))
        grads = torch.autograd.grad(s, leaves, torch.where(i >= 0, torch.ones_like(s), torch.zeros_like(s))) if record else ()
        return (s, i) + tuple(grads)

    whole = [both(r) for r in (False, True)]
    monkeypatch.setattr(ops, "indexer_forward", lambda *a, **k: None)
    steps = both(True)
    assert all(torch.equal(a, b) for res in whole for a, b in zip(res, steps))
    if packed is not None:
        monkeypatch.undo()
        short = PackedSeqParams(qkv_format="thd", cu_seqlens_q=packed.cu_seqlens_q[:4], cu_seqlens_kv=packed.cu_seqlens_kv[:4],
                                max_seqlen_q=32, max_seqlen_kv=32)
        with torch.no_grad(), pytest.raises(ValueError, match="packed sequences"):
            kern(q, k, w, 64, 0, short, True)


@pytest.mark.parametrize("shape,interleaved", [((5, 2, 3), False), ((1, 1, 1), True), ((7,), False)])
def test_absorbed_key_without_gradients_is_that_of_the_autograd_function(gpu, shape, interleaved):
    """Also for strided inputs, which the one native call leaves to the autograd function."""
    from loongforge_amd import dsa_fused_kernels as K, ops

    packed = len(shape) == 1
    lead, heads = (shape, 2) if packed else (shape[:2], shape[2])
    kv = torch.randn(*lead, heads, 512, device=gpu).to(torch.bfloat16)
    pe = torch.randn(*lead, 1, 64, device=gpu).to(torch.bfloat16)
    ang = torch.rand(8, 1, 1, 64, device=gpu)
    cu = torch.tensor([0, 3, 7], dtype=torch.int32, device=gpu) if packed else None
    args = (ang.cos().contiguous(), ang.sin().contiguous(), 64, 512, cu, 0, 1, interleaved)
    want = K.fused_apply_mla_rope_for_absorb_kv(kv.clone().requires_grad_(True), pe, *args)
    wide = torch.cat([kv, kv], -1)[..., :512]
    with torch.no_grad():
        for x in (kv, wide) if packed else (kv,):
            assert torch.equal(K.fused_apply_mla_rope_for_absorb_kv(x, pe, *args), want)
    with pytest.raises((AssertionError, RuntimeError)):
        with torch.no_grad():
            K.fused_apply_mla_rope_for_absorb_kv(kv, pe, ang.cos(), ang.sin()[:, :, :, ::2], 64, 512, cu, 0, 1, interleaved)


def test_calls_that_are_not_eager_take_the_functions(gpu):
    """Under a transform, a dispatch mode or a trace the native calls do nothing."""
    from torch._subclasses import FakeTensorMode

    from loongforge_amd import ops

    mk = lambda: (torch.zeros(4, 32, 128, device=gpu, dtype=torch.bfloat16), torch.zeros(9, 128, device=gpu, dtype=torch.bfloat16),     # noqa: E731
                  torch.zeros(4, 32, device=gpu))
    q, k, w = mk()
    assert ops.indexer_forward(q, k, w, True, 1.0, None, 0, 64, True) is not None
    assert ops.indexer_forward(q.requires_grad_(True), k, w, True, 1.0, None, 0, 64, True) is None
    with FakeTensorMode():
        assert ops.indexer_forward(*mk(), True, 1.0, None, 0, 64, True) is None
    seen = []
    torch.func.vmap(lambda x: (seen.append(ops.indexer_forward(x, k, w, True, 1.0, None, 0, 64, True)), x)[1])(torch.stack([q.detach(), q.detach()]))
    assert seen == [None]


@pytest.mark.parametrize("heads,S,packed", [(16, 1, False), (16, 900, False), (40, 450, True), (100, 130, False), (1, 70, True)])
def test_heads_are_padded_inside_the_attention(gpu, heads, S, packed):
    """Head counts that are no multiple of 32: the same bits as with the query padded and the output cut outside the attention, forward and
    gradients, where queries are worked as one (900 x 16 and 450 x 40 heads) and where not."""
    from loongforge_amd import ops
    from loongforge_amd.dsa_fused_kernels import DSADotProductAttention
    from loongforge_amd.megatron_compat import PackedSeqParams

    g = torch.Generator().manual_seed(heads)
    K, total = 128, (heads + 31) // 32 * 32
    attn = DSADotProductAttention(_cfg(num_attention_heads=heads), softmax_scale=192 ** -0.5)
    lead = (S,) if packed else (S, 1)
    q = torch.randn(*lead, heads, 576, generator=g).to(gpu, torch.bfloat16).requires_grad_(True)
    kv = torch.randn(*lead, 576, generator=g).to(gpu, torch.bfloat16).requires_grad_(True)
    # neighbouring queries share their keys, so that joint units pay
    seen = [torch.randperm(max(i, 1), generator=g)[:K].tolist() for i in range(0, S, 8)]
    ids = torch.tensor([(seen[i // 8] + [-1] * K)[:K] for i in range(S)], dtype=torch.int32, device=gpu)
    psp = PackedSeqParams(qkv_format="thd") if packed else None
    dout = torch.randn(*((S,) if packed else (1, S)), heads, 512, generator=g).to(gpu, torch.bfloat16)
    inside, dist = attn(q, kv, ids.unsqueeze(0), 0, packed_seq_params=psp, return_attn_dist=heads, padded_heads=total)
    got = torch.autograd.grad(inside, [q, kv], dout)
    outside, dist2 = attn(torch.nn.functional.pad(q, (0, 0, 0, total - heads)), kv, ids.unsqueeze(0), 0, packed_seq_params=psp, return_attn_dist=heads)
    outside = outside[..., :heads, :]
    want = torch.autograd.grad(outside, [q, kv], dout)
    assert inside.shape == outside.shape and torch.equal(inside, outside) and torch.equal(dist, dist2)
    assert got[0].shape == q.shape and got[0].is_contiguous() and torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    with pytest.raises(ValueError):
        attn(q, kv, ids.unsqueeze(0), 0, packed_seq_params=psp)                       # still refused without the padding
    x = q.detach().reshape(-1)[4:4 + S // 2 * heads * 576].view(-1, heads, 576)       # starts inside a 16-byte piece
    if x.numel():
        assert torch.equal(ops.pad_heads(x, total), torch.nn.functional.pad(x, (0, 0, 0, total - heads)))


def _loss_scale(scale, gpu):
    return torch.tensor([3.7], device=gpu) if scale == "one element" else torch.tensor(3.7) if scale == "on the host" else torch.tensor(scale, device=gpu)


@pytest.mark.parametrize("scale", [None, 3.7, 2.0 ** 70, "one element", "on the host"])
def test_gradient_of_the_attached_loss_belongs_to_its_receiver(gpu, scale, monkeypatch):
    """A hook that writes into the gradient of the scores changes what this pass hands on and nothing else: a second pass over a kept graph
    has the bits of the first, and those of the loss function and the auto-scaler by themselves (for a scale that makes up for a factor
    below what 32 bits hold of the gradients, too)."""
    from loongforge_amd import megatron_compat, ops

    S, K, factor = 40, 256, 1.5e-38 if scale == 2.0 ** 70 else 1.5 / 40
    g = torch.Generator(device=gpu).manual_seed(3)
    x, start = torch.randn(S, 8, generator=g, device=gpu), torch.randn(S, K, generator=g, device=gpu)
    target, scaler = torch.softmax(torch.randn(S, K, generator=g, device=gpu), -1), megatron_compat.DSAIndexerLossAutoScaler
    monkeypatch.setattr(scaler, "main_loss_backward_scale", None if scale is None else _loss_scale(scale, gpu))
    results = []
    for one in (True, False):
        leaf = start.clone().requires_grad_(True)
        scores = leaf * 1.0
        scores.register_hook(lambda grad: grad.mul_(3.0))
        if one:
            out, loss = ops.attached_indexer_kl_loss(x, scores, target, 1e-10, factor, scaler)
        else:
            loss = ops.indexer_kl_loss(scores, target, 1e-10, factor)
            out = scaler.apply(x, loss)
        for _ in range(2):
            results.append((loss.detach(), torch.autograd.grad(out, leaf, torch.ones_like(out), retain_graph=True)[0]))
    assert results[0][1].abs().max().item() > 0
    for loss, grad in results[1:]:
        assert torch.equal(loss, results[0][0]) and torch.equal(grad, results[0][1])


@pytest.mark.parametrize("scale", [None, 4.0, 3.7, "one element", "on the host"])
def test_loss_attached_in_one_node_is_that_of_the_two(gpu, scale, monkeypatch):
    """The indexer's loss with its attachment in one node: the bits of the loss function and the auto-scaler by themselves, for no loss scale
    and for one, in a second backward pass, with saved tensors on their way through a hook and where the indexer needs no gradient."""
    from loongforge_amd import dsa_fused, megatron_compat, ops
    from loongforge_amd.megatron_compat import AttnMaskType, ModuleSpec

    S, H, hid, qlr = 300, 32, 96, 48
    cfg = _cfg(num_attention_heads=H, hidden_size=hid, q_lora_rank=qlr, dsa_indexer_n_heads=32, dsa_indexer_head_dim=128, dsa_indexer_topk=128,
               dsa_indexer_loss_coeff=1.5, rope_type="rope", rotary_percent=1.0, rotary_base=10000, init_method=None, layernorm_epsilon=1e-5,
               dsa_indexer_rotate_activation=True, enable_chunkpipe=False, apply_rope_fusion=True)
    sub = dsa_fused.DSAttentionFusedSubmodules(indexer=ModuleSpec(
        module=dsa_fused.DSAIndexerFused,
        submodules=dsa_fused.DSAIndexerFusedSubmodules(linear_wq_b=_Linear, linear_wk=_Linear, k_norm=_Norm, linear_weights_proj=_Linear)))
    torch.manual_seed(0)
    mod = dsa_fused.DSAttentionFused(cfg, sub, layer_number=1, attn_mask_type=AttnMaskType.causal, attention_type="self", k_channels=192)
    for p in mod.parameters():
        if p.ndim == 2:
            torch.nn.init.normal_(p, std=p.shape[1] ** -0.5)
    mod = mod.to(gpu).train()
    g = torch.Generator(device=gpu).manual_seed(0)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=gpu, dtype=torch.bfloat16)      # noqa: E731
    query, key, x, qr, dout = rnd(S, 1, H, 576).requires_grad_(True), rnd(S, 1, 576).requires_grad_(True), rnd(S, 1, hid), rnd(S, 1, qlr), rnd(1, S, H, 512)
    value = None if scale is None else _loss_scale(scale, gpu)

    class Subclass(megatron_compat.DSAIndexerLossAutoScaler):        # no longer the class itself: the two nodes
        pass

    calls = []
    attach = ops.attached_indexer_kl_loss
    monkeypatch.setattr(ops, "attached_indexer_kl_loss", lambda *a: (calls.append(1), attach(*a))[1])
    monkeypatch.setattr(megatron_compat.DSAIndexerLossAutoScaler, "main_loss_backward_scale", value)

    def run():
        inputs = [query, key] + [p for p in mod.parameters() if p.requires_grad]
        out = mod(query, key, None, None, x=x, qr=qr, attn_mask_type=AttnMaskType.causal)
        first = torch.autograd.grad(out, inputs, dout, retain_graph=True, allow_unused=True)
        again = torch.autograd.grad(out, inputs, dout, allow_unused=True)
        assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(first, again))
        return [out.detach(), dsa_fused.DSAIndexerLossLoggingHelperFused.tracker[1], *first]

    def same(a, b):
        assert len(a) == len(b) and all((u is None and v is None) or torch.equal(u, v) for u, v in zip(a, b))

    one = run()
    assert calls == [1]
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.clone())[1], lambda t: t):
        same(run(), one)
    assert (S, 128) in packed
    with monkeypatch.context() as m:
        m.setattr(dsa_fused, "DSAIndexerLossAutoScaler", Subclass)
        same(run(), one)
    assert len(calls) == 2
    mod.indexer.requires_grad_(False)
    frozen = run()
    same(frozen, one[:4])


@pytest.mark.parametrize("heads,sinks", [(16, 16), (16, 4), (48, 48), (40, 64)])
def test_attention_sinks_of_padded_heads(gpu, heads, sinks):
    """A sink for every head, or one for several neighbouring ones, goes with the heads of the query and not with the padded ones; one that
    has a value for each padded head is taken as it is."""
    from loongforge_amd.dsa_fused_kernels import DSADotProductAttention

    g = torch.Generator().manual_seed(heads + sinks)
    S, K, total = 70, 64, (heads + 31) // 32 * 32
    attn = DSADotProductAttention(_cfg(num_attention_heads=heads), softmax_scale=192 ** -0.5)
    q = torch.randn(S, 1, heads, 576, generator=g).to(gpu, torch.bfloat16)
    kv = torch.randn(S, 1, 576, generator=g).to(gpu, torch.bfloat16)
    ids = torch.arange(S, dtype=torch.int32)[:, None] - torch.arange(K, dtype=torch.int32)
    ids = ids.clamp(min=-1).to(gpu).unsqueeze(0)
    sink = torch.randn(sinks, generator=g).to(gpu) * 3
    each = sink if sinks == total else torch.nn.functional.pad(sink.repeat_interleave(heads // sinks), (0, total - heads))
    got = attn(q, kv, ids, 0, attn_sink=sink, padded_heads=total)
    want = attn(torch.nn.functional.pad(q, (0, 0, 0, total - heads)), kv, ids, 0, attn_sink=each)[..., :heads, :]
    assert torch.equal(got, want)
