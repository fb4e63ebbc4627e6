"""GPU parity of the fused indexer front end (LayerNorm -> RoPE -> Hadamard rotation -> e4m3 quantiser in one
kernel): bit for bit against the CPU oracle, and against the separate kernels it replaces."""
import pytest
import torch

from oracle import front_oracle as F
from oracle import rope_oracle as R

pytestmark = pytest.mark.gpu


def _case(seed, tokens, heads, scale=2.0):
    g = torch.Generator().manual_seed(seed)
    x = (torch.randn(tokens, heads, 128, generator=g) * scale).to(torch.bfloat16)
    w, b = torch.randn(128, generator=g), torch.randn(128, generator=g)
    hw = torch.randn(tokens, heads, generator=g)
    pos = torch.randint(0, 96, (tokens,), generator=g, dtype=torch.int32)
    return x, w, b, hw, pos


def _same(got, ref):
    x8, si, rows, ws = got
    r8, rs, rrows, rws = ref
    assert torch.equal(rows.cpu(), rrows), "rows that were quantised"
    assert torch.equal(x8.cpu().view(torch.uint8), r8.view(torch.uint8)) and torch.equal(si.cpu(), rs)
    if rws is not None:
        assert torch.equal(ws.cpu(), rws)


@pytest.mark.parametrize("pairing", [R.ADJACENT, R.SPLIT])
@pytest.mark.parametrize("table_dtype", [torch.bfloat16, torch.float32])
def test_front_end_kernel_equals_the_oracle_bit_for_bit(gpu, pairing, table_dtype):
    from loongforge_amd import ops

    cos, sin = R.rope_tables(96, 64, dtype=table_dtype)
    # key side: one row per token, LayerNorm, positions from a table (packed documents)
    x, w, b, hw, pos = _case(1, 333, 1)
    x[7] = 0                                     # LayerNorm of a zero row is the bias
    x[8] = 3.0                                   # ... and so is that of a constant row
    got = ops.indexer_front_e4m3(x.to(gpu), 1, w.to(gpu), b.to(gpu), 1e-6, cos.to(gpu), sin.to(gpu), pairing, pos.to(gpu),
                                 1, True, return_rows=True)
    _same(got, F.indexer_front(x, 1, w, b, 1e-6, cos, sin, pairing, pos, 1, True))
    # query side: 64 rows per token, no LayerNorm, position = token // batch, scaled head weights
    x, w, b, hw, pos = _case(2, 190, 64)
    got = ops.indexer_front_e4m3(x.to(gpu), 64, None, None, 0.0, cos.to(gpu), sin.to(gpu), pairing, None, 2, True,
                                 hw.to(gpu), 128 ** -0.5, return_rows=True)
    _same(got, F.indexer_front(x, 64, None, None, 0.0, cos, sin, pairing, None, 2, True, hw, 128 ** -0.5))
    # no rotation (models that do not rotate their indexer activations)
    x, w, b, hw, pos = _case(3, 50, 4)
    got = ops.indexer_front_e4m3(x.to(gpu), 4, None, None, 0.0, cos.to(gpu), sin.to(gpu), pairing, pos.to(gpu), 1, False,
                                 return_rows=True)
    _same(got, F.indexer_front(x, 4, None, None, 0.0, cos, sin, pairing, pos, 1, False))


def test_front_end_kernel_equals_the_separate_kernels(gpu):
    """The stages as the separate kernels run them: torch LayerNorm (fp32 statistics in torch's own summation
    order: a bf16 step apart now and then), the in-place rotary kernel, the rotation + quantiser kernel."""
    from loongforge_amd import ops

    x, w, b, hw, pos = _case(4, 2048, 1)
    cos, sin = R.rope_tables(96, 64, dtype=torch.bfloat16)
    xd, cd, sd, pd = x.to(gpu), cos.to(gpu), sin.to(gpu), pos.to(gpu)
    x8, si, rows, _ = ops.indexer_front_e4m3(xd, 1, w.to(gpu), b.to(gpu), 1e-5, cd, sd, R.SPLIT, pd, 1, True, return_rows=True)
    v = torch.nn.functional.layer_norm(xd.float(), (128,), w.to(gpu), b.to(gpu), 1e-5).to(torch.bfloat16)
    pe = v[:, :, :64]
    ops.rope_rows(pe, pe, cd, sd, ops.ROPE_SPLIT, ops.ROPE_SPLIT, False, pd, 1)
    r8, rs, rrows = ops.rotate_quant_e4m3(v, return_rotated=True)
    err = (rows.float() - rrows.float()).abs()
    assert (err <= 2.0 ** -7 * rrows.float().abs() + 2.0 ** -9 * rrows.float().abs().amax(-1, keepdim=True)).all()
    assert (err == 0).float().mean().item() > 0.97
    # without LayerNorm every stage is exact arithmetic on the same values: identical bits
    x8b, sib, rowsb, _ = ops.indexer_front_e4m3(xd, 1, None, None, 0.0, cd, sd, R.SPLIT, pd, 1, True, return_rows=True)
    v2 = xd.clone()
    pe2 = v2[:, :, :64]
    ops.rope_rows(pe2, pe2, cd, sd, ops.ROPE_SPLIT, ops.ROPE_SPLIT, False, pd, 1)
    r8, rs, rrows = ops.rotate_quant_e4m3(v2, return_rotated=True)
    assert torch.equal(rowsb, rrows) and torch.equal(x8b.view(torch.uint8), r8.view(torch.uint8)) and torch.equal(sib, rs)
    with pytest.raises(ValueError):
        ops.indexer_front_e4m3(xd, 1, w.to(gpu), None)
    with pytest.raises(ValueError):
        ops.indexer_front_e4m3(xd, 3)


class _Linear(torch.nn.Module):
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


@pytest.mark.parametrize("packed", [False, True])
def test_indexer_module_with_the_front_end_inside_the_kernel(gpu, packed):
    """DSAIndexerFused.forward with the fused front end (projections -> one kernel per side) against the
    same module running k_norm, the rotary kernel and the rotating quantiser one after the other: same
    selection, same scores to the rounding of the LayerNorm statistics, and gradients of every indexer
    weight (the LayerNorm's included) that agree."""
    import copy
    from types import SimpleNamespace

    from loongforge_amd import dsa_fused
    from loongforge_amd.megatron_compat import PackedSeqParams

    S, Hi, hid, qlr, K = 384, 8, 96, 48, 64
    cfg = SimpleNamespace(qk_pos_emb_head_dim=64, v_head_dim=128, kv_lora_rank=512, apply_rope_fusion=True,
                          num_attention_heads=16, kv_channels=192, num_layers=2, hidden_size=hid, q_lora_rank=qlr,
                          dsa_indexer_n_heads=Hi, dsa_indexer_head_dim=128, dsa_indexer_topk=K, dsa_indexer_loss_coeff=1.0,
                          rope_type="rope", rotary_percent=1.0, rotary_base=10000, init_method=None, layernorm_epsilon=1e-5,
                          dsa_indexer_rotate_activation=True, enable_chunkpipe=False)
    sub = dsa_fused.DSAIndexerFusedSubmodules(linear_wq_b=_Linear, linear_wk=_Linear, k_norm=_Norm, linear_weights_proj=_Linear)
    torch.manual_seed(11)
    fused = dsa_fused.DSAIndexerFused(cfg, sub)
    for p in fused.parameters():
        if p.ndim == 2:
            torch.nn.init.normal_(p, std=p.shape[1] ** -0.5)
    with torch.no_grad():
        fused.k_norm.weight.add_(0.2 * torch.randn(128))
        fused.k_norm.bias.add_(0.2 * torch.randn(128))
    fused = fused.to(gpu)
    staged = copy.deepcopy(fused)
    staged.indexer_kernel.supports_fused_front_end = False           # instance attribute: this copy keeps the separate stages
    g = torch.Generator().manual_seed(12)
    shape = (S, hid) if packed else (S, 1, hid)
    x = torch.randn(*shape, generator=g).to(torch.bfloat16).to(gpu)
    qr = torch.randn(*shape[:-1], qlr, generator=g).to(torch.bfloat16).to(gpu)
    psp = None
    if packed:
        cu = torch.tensor([0, 100, 101, 384], dtype=torch.int32, device=gpu)
        psp = PackedSeqParams(qkv_format="thd", cu_seqlens_q=cu, cu_seqlens_kv=cu, max_seqlen_q=283, max_seqlen_kv=283)
    assert fused._fused_front_end(x, psp) is not None and staged._fused_front_end(x, psp) is None
    sc1, id1 = fused(x, qr, psp)
    sc2, id2 = staged(x, qr, psp)
    fin = torch.isfinite(sc2)
    assert torch.equal(torch.isfinite(sc1), fin)
    tol = 5e-3 * sc2[fin].abs().max().item()
    assert (sc1[fin] - sc2[fin]).abs().max().item() <= tol
    assert (torch.sort(id1, 1).values == torch.sort(id2, 1).values).float().mean().item() > 0.99
    gsc = torch.randn(S, K, generator=torch.Generator().manual_seed(13)).to(gpu)
    torch.where(fin, sc1, torch.zeros_like(sc1)).mul(gsc).sum().backward()
    torch.where(fin, sc2, torch.zeros_like(sc2)).mul(gsc).sum().backward()
    for (n, a), b in zip(fused.named_parameters(), staged.parameters()):
        assert a.grad is not None and b.grad is not None, n
        scale = b.grad.float().abs().max().item()
        assert (a.grad.float() - b.grad.float()).abs().max().item() <= 3e-2 * scale, n


@pytest.mark.parametrize("heads_in,dim,heads_out", [(1, 64, 1), (4, 64, 32), (5, 100, 32), (33, 128, 64), (64, 7, 64)])
def test_quantiser_pads_on_the_way(gpu, heads_in, dim, heads_out):
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(dim)
    x = torch.randn(37, heads_in, dim, generator=g).to(torch.bfloat16).to(gpu)
    x[3] = 0.0
    padded = torch.nn.functional.pad(x, (0, 128 - dim, 0, heads_out - heads_in)).contiguous()
    for w in (torch.randn(37, heads_in, generator=g).to(gpu), torch.randn(37, heads_in, generator=g).to(gpu, torch.bfloat16)):
        want = ops.quant_rowwise_e4m3_weights(padded, torch.nn.functional.pad(w.float(), (0, heads_out - heads_in)), 0.3)
        got = ops.quant_padded_e4m3(x, heads_out, w, 0.3)
        assert torch.equal(got[0].view(torch.uint8), want[0].view(torch.uint8))
        assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
    assert ops.quant_padded_e4m3(x, heads_out)[2] is None


@pytest.mark.parametrize("shape,interleaved,mscale", [((1, 1, 1, 2), False, 1.0), ((65, 1, 4, 64), False, 1.0), ((33, 2, 3, 62), True, 1.25),
                                                      ((7, 5, 64), True, 1.0)])
def test_rope_in_rounded_steps_equals_the_separate_operations(gpu, shape, interleaved, mscale):
    """One kernel for the unfused rotary embedding: bit for bit what the bf16 tensor operations give, forward and gradient."""
    from loongforge_amd import megatron_compat as M, ops

    g = torch.Generator().manual_seed(5)
    rot = M.RotaryEmbedding(shape[-1]).to(gpu)
    ang = rot(shape[0] + 3, offset=11)
    ref_ang = torch.outer(torch.arange(shape[0] + 3, dtype=torch.float32, device=gpu) + 11, rot.inv_freq)
    assert torch.equal(ang, torch.cat((ref_ang, ref_ang), -1)[:, None, None, :])
    for dt in (torch.float32, torch.bfloat16):
        cos, sin = rot.get_cached_cos_sin(shape[0], dtype=dt)
        a = rot(shape[0])
        assert torch.equal(cos, a.cos().to(dt)) and torch.equal(sin, a.sin().to(dt))
    base = torch.randn(*shape[:-1], shape[-1] + 6, generator=g).to(torch.bfloat16).to(gpu)
    dout = torch.randn(*shape, generator=g).to(torch.bfloat16).to(gpu)

    def separate(t):
        if interleaved:
            t = torch.cat((t[..., 0::2], t[..., 1::2]), dim=-1)
        f = ang[: t.shape[0]].reshape(t.shape[0], *([1] * (t.ndim - 2)), t.shape[-1])
        cos, sin = (torch.cos(f) * mscale).to(t.dtype), (torch.sin(f) * mscale).to(t.dtype)
        x1, x2 = torch.chunk(t, 2, dim=-1)
        return t * cos + torch.cat((-x2, x1), dim=-1) * sin

    res = []
    for fn in (separate, lambda t: ops.rope_steps(t, ang, mscale, interleaved)):
        x = base.clone().requires_grad_(True)
        y = fn(x[..., : shape[-1]])
        res.append((y.detach(), torch.autograd.grad(y, x, dout)[0]))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])


@pytest.mark.parametrize("batch", [1, 2])
@pytest.mark.parametrize("interleaved", [False, True])
def test_rope_in_rounded_steps_of_batch_first_views(gpu, batch, interleaved):
    """[s, b, h, d] as a transposed view of [b, s, h, d], and a gradient that comes back through such a transpose: with one
    sequence in the batch the view counts as contiguous and its batch stride is that of the whole sequence."""
    from types import SimpleNamespace

    from loongforge_amd.megatron_compat import RotaryEmbedding, apply_rotary_pos_emb

    g = torch.Generator().manual_seed(9)
    angles, cfg = RotaryEmbedding(64).to(gpu)(5), SimpleNamespace(multi_latent_attention=interleaved)
    base, dout = (torch.randn(batch, 5, 2, 64, generator=g).to(torch.bfloat16).to(gpu) for _ in range(2))
    res = []
    for lay in (lambda t: t.transpose(0, 1), lambda t: t.transpose(0, 1).clone(memory_format=torch.contiguous_format)):
        x = base.clone().requires_grad_(True)
        y = apply_rotary_pos_emb(lay(x), angles, config=cfg)
        res.append((y.detach(), torch.autograd.grad(y.transpose(0, 1), x, dout)[0]))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    one = torch.cat([apply_rotary_pos_emb(base[i], angles, config=cfg).unsqueeze(1) for i in range(batch)], 1)
    assert torch.equal(res[0][0], one)


def test_rotary_angles_with_other_arguments(gpu):
    """Lengths, offsets and frequencies that the kernel does not take give what the tensor operations give."""
    from loongforge_amd.megatron_compat import RotaryEmbedding

    rot, ref = RotaryEmbedding(64).to(gpu), RotaryEmbedding(64)
    offsets = torch.tensor([7.0, 7.0, 3.0, 0.5])
    for length, offset in ((4, offsets), (4, torch.tensor(9.0)), (3.5, 2), (0, 0)):
        got = rot(length, offset.to(gpu) if torch.is_tensor(offset) else offset)
        assert torch.equal(got.cpu(), ref(length, offset))
    assert RotaryEmbedding(0).to(gpu)(4).shape == (4, 1, 1, 0)
    with pytest.raises(RuntimeError):
        rot.inv_freq = rot.inv_freq.view(2, 16)
        rot(4)


def test_rotary_embedding_with_a_scale_on_the_device(gpu):
    """A scale that is a tensor gets its gradient and is not read on the host."""
    from loongforge_amd.megatron_compat import RotaryEmbedding, apply_rotary_pos_emb

    x = torch.randn(5, 2, 3, 64, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(gpu)
    angles = RotaryEmbedding(64).to(gpu)(5)
    scale = torch.tensor(1.25, device=gpu, requires_grad=True)
    y = apply_rotary_pos_emb(x, angles, mscale=scale)
    assert torch.equal(y.detach(), apply_rotary_pos_emb(x, angles, mscale=1.25))
    (got,) = torch.autograd.grad(y.double().sum(), scale)
    half = x.double().roll(32, -1) * torch.cat((-torch.ones(32), torch.ones(32))).to(gpu)
    terms = x.double() * angles.double().cos() + half * angles.double().sin()
    # sums and gradients pass through bf16: per term a few roundings, and the sum over tokens and heads one per addend
    assert (got.double() - terms.sum()).abs() <= 2.0 ** -5 * terms.abs().sum()


@pytest.mark.parametrize("shape", [(0, 1, 2, 64), (5, 0, 2, 64), (5, 1, 0, 64), (0, 2, 64)])
def test_rotary_embedding_and_rotation_of_nothing(gpu, shape):
    """Empty tensors go through, forward and backward, as through the tensor operations."""
    from loongforge_amd.dsa_fused import rotate_activation
    from loongforge_amd.megatron_compat import RotaryEmbedding, apply_rotary_pos_emb

    x = torch.zeros(shape, dtype=torch.bfloat16, device=gpu, requires_grad=True)
    angles = RotaryEmbedding(64).to(gpu)(5)
    for f in (rotate_activation, lambda t: apply_rotary_pos_emb(t, angles)):
        y = f(x)
        assert y.shape == x.shape and y.dtype == x.dtype
        assert torch.autograd.grad(y, x, torch.zeros_like(y))[0].shape == x.shape


@pytest.mark.parametrize("n", [32, 64, 128, 256, 512])
def test_hadamard_rotation_of_other_widths(gpu, n):
    from loongforge_amd import dsa_fused

    g = torch.Generator().manual_seed(n)
    x = torch.randn(19, 3, n, generator=g).to(torch.bfloat16).to(gpu).requires_grad_(True)
    dout = torch.randn(19, 3, n, generator=g).to(torch.bfloat16).to(gpu)
    y = dsa_fused.rotate_activation(x)
    (dx,) = torch.autograd.grad(y, x, dout)
    h = dsa_fused._hadamard(n, torch.device("cpu"), torch.float64)
    for got, ref in ((y, x), (dx, dout)):
        want = ref.detach().double().cpu() @ h * n ** -0.5
        assert ((got.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all()


@pytest.mark.parametrize("interleaved", [False, True])
def test_separate_operations_under_transforms(gpu, interleaved):
    """What the tensor operations took before there were kernels: gradients of gradients, batched gradients, vmap, forward mode,
    views that start inside a 16-byte piece."""
    from types import SimpleNamespace

    from loongforge_amd.dsa_fused import rotate_activation
    from loongforge_amd.megatron_compat import RotaryEmbedding, apply_rotary_pos_emb

    g = torch.Generator().manual_seed(5)
    rnd = lambda *shape: torch.randn(*shape, generator=g).to(torch.bfloat16).to(gpu)                  # noqa: E731
    angles = RotaryEmbedding(64, 1.0).to(gpu)(9)
    cfg = SimpleNamespace(multi_latent_attention=interleaved)
    near = dict(rtol=2.0 ** -7, atol=2.0 ** -6)          # two roundings to bf16 of values up to 2
    for f in (rotate_activation, lambda t: apply_rotary_pos_emb(t, angles, config=cfg)):
        x, go, v = rnd(9, 2, 3, 64).requires_grad_(), rnd(9, 2, 3, 64).requires_grad_(), rnd(9, 2, 3, 64)
        y = f(x)
        (gx,) = torch.autograd.grad(y, x, go, create_graph=True)
        (gg,) = torch.autograd.grad(gx, go, v)
        assert torch.equal(gg, f(v))
        rows = torch.stack([rnd(9, 2, 3, 64) for _ in range(2)])
        (many,) = torch.autograd.grad(f(x), x, rows, is_grads_batched=True)
        for i in range(2):
            torch.testing.assert_close(many[i], torch.autograd.grad(f(x), x, rows[i])[0], **near)
        torch.testing.assert_close(torch.func.vmap(f)(rows), torch.stack([f(r) for r in rows]), **near)
        out, tangent = torch.func.jvp(f, (x.detach(),), (v,))
        torch.testing.assert_close(out, y.detach(), **near)
        torch.testing.assert_close(tangent, f(v), **near)
    odd = rnd(4 * 64 + 1)[1:].view(4, 64)
    assert torch.equal(rotate_activation(odd), rotate_activation(odd.clone()))


@pytest.mark.parametrize("S,Sk,heads,bf16_weights", [(1, 1, 1, True), (15, 15, 4, True), (17, 17, 32, False), (257, 300, 33, True), (1030, 1030, 64, False)])
def test_narrow_heads_in_one_kernel_are_those_of_the_separate_kernels(gpu, S, Sk, heads, bf16_weights):
    """Rotary embedding in rounded steps, rotation, padded quantisers and windows of 64-channel heads: the same bits in one launch, also
    for views that do not start on 16 bytes or do not lie in order; finished gradients against the same steps in 32 bits, each rounded
    to bf16 once (2^-8 relative each)."""
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(S + heads)
    K, factor, offset = 64, 64 ** -0.5, Sk - S
    q = torch.randn(S * heads * 64 + 1, generator=g).to(gpu, torch.bfloat16)[1:].view(S, heads, 64)
    k = torch.randn(64, Sk, generator=g).to(gpu, torch.bfloat16).t()
    w = torch.randn(S, heads, generator=g).to(gpu, torch.bfloat16 if bf16_weights else torch.float32)
    q[S // 2] = 0.0
    inv_freq = (10000.0 ** (-torch.arange(0, 64, 2, dtype=torch.float32) / 64)).to(gpu)
    angles = ops.rotary_angles(inv_freq, Sk)
    cos, sin = ops.rotary_cos_sin(inv_freq, Sk, 0.0, torch.bfloat16)
    scores, ids, q8, q_scale, scaled, k8, k_scale = ops.indexer_forward_narrow(q, k, w, cos, sin, factor, offset, K, True)
    qr = ops.hadamard(ops.rope_steps(q.contiguous(), angles))
    kr = ops.hadamard(ops.rope_steps(k.contiguous().unsqueeze(1), angles))
    want_q = ops.quant_padded_e4m3(qr, 32 if heads <= 32 else 64, w, factor)
    want_k = ops.quant_padded_e4m3(kr, 1)
    for a, b in zip((q8.view(torch.uint8), q_scale, scaled, k8.view(torch.uint8), k_scale),
                    (want_q[0].view(torch.uint8), want_q[1], want_q[2], want_k[0].squeeze(1).view(torch.uint8), want_k[1].squeeze(1))):
        assert torch.equal(a, b)
    ks, ke, _ = ops.indexer_window(None, S, offset, q8)
    want = ops.indexer_topk(q8, scaled, k8, k_scale, ks, ke, K)
    assert torch.equal(scores, want[0]) and torch.equal(ids, want[1])
    grad = torch.randn(S, K, generator=g).to(gpu) * (ids >= 0)
    args = (grad, q8, k8, k_scale, scaled, ids, q_scale, factor, heads, 64)
    got = ops.indexer_grads(*args, (torch.float32,) * 3, narrow=[cos, sin])
    ref = ops._indexer_grads_narrow(*args, (torch.float32,) * 3, cos, sin)
    for a, b in zip(got[:3], ref[:3]):
        assert a.shape == b.shape
        assert (a - b).norm().item() <= 2.0 ** -7 * b.norm().item() + 1e-12
    assert ops.indexer_forward_narrow(q, k, w, cos[:Sk - 1], sin[:Sk - 1], factor, offset, K, True) is None


@pytest.mark.parametrize("S,heads", [(1, 4), (129, 4), (1024, 40)])
def test_indexer_module_of_narrow_heads_in_one_kernel(gpu, S, heads):
    """DSAIndexerFused with 64-channel heads: the same scores and ids as with the separate operations, gradients of its
    projections and its norm within the bf16 roundings that the one kernel leaves out."""
    from types import SimpleNamespace

    from loongforge_amd import dsa_fused

    hid, qlr, K = 96, 48, 64
    cfg = SimpleNamespace(qk_pos_emb_head_dim=64, apply_rope_fusion=False, hidden_size=hid, q_lora_rank=qlr, dsa_indexer_n_heads=heads,
                          dsa_indexer_head_dim=64, dsa_indexer_topk=K, rope_type="rope", rotary_percent=1.0, rotary_base=10000, init_method=None,
                          layernorm_epsilon=1e-5, dsa_indexer_rotate_activation=True, enable_chunkpipe=False)
    sub = dsa_fused.DSAIndexerFusedSubmodules(linear_wq_b=_Linear, linear_wk=_Linear, k_norm=_Norm, linear_weights_proj=_Linear)
    torch.manual_seed(5)
    mod = dsa_fused.DSAIndexerFused(cfg, sub)
    for p in mod.parameters():
        if p.ndim == 2:
            torch.nn.init.normal_(p, std=p.shape[1] ** -0.5)
    mod = mod.to(gpu)
    g = torch.Generator().manual_seed(6)
    x, qr = torch.randn(S, 1, hid, generator=g).to(gpu, torch.bfloat16), torch.randn(S, 1, qlr, generator=g).to(gpu, torch.bfloat16)
    grad = torch.randn(S, K, generator=g).to(gpu)

    def passes():
        scores, ids = mod(x, qr)
        return scores.detach(), ids, torch.autograd.grad(scores, list(mod.parameters()), grad * (ids >= 0))

    assert mod._narrow_tables(x, None) is not None
    narrow = passes()
    mod._apply_rope = lambda *a: dsa_fused.DSAIndexerFused._apply_rope(mod, *a)        # not the class's own: the separate operations
    assert mod._narrow_tables(x, None) is None
    apart = passes()
    assert torch.equal(narrow[0], apart[0]) and torch.equal(narrow[1], apart[1])
    for a, b in zip(narrow[2], apart[2]):
        # three bf16 roundings each way, and the one of the result
        assert (a - b).float().norm().item() <= 2.0 ** -6 * b.float().norm().item() + 1e-6


@pytest.mark.parametrize("S,heads,pairing,packed,bf16_weights,rotate", [
    (1, 32, R.SPLIT, False, True, True), (17, 64, R.ADJACENT, False, False, True), (300, 32, R.SPLIT, True, True, True),
    (515, 64, R.SPLIT, "int64", True, False), (257, 64, R.ADJACENT, True, False, False)])
def test_both_fronts_and_the_windows_in_one_launch_are_those_of_separate_launches(gpu, S, heads, pairing, packed, bf16_weights, rotate):
    """Payloads, scales, head weights (scaled and rounded to their type on the way) and selection bit for bit; a table, a
    packed batch or an alignment that the separate kernels refuse is refused."""
    from loongforge_amd import ops
    from loongforge_amd.dsa_fused_kernels import IndexerFrontEnd

    g = torch.Generator().manual_seed(S)
    q = torch.randn(S, heads, 128, generator=g).to(gpu, torch.bfloat16)
    k = torch.randn(S, 128, generator=g).to(gpu, torch.bfloat16)
    w = torch.randn(S, heads, generator=g).to(gpu, torch.bfloat16 if bf16_weights else torch.float32)
    lw, lb = torch.randn(128, generator=g).to(gpu), torch.randn(128, generator=g).to(gpu)
    cos, sin = (t.to(gpu) for t in R.rope_tables(S, 64, dtype=torch.bfloat16))
    cu = pos = None
    if packed:
        cu = torch.tensor([0, S // 3, S // 3, S // 3 + 1, S], dtype=torch.int64 if packed == "int64" else torch.int32, device=gpu)
        pos = ops.thd_positions(cu, S)
    front = IndexerFrontEnd(cos=cos, sin=sin, pairing=pairing, positions_q=pos, positions_k=pos, batch=1, k_norm_eps=1e-6)
    scale, factor, K = heads ** -0.5, 128 ** -0.5, 64
    scores, ids, q8, q_scale, scaled, k8, k_scale, check = ops.indexer_forward(q, k, w, rotate, factor, cu, 0, K, True, front, lw, lb, weights_scale=scale)
    assert (check is not None) == bool(packed)
    if check is not None:
        check.wait()
    want_q = ops.indexer_front_e4m3(q, heads, None, None, 0.0, cos, sin, pairing, pos, 1, rotate, (w * scale).float(), factor)
    want_k = ops.indexer_front_e4m3(k, 1, lw, lb, 1e-6, cos, sin, pairing, pos, 1, rotate)
    for a, b in ((q8, want_q[0]), (k8, want_k[0])):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    assert torch.equal(q_scale, want_q[1]) and torch.equal(scaled, want_q[3]) and torch.equal(k_scale, want_k[1])
    ks, ke, _ = ops.indexer_window(cu, S, 0, q8)
    want = ops.indexer_topk(q8, scaled, k8, k_scale, ks, ke, K)
    assert torch.equal(scores, want[0]) and torch.equal(ids, want[1])
    if packed:
        short = ops.indexer_forward(q, k, w, rotate, factor, cu[:-1], 0, K, True, front, lw, lb)[-1]
        with pytest.raises(ValueError, match="inconsistent shapes"):
            short.wait()
    else:
        with pytest.raises(ValueError, match="shorter than the sequence"):
            ops.indexer_forward(q, k, w, rotate, factor, None, 0, K, True, IndexerFrontEnd(cos=cos[1:], sin=sin[1:], pairing=pairing), lw, lb)
