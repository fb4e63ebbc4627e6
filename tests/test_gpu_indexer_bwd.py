"""GPU parity: sparse backward of the indexer logits, and the autograd wrapper around the indexer."""
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu


def _reference(aux, idx, g, noise=2.0 ** -18):
    """fp64 autograd through the gathered logits + the set of (query, head) rows / keys touched by a
    ReLU gate whose exact pre-activation is within fp32 accumulation noise of zero (there the gate
    may legitimately fall on either side)."""
    q8f, k8f = aux["q8"], aux["k8"]
    qf = q8f.double().requires_grad_(True)
    kf = k8f.double().requires_grad_(True)
    wf = aux["weight_scaled"].double().requires_grad_(True)
    sel = O.gathered_indexer_logits(qf, wf, kf, aux["k_scale"], idx, dtype=torch.float64)
    (torch.where(idx >= 0, sel, torch.zeros_like(sel)) * g.double()).sum().backward()
    safe = idx.clamp(min=0).long()
    ksel = k8f.double()[safe]
    rex = torch.einsum("mhd,mkd->mhk", q8f.double(), ksel)
    mag = torch.einsum("mhd,mkd->mhk", q8f.double().abs(), ksel.abs())
    amb = (rex.abs() <= noise * mag) & (idx >= 0)[:, None, :]
    amb_key = torch.zeros(k8f.shape[0], dtype=torch.bool)
    amb_key[safe[amb.any(1)]] = True
    return qf.grad, kf.grad, wf.grad, amb.any(-1), amb_key


@pytest.mark.parametrize("S,Hi,K,seed", [(256, 64, 128, 1), (300, 32, 128, 2), (200, 64, 192, 3)])
def test_indexer_bwd_against_oracle(gpu, S, Hi, K, seed):
    from loongforge_amd import ops

    iq, ik, w = O.make_indexer_inputs(S, Hi, 128, seed=seed)
    _, idx, aux = O.indexer_forward(iq, ik, w, K, 0, None)
    g = torch.randn(S, K, generator=torch.Generator().manual_seed(seed + 1))
    g = torch.where(idx >= 0, g, torch.zeros_like(g))
    rq, rk, rw, amb_qh, amb_key = _reference(aux, idx, g)
    args = (g.to(gpu), aux["q8"].to(gpu), aux["k8"].to(gpu), aux["k_scale"].to(gpu),
            aux["weight_scaled"].to(gpu).contiguous(), idx.to(gpu))
    dq, dk, dw = ops.indexer_bwd(*args)
    dq2, dk2, dw2 = ops.indexer_bwd(*args)
    assert torch.equal(dq, dq2) and torch.equal(dk, dk2) and torch.equal(dw, dw2)      # bit-identical
    eq = (dq.double().cpu() - rq).abs().masked_fill(amb_qh[..., None], 0)
    ek = (dk.double().cpu() - rk).abs().masked_fill(amb_key[:, None], 0)
    ew = (dw.double().cpu() - rw).abs()
    assert eq.max().item() <= 1e-4 * rq.abs().max().item()
    assert ek.max().item() <= 4e-3 * rk.abs().max().item()       # a key's rows are summed in fp32 from bf16 rows
    assert ew.max().item() <= 1e-4 * rw.abs().max().item()


def test_indexer_bwd_with_a_repeated_id_returns_nan_keys(gpu):
    from loongforge_amd import ops

    iq, ik, w = O.make_indexer_inputs(256, 64, 128, seed=5)
    _, idx, aux = O.indexer_forward(iq, ik, w, 128, 0, None)
    idx = idx.clone()
    idx[200, 3] = idx[200, 17]
    g = torch.ones(256, 128)
    dq, dk, dw = ops.indexer_bwd(g.to(gpu), aux["q8"].to(gpu), aux["k8"].to(gpu), aux["k_scale"].to(gpu),
                                 aux["weight_scaled"].to(gpu).contiguous(), idx.to(gpu))
    assert torch.isnan(dk).all()


def test_indexer_kernel_module_forward_and_backward(gpu):
    """DSAIndexerKernel with the reference's call signature: unpadded head count / head dim (the
    reference's own CPU-sized configuration uses 4 heads of dim 64), packed documents, autograd."""
    from loongforge_amd.dsa_fused_kernels import DSAIndexerKernel
    from loongforge_amd.megatron_compat import PackedSeqParams

    S, Hi, D, K = 384, 4, 64, 64
    cu = torch.tensor([0, 100, 257, 384], dtype=torch.int32)
    iq, ik, w = O.make_indexer_inputs(S, Hi, D, seed=7, w_uniform=True)
    sc_ref, idx_ref, aux = O.indexer_forward(iq, ik, w, K, 0, cu, dtype=torch.float64)
    psp = PackedSeqParams(qkv_format="thd", cu_seqlens_q=cu.to(gpu), cu_seqlens_kv=cu.to(gpu), max_seqlen_q=157,
                          max_seqlen_kv=157)
    q = iq.to(gpu).requires_grad_(True)
    k = ik.to(gpu).requires_grad_(True)
    wt = w.to(gpu).requires_grad_(True)
    sc, ids = DSAIndexerKernel()(q, k, wt, K, 0, psp)
    assert sc.shape == (S, K) and ids.dtype == torch.int32
    noise = 1e-4 * sc_ref[torch.isfinite(sc_ref)].abs().max().item()
    assert torch.equal(torch.isfinite(sc.cpu()), torch.isfinite(sc_ref))
    fin = torch.isfinite(sc_ref)
    assert (sc.cpu()[fin].double() - sc_ref[fin].double()).abs().max().item() <= noise   # both sorted descending
    v = ids.cpu() >= 0
    ks, ke = aux["ks"], aux["ke"]
    assert ((ids.cpu() >= ks[:, None]) | ~v).all() and ((ids.cpu() < ke[:, None]) | ~v).all()
    # backward: gradient of sum(score * g) through the HIP indexer backward vs the oracle
    g = torch.randn(S, K, generator=torch.Generator().manual_seed(8))
    torch.where(torch.isfinite(sc), sc, torch.zeros_like(sc)).mul(g.to(gpu)).sum().backward()
    idc = ids.cpu()
    gz = torch.where(idc >= 0, g, torch.zeros_like(g))
    d_q, d_k, d_w = O.indexer_bwd(gz, aux["q8"], aux["k8"], aux["q_scale"], aux["k_scale"], aux["weight_scaled"], idc,
                                  dtype=torch.float64)
    # the oracle's d_w is w.r.t. the un-scaled weights already (d_w' * q_scale * d^-0.5)
    for name, got, ref in (("d_q", q.grad, d_q), ("d_k", k.grad, d_k), ("d_w", wt.grad, d_w)):
        err = (got.double().cpu() - ref).abs()
        lim = 2e-2 * ref.abs().max().item()       # bf16 grads; ReLU-gate flips are rarer than 1e-4 of pairs
        assert (err > lim).float().mean().item() < 1e-3, name


@pytest.mark.parametrize("S,Sk,heads,dim,K,rotate,pairing,dtypes", [
    (1, 1, 32, 128, 128, False, -1, "fff"),          # one pair
    (37, 45, 5, 64, 130, False, -1, "bbb"),          # few heads of few channels, slots padded to a tile
    (70, 300, 64, 128, 256, True, 0, "bbf"),
    (129, 129, 64, 128, 129, True, 1, "bfb"),
    (33, 700, 20, 100, 640, False, -1, "hfb"),       # rows of 100 channels, half precision
    (300, 40, 32, 128, 40, True, 1, "bbb"),          # rows without a valid slot, more queries than keys
])
def test_indexer_grads_equal_the_separate_steps(gpu, S, Sk, heads, dim, K, rotate, pairing, dtypes):
    """Payload gradients -> unscale -> rotation -> rotary transpose -> LayerNorm backward in the kernels, against the same
    steps one by one (from the kernels' own payload gradients, which the oracle test above covers)."""
    from loongforge_amd import ops
    from loongforge_amd.dsa_fused_kernels import IndexerFrontEnd, _unscale_indexer_grad

    gen = torch.Generator().manual_seed(S + K)
    hp = 32 if heads <= 32 else 64
    q = torch.zeros(S, hp, 128)
    q[:, :heads, :dim] = torch.randn(S, heads, dim, generator=gen)
    k = torch.zeros(Sk, 128)
    k[:, :dim] = torch.randn(Sk, dim, generator=gen)
    k[0] = 0.0                                                  # on the quantiser's epsilon floor
    w = torch.zeros(S, hp)
    w[:, :heads] = torch.randn(S, heads, generator=gen)
    q8, qs = ops.quant_rowwise_e4m3(q.to(torch.bfloat16).to(gpu))
    k8, ksc = ops.quant_rowwise_e4m3(k.to(torch.bfloat16).to(gpu))
    ws = (w.to(gpu) * qs * dim ** -0.5).contiguous()
    ids = torch.stack([torch.randperm(max(Sk, K), generator=gen)[:K] for _ in range(S)]).int()
    ids[ids >= Sk] = -1
    ids[S // 2] = -1 if S > 1 else ids[0]
    g = torch.randn(S, K, generator=gen)
    g[ids < 0] = float("nan")
    ids, g = ids.to(gpu), g.to(gpu)
    front = k_in = ln_w = None
    if pairing >= 0:
        ang = torch.rand(max(S, Sk), 64, generator=gen) * 6
        pos_q = torch.randint(0, max(S, Sk), (S,), generator=gen).int().to(gpu) if pairing == 1 else None
        front = IndexerFrontEnd(cos=ang.cos().to(gpu), sin=ang.sin().to(gpu, torch.float32), pairing=pairing, positions_q=pos_q, k_norm_eps=1e-5)
        k_in = torch.randn(Sk, 128, generator=gen).to(torch.bfloat16).to(gpu)
        ln_w = torch.randn(128, generator=gen).to(gpu)
    types = [dict(f=torch.float32, b=torch.bfloat16, h=torch.float16)[c] for c in dtypes]
    got = ops.indexer_grads(g, q8, k8, ksc, ws, ids, qs, dim ** -0.5, heads, dim, types, rotate, front, k_in, ln_w)
    again = ops.indexer_grads(g, q8, k8, ksc, ws, ids, qs, dim ** -0.5, heads, dim, types, rotate, front, k_in, ln_w)
    assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(got, again))

    d_q, d_k, d_w = ops.indexer_bwd(torch.where(ids >= 0, g, torch.zeros_like(g)), q8, k8, ksc, ws, ids)
    d_w = d_w * qs * dim ** -0.5
    d_q, d_k = _unscale_indexer_grad(d_q, qs), _unscale_indexer_grad(d_k, ksc)
    if rotate:
        h = O.hadamard(128).float().to(gpu) if hasattr(O, "hadamard") else None
        if h is None:
            h = torch.ones(1, 1, device=gpu)
            while h.shape[0] < 128:
                h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        d_q, d_k = (d_q @ h) * 128 ** -0.5, (d_k @ h) * 128 ** -0.5
    ref_ln = [None, None]
    if front is not None:
        d_q, d_k = d_q.to(torch.bfloat16).contiguous(), d_k.to(torch.bfloat16).contiguous()
        ops.rope_rows(d_q[:, :, :64], d_q[:, :, :64], front.cos, front.sin, pairing, pairing, True, front.positions_q)
        ops.rope_rows(d_k[:, None, :64], d_k[:, None, :64], front.cos, front.sin, pairing, pairing, True)
        x = k_in.float().requires_grad_(True)
        lw, lb = ln_w.clone().requires_grad_(True), torch.zeros(128, device=gpu, requires_grad=True)
        d_k, *ref_ln = torch.autograd.grad(torch.nn.functional.layer_norm(x, (128,), lw, lb, 1e-5), [x, lw, lb], d_k.float())
    want = [d_q[:, :heads, :dim].to(types[0]), d_k[:, :dim].to(types[1]), d_w[:, :heads].to(types[2])] + ref_ln
    for a, b, t in zip(got, want, types + [torch.float32] * 2):
        if b is None:
            assert a is None
            continue
        assert a.shape == b.shape and a.dtype == b.dtype
        # the same values up to the order of fp32 sums, i.e. now and then one step of the output's grid (or of the bf16
        # grid that the rotary part works on)
        scale = b.float().abs().max().item()
        step = {torch.float32: 2e-6, torch.float16: 2e-3, torch.bfloat16: 8e-3}[t]
        err = (a.float() - b.float()).abs()
        assert torch.isfinite(a.float()).all()
        if front is not None:
            assert (err <= 8e-3 * b.float().abs() + 8e-3 * scale).all() and err.mean() <= 2e-4 * scale
        else:
            assert (err <= step * b.float().abs() + 2e-6 * scale).all()


@pytest.mark.parametrize("S,Sk,K", [(1, 40000, 128), (70, 16385, 128), (33, 33000, 2048), (300, 16384, 2304)])
def test_key_sums_over_many_keys(gpu, S, Sk, K):
    """More keys than the order's lookup table holds at a time, and slot lists above and below the kernel's ring sizes."""
    from loongforge_amd import ops

    gen = torch.Generator().manual_seed(S)
    q8 = torch.randn(S, 32, 128, generator=gen).to(torch.float8_e4m3fn)
    k8 = torch.randn(Sk, 128, generator=gen).to(torch.float8_e4m3fn)
    ksc, w, g = torch.rand(Sk, generator=gen) + 0.5, torch.randn(S, 32, generator=gen), torch.randn(S, K, generator=gen)
    ids = torch.stack([torch.randperm(Sk, generator=gen)[:K] for _ in range(S)]).int()
    ids[:, K // 2:][torch.rand(S, K - K // 2, generator=gen) < 0.3] = -1
    for i in range(S):       # no gate within accumulation noise of zero
        q, k = q8[i].double(), k8[ids[i].clamp(min=0).long()].double()
        g[i, ((q @ k.T).abs() <= 2.0 ** -16 * (q.abs() @ k.abs().T)).any(0)] = 0.0
    dq, dk, dw = ops.indexer_bwd(*(t.to(gpu) for t in (g, q8, k8, ksc, w, ids)))
    rq, rk, rw = torch.zeros(S, 32, 128, dtype=torch.float64), torch.zeros(Sk, 128, dtype=torch.float64), torch.zeros(S, 32, dtype=torch.float64)
    rk_abs = torch.zeros(Sk, dtype=torch.float64)
    for i in range(S):
        live = ids[i] >= 0
        j = ids[i][live].long()
        q, k = q8[i].double(), k8[j].double()
        r = q @ k.T
        a = (g[i][live] * ksc[j]).double()
        e = w[i].double()[:, None] * a * (r > 0)
        rq[i], rw[i] = e @ k, (r.clamp(min=0) * a).sum(1)
        rk[j] += e.T @ q
        rk_abs[j] += (e.T @ q).abs().amax(1)
    assert (dq.cpu() - rq).abs().max() <= 1e-4 * rq.abs().max() and (dw.cpu() - rw).abs().max() <= 1e-4 * rw.abs().max()
    # pair rows are bf16, from head factors w q in bf16
    assert ((dk.cpu() - rk).abs() <= 2e-2 * rk_abs[:, None] + 1e-3).all()


def _pairs(S, Sk, K, Hi, seed, full):
    """Inputs of a backward whose queries select about `full` of K slots, no gate within accumulation noise of zero."""
    gen = torch.Generator().manual_seed(seed)
    q8 = torch.randn(S, Hi, 128, generator=gen).to(torch.float8_e4m3fn)
    k8 = torch.randn(Sk, 128, generator=gen).to(torch.float8_e4m3fn)
    ksc, w, g = torch.rand(Sk, generator=gen) + 0.5, torch.randn(S, Hi, generator=gen), torch.randn(S, K, generator=gen)
    ids = torch.full((S, K), -1, dtype=torch.int32)
    n = min(K, Sk)
    ids[:, :n] = torch.rand(S, Sk, generator=gen).topk(n, dim=1).indices.int()
    ids[torch.rand(S, K, generator=gen) > full] = -1
    ids[S // 3] = -1
    k = k8.double()[ids.clamp(min=0).long()]
    r = q8.double() @ k.transpose(1, 2)
    noise = r.abs() <= 2.0 ** -16 * (q8.double().abs() @ k.abs().transpose(1, 2))
    g[noise.any(1)] = 0.0
    return g, q8, k8, ksc, w, ids, r, k


def _grads(gpu, g, q8, k8, ksc, w, ids, span):
    from loongforge_amd import ops

    S, Hi = w.shape
    t = [x.to(gpu) for x in (g, q8, k8, ksc, w, ids)]
    d_q, d_k, d_w, _, _ = ops.indexer_grads(*t, torch.ones(S, Hi, device=gpu), 1.0, Hi, 128, [torch.float32] * 3, span=span)
    return d_q.cpu().double(), d_k.cpu().double() * ksc.double()[:, None], d_w.cpu().double()


# From 1600 queries on a span of one key makes the products with whole key tiles the cheaper way whatever the sizes.
@pytest.mark.parametrize("S,Sk,K,Hi,full", [
    (1600, 1, 128, 32, 0.9),
    (1601, 255, 128, 64, 0.5),           # one tile, a key short
    (1663, 257, 256, 32, 1.0),           # one key in the second tile
    (1605, 513, 384, 64, 0.01),          # tiles that few queries touch
    (1600, 4097, 128, 64, 1.0),          # one key in the second piece of factors
    (1700, 9000, 256, 32, 0.3),
])
def test_key_gradients_by_key_tiles(gpu, S, Sk, K, Hi, full):
    g, q8, k8, ksc, w, ids, r, k = _pairs(S, Sk, K, Hi, S + Sk, full)
    live = ids >= 0
    a = torch.where(live, g.double() * ksc.double()[ids.clamp(min=0).long()], torch.zeros(()).double())
    m = (r > 0).double()
    wq = w.double()[:, :, None] * q8.double()
    rk, rk_abs = torch.zeros(Sk, 128).double(), torch.zeros(Sk, 128).double()
    flat = ids.clamp(min=0).long().flatten()
    rk.index_add_(0, flat, (a[:, :, None] * (m.transpose(1, 2) @ wq)).flatten(0, 1))
    rk_abs.index_add_(0, flat, (a.abs()[:, :, None] * (m.transpose(1, 2) @ wq.abs())).flatten(0, 1))
    rq = w.double()[:, :, None] * ((a[:, None, :] * m) @ k)
    rw = (a[:, None, :] * r.clamp(min=0)).sum(2)
    d_q, d_k, d_w = _grads(gpu, g, q8, k8, ksc, w, ids, 1)
    assert (d_q - rq).abs().max() <= 1e-4 * rq.abs().max() and (d_w - rw).abs().max() <= 1e-4 * rw.abs().max()
    # w q is rounded to bf16 (half a step: 2^-9); everything behind it is 32-bit sums of at most 64 S terms
    assert ((d_k - rk).abs() <= (2.0 ** -9 + 1e-5) * rk_abs + 1e-30).all()
    again = _grads(gpu, g, q8, k8, ksc, w, ids, 1)
    assert torch.equal(d_q, again[0]) and torch.equal(d_k, again[1]) and torch.equal(d_w, again[2])


def test_key_gradients_by_key_tiles_of_values_that_are_not_finite(gpu):
    """An infinite weight or factor, a NaN: the keys that the query selected get them, no others do - as with a row per pair."""
    g, q8, k8, ksc, w, ids, _, _ = _pairs(1600, 4500, 128, 64, 3, 1.0)
    w[17, 5], w[900, 0], g[1200, 3], g[1300, 4] = float("inf"), float("nan"), float("inf"), float("nan")
    g[900, 7] = g[17, 9] = 0.0
    rows, tiles = _grads(gpu, g, q8, k8, ksc, w, ids, 0), _grads(gpu, g, q8, k8, ksc, w, ids, 1)
    for a, b in zip(rows, tiles):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b)) and not torch.isfinite(a).all()
    fin = torch.isfinite(rows[1])
    assert fin.any() and (rows[1] - tiles[1])[fin].norm() <= 1e-2 * rows[1][fin].norm()


def test_key_gradients_by_key_tiles_with_a_repeated_id(gpu):
    g, q8, k8, ksc, w, ids, _, _ = _pairs(1600, 4500, 128, 32, 4, 1.0)
    ids[1599, 100] = ids[1599, 3]
    assert torch.isnan(_grads(gpu, g, q8, k8, ksc, w, ids, 1)[1]).all()


@pytest.mark.parametrize("Hi", [32, 64])
def test_key_gradients_where_the_number_of_heads_decides(gpu, Hi):
    """900 visible keys: whole key tiles for 32 heads, rows for 64, whose sums are the same bits with and without a span."""
    g, q8, k8, ksc, w, ids, _, _ = _pairs(1600, 4500, 128, Hi, 5, 1.0)
    rows, chosen = _grads(gpu, g, q8, k8, ksc, w, ids, 0), _grads(gpu, g, q8, k8, ksc, w, ids, 900)
    for a, b in zip(rows, chosen):
        assert (a - b).norm() <= 1e-2 * a.norm()       # the rows' bf16 pairs, as in the comparisons above
    assert torch.equal(rows[1], chosen[1]) == (Hi == 64)
