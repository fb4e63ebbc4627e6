"""GPU parity of the fused KL indexer loss (softmax + F.kl_div + backward in one kernel) against the
oracle's restatement of dsa_fused.py:931-944 and torch autograd through it."""
import pytest
import torch
import torch.nn.functional as F

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu


def _case(S, K, seed, pad_from=None, target_kind="dist"):
    g = torch.Generator().manual_seed(seed)
    sc = torch.randn(S, K, generator=g) * 3.0
    tg = torch.rand(S, K, generator=g)
    if pad_from is not None:                         # rows with fewer than K valid slots: score -inf, target 0 behind them
        for i in range(S):
            n = int(pad_from[i])
            sc[i, n:] = float("-inf")
            tg[i, n:] = 0.0
    if target_kind == "dist":
        tg = tg / tg.sum(-1, keepdim=True)
    elif target_kind == "onehot":
        tg = F.one_hot(torch.randint(0, K if pad_from is None else 1, (S,), generator=g), K).float()
    return sc, tg


@pytest.mark.parametrize("S,K,padded,kind", [(37, 64, False, "dist"), (130, 2048, True, "dist"), (9, 200, True, "dist"),
                                             (5, 4096, False, "onehot"), (3, 8192, True, "dist"), (1, 1, False, "dist"),
                                             # a row to a wave up to 512 slots, four slots a thread up to 1024
                                             (6, 256, True, "dist"), (7, 257, False, "onehot"), (5, 512, True, "dist"),
                                             (9, 513, True, "dist"), (5, 1024, True, "dist"), (6, 1025, True, "dist")])
def test_kl_loss_and_gradient_match_the_oracle(gpu, S, K, padded, kind):
    from loongforge_amd import ops

    pad = torch.randint(1, K + 1, (S,), generator=torch.Generator().manual_seed(3)) if padded else None
    sc, tg = _case(S, K, seed=S + K, pad_from=pad, target_kind=kind)
    ref_sc = sc.double().requires_grad_(True)
    ref = O.indexer_kl_loss(ref_sc, tg.double(), 1.0, 1)       # coeff 1, norm 1: the plain "sum" reduction
    # the oracle computes in float: redo it in double for the comparison below
    pred = torch.softmax(ref_sc, -1)
    u = tg.double() + 1e-10
    ref64 = (u * (u.log() - (pred + 1e-10).log())).sum()
    ref64.backward()
    got_sc = sc.to(gpu).requires_grad_(True)
    loss = ops.indexer_kl_loss(got_sc, tg.to(gpu))
    (loss * 0.5).backward()                                     # an upstream factor must reach the gradient
    # float arithmetic against double: tolerance 1e-5 relative to the loss / the largest gradient of a row
    assert abs(loss.item() - ref64.item()) <= 1e-5 * max(1.0, abs(ref64.item())), (loss.item(), ref64.item())
    assert abs(ref.item() - ref64.item()) <= 1e-3 * max(1.0, abs(ref64.item()))
    gref = ref_sc.grad * 0.5
    err = (got_sc.grad.double().cpu() - gref).abs().max().item()
    assert err <= 1e-5 * max(1.0, gref.abs().max().item()), err
    if padded:
        assert (got_sc.grad.cpu()[sc == float("-inf")] == 0).all()


def test_kl_loss_equals_f_kl_div_and_vanishes_for_equal_distributions(gpu):
    from loongforge_amd import ops

    sc, tg = _case(64, 512, seed=11)
    want = F.kl_div((torch.softmax(sc, -1) + 1e-10).log(), tg + 1e-10, reduction="sum")
    got = ops.indexer_kl_loss(sc.to(gpu), tg.to(gpu))
    assert abs(got.item() - want.item()) <= 1e-4 * abs(want.item())
    # identical distributions: loss ~ 0 and zero gradient
    s2 = sc.to(gpu).requires_grad_(True)
    same = torch.softmax(sc, -1).to(gpu)
    l2 = ops.indexer_kl_loss(s2, same)
    l2.backward()
    assert abs(l2.item()) < 1e-4 and s2.grad.abs().max().item() < 1e-5
    # a sliced (strided) target, as the attention module hands it over
    wide = torch.cat([tg, torch.zeros(64, 64)], -1).to(gpu)
    got3 = ops.indexer_kl_loss(sc.to(gpu), wide[:, :512])
    assert got3.item() == got.item()


@pytest.mark.parametrize("S,K", [(1, 1), (3, 65), (1025, 64), (5000, 131)])
def test_scaled_sum_and_its_gradient(gpu, S, K):
    """The loss times a factor and its gradient in a launch each: the sum within S half-ulps of 64 bits, the gradient's bits those of the
    product with (g * factor); with a graph of the backward the tensor operations."""
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(S)
    scores = torch.randn(S, K, generator=g).to(gpu).requires_grad_(True)
    target = torch.softmax(torch.randn(S, K, generator=g), -1).to(gpu)
    rows, grad = ops._kl_loss_op(scores.detach(), target, 1e-10)
    up = torch.tensor(1.7, device=gpu)
    loss = ops.indexer_kl_loss(scores, target, 1e-10, 0.37)
    want = rows.double().sum().item() * 0.37
    assert loss.shape == () and abs(loss.item() - want) <= (S + 1) * 2.0 ** -24 * rows.double().abs().sum().item() * 0.37 + 1e-12
    (got,) = torch.autograd.grad(loss, scores, up, retain_graph=True)
    assert torch.equal(got, grad * (up * 0.37))
    (again,) = torch.autograd.grad(loss, scores, up, create_graph=True)
    assert torch.equal(again, got)


@pytest.mark.parametrize("S,step", [(1, 1), (63, 1), (1024, 64), (1025, 1024), (8191, 64), (8193, 1024), (32768, 1024)])
def test_sum_of_the_rows_losses_is_rounded_once(gpu, S, step):
    """Sums in 64 bits: the result is half an ulp from the exact one and no more, also for rows that a chain of 32-bit additions over a
    thread's values or over the waves loses one by one behind the first (0.9 times half its ulp each)."""
    from loongforge_amd import ops

    rows = torch.zeros(S)
    rows[::step] = 0.9 * 2.0 ** -24
    rows[0] = 1.0
    for x in (rows, torch.rand(S, generator=torch.Generator().manual_seed(S))):
        want = x.double().sum()
        got = ops._native().kl_total(x.to(gpu), 1.0).cpu()
        assert got == want.float() or abs(got.double() - want) <= (2.0 ** -24 + S * 2.0 ** -52) * want


@pytest.mark.parametrize("S,H,K", [(1, 4, 1), (5, 3, 200), (9, 16, 256), (7, 16, 264), (33, 64, 512), (6, 8, 1000), (5, 32, 2048), (3, 2, 2500)])
def test_distribution_and_targets_in_bf16(gpu, S, H, K):
    """The kernels that round the distribution to the logits' bf16 and that read bf16 targets have the bits of the conversions beside
    them, with rows at a stride too."""
    from loongforge_amd import ops
    from loongforge_amd.dsa_fused_kernels import triton_attn_dist

    gen = torch.Generator().manual_seed(K)
    p = torch.randn(S, H, K, generator=gen).to(torch.bfloat16)
    p[:, :, K // 2:][torch.rand(S, H, K - K // 2, generator=gen) < 0.1] = float("-inf")
    p = p.to(gpu)
    target = triton_attn_dist(p, 0.3)
    assert target.dtype == torch.bfloat16 and torch.equal(target, ops.attn_dist(p, 0.3).to(torch.bfloat16))
    assert triton_attn_dist(p.float(), 0.3).dtype == torch.float32
    scores = torch.randn(S, K, generator=gen).to(gpu)
    wide = torch.nn.functional.pad(target, (0, 3))
    for t in (target, wide[:, :K]):
        got, want = ops._kl_loss_op(scores, t, 1e-10), ops._kl_loss_op(scores, t.float(), 1e-10)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("S,K", [(1, 3), (7, 1), (9, 256), (5, 700)])
def test_targets_in_bf16_of_any_strides(gpu, S, K):
    """One row for all queries, rows that overlap, columns of a wider tensor and a transposed one: what their copies give."""
    from loongforge_amd import ops

    gen = torch.Generator().manual_seed(S + K)
    scores = torch.randn(S, K, generator=gen).to(gpu)
    base = torch.softmax(torch.randn(S * (K + 2), generator=gen), 0).to(torch.bfloat16).to(gpu)
    for target in (base[:K].expand(S, K), base.as_strided((S, K), (1, 1)), base.view(S, K + 2)[:, 1:K + 1], base[:S * K].view(K, S).t(),
                   base.as_strided((S, K), (2, 2)) if S * 2 + K * 2 < base.numel() else base[:K].expand(S, K)):
        got, want = ops._kl_loss_op(scores, target, 1e-10), ops._kl_loss_op(scores, target.contiguous(), 1e-10)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    if S > 1 and K > 1:                                             # in fp32 such rows are refused, as ever
        with pytest.raises((RuntimeError, ValueError)):
            ops._kl_loss_op(scores, base.float()[:K].expand(S, K), 1e-10)


@pytest.mark.parametrize("factor", [1.0, 1.5 / 40, -3.7])
def test_scaled_gradient_through_the_c_abi(gpu, factor):
    """The gradients of the plain call times the factor, rounded once more; the rows' losses without it."""
    from loongforge_amd import _lib

    lib, S, K = _lib.load(), 33, 300
    gen = torch.Generator().manual_seed(5)
    scores, target = torch.randn(S, K, generator=gen).to(gpu), torch.softmax(torch.randn(S, K, generator=gen), -1).to(gpu)
    results = []
    for scaled in (False, True):
        loss, grad = torch.full((S,), 7.0, device=gpu), torch.full((S, K), 7.0, device=gpu)
        out, stream = (loss.data_ptr(), grad.data_ptr()), torch.cuda.current_stream().cuda_stream
        if scaled:
            rc = lib.dsa_indexer_kl_loss_scaled(scores.data_ptr(), K, target.data_ptr(), 0, K, S, K, 1e-10, factor, *out, stream)
        else:
            rc = lib.dsa_indexer_kl_loss(scores.data_ptr(), K, target.data_ptr(), K, S, K, 1e-10, *out, stream)
        assert rc == 0, lib.dsa_last_error()
        results.append((loss, grad))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1] * factor, results[1][1])
