"""GPU parity: quantiser, indexer logits, top-k (through the C ABI via loongforge_amd.ops)."""
import pytest
import torch

from oracle import dsa_oracle as O
from tests.gpu_util import valid_sets_equal_up_to_noise

pytestmark = pytest.mark.gpu


def _quant_pair(iq, ik, dev):
    from loongforge_amd import ops

    q8, qs = ops.quant_rowwise_e4m3(iq.to(dev))
    k8, ks = ops.quant_rowwise_e4m3(ik.to(dev))
    return q8, qs, k8, ks


def test_quantiser_is_bit_exact(gpu):
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(3)
    x = (torch.randn(2000, 128, generator=g) * torch.logspace(-10, 6, 2000).unsqueeze(-1)).to(torch.bfloat16)
    x[7] = 0
    x[8, 0] = 3.5            # amax exactly on a power-of-two boundary of 448/amax
    x[9, 0] = 3.515625
    x[10, 3] = float(torch.finfo(torch.bfloat16).max)
    r8, rs = O.quant_rowwise_e4m3(x)
    x8, si = ops.quant_rowwise_e4m3(x.to(gpu))
    assert torch.equal(x8.view(torch.uint8).cpu(), r8.view(torch.uint8))
    assert torch.equal(si.cpu(), rs)
    assert si[7].item() == 2.0 ** -48
    # 3-D input (tokens, heads, 128) quantises per (token, head) row
    y = torch.randn(33, 5, 128, generator=g).to(torch.bfloat16)
    y8, ys = ops.quant_rowwise_e4m3(y.to(gpu))
    r8, rs = O.quant_rowwise_e4m3(y)
    assert ys.shape == (33, 5) and torch.equal(y8.view(torch.uint8).cpu(), r8.view(torch.uint8)) and torch.equal(ys.cpu(), rs)
    with pytest.raises(ValueError):
        ops.quant_rowwise_e4m3(torch.zeros(4, 64, dtype=torch.bfloat16, device=gpu))


@pytest.mark.parametrize("S,Hi,K,cu,seed", [
    (200, 64, 64, None, 42),
    (333, 32, 128, None, 5),
    (512, 64, 64, [0, 100, 101, 300, 512], 9),
    (70, 64, 128, None, 11),          # every row has fewer than K visible keys
])
def test_logits_and_topk_against_oracle(gpu, S, Hi, K, cu, seed):
    from loongforge_amd import ops

    cu_t = torch.tensor(cu, dtype=torch.int32) if cu else None
    iq, ik, w = O.make_indexer_inputs(S, Hi, 128, seed=seed)
    sc_ref, idx_ref, aux = O.indexer_forward(iq, ik, w, K, 0, cu_t, dtype=torch.float64)
    q8, qs, k8, ksc = _quant_pair(iq, ik, gpu)
    assert torch.equal(q8.view(torch.uint8).cpu(), aux["q8"].view(torch.uint8))
    ws = (w.to(gpu) * qs * 128 ** -0.5).contiguous()
    ks, ke = aux["ks"].to(gpu), aux["ke"].to(gpu)

    logits = ops.indexer_logits(q8, ws, k8, ksc, ks, ke)
    L, R = logits.cpu(), aux["logits"]
    fin = torch.isfinite(R)
    assert torch.equal(torch.isfinite(L), fin)                      # -inf exactly outside [ks, ke)
    # 64 signed terms of magnitude ~|w'| * |q.k| cancel; fp32 noise is relative to the term size
    noise = 1e-4 * R[fin].abs().max().item()
    assert (L[fin].double() - R[fin]).abs().max().item() <= noise

    for srt in (True, False):
        sc, ids = ops.topk(logits, K, ks, ke, None, sorted=srt)
        v2, _ = O.topk_select(L, K)                                  # library routine on the same logits
        scc, idc = sc.cpu(), ids.cpu()
        if srt:
            assert torch.equal(scc, v2)
        else:
            assert torch.equal(torch.sort(scc, descending=True).values, v2)
            big = torch.where(idc >= 0, idc, torch.full_like(idc, 1 << 30)).long()
            assert (torch.diff(big, dim=1) >= 0).all()             # ascending column order
        got = torch.where(idc >= 0, L.gather(1, idc.clamp(min=0).long()), torch.full_like(scc, float("-inf")))
        assert torch.equal(got, scc)                                # slot t of scores and ids stay aligned
        for i in range(S):
            a = idc[i][idc[i] >= 0]
            assert a.numel() == len(set(a.tolist())) == min(K, int(ke[i] - ks[i]))
            assert (a >= int(ks[i])).all() and (a < int(ke[i])).all()

    sc, ids = ops.indexer_topk(q8, ws, k8, ksc, ks, ke, K)
    assert valid_sets_equal_up_to_noise(ids, idx_ref, R, band=2 * noise) == 0


def test_topk_is_bit_exact_when_the_arithmetic_is_exact(gpu):
    """Small-integer payloads, unit scales and power-of-two weights make every product and sum
    exact in fp32, so the selected sets must equal the oracle's with no tolerance band (scores are
    made distinct so that there are no ties at the boundary)."""
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(0)
    S, Hi, K = 300, 32, 64
    q = torch.randint(-3, 4, (S, Hi, 128), generator=g).float()
    k = torch.randint(-3, 4, (S, 128), generator=g).float()
    w = torch.full((S, Hi), 2.0 ** -4)
    k[:, 0] = 0
    q8, k8 = q.to(torch.float8_e4m3fn), k.to(torch.float8_e4m3fn)
    ksc = torch.ones(S) + torch.arange(S) * 2.0 ** -12              # distinct, exactly representable scales
    ks, ke = O.indexer_window(S, 0)
    R = O.indexer_logits(q8, w, k8, ksc, ks, ke, dtype=torch.float64)
    L = ops.indexer_logits(q8.to(gpu), w.to(gpu), k8.to(gpu), ksc.to(gpu), ks.to(gpu), ke.to(gpu)).cpu()
    fin = torch.isfinite(R)
    assert torch.equal(L[fin].double(), R[fin])
    sc, ids = ops.indexer_topk(q8.to(gpu), w.to(gpu), k8.to(gpu), ksc.to(gpu), ks.to(gpu), ke.to(gpu), K)
    vref, iref = O.topk_select(R.float(), K)
    assert torch.equal(sc.cpu(), vref)
    for i in range(S):
        row = vref[i][vref[i] > float("-inf")]
        if row.numel() == K and (R[i, : i + 1] == row.min().item()).sum() > 1:
            continue                                                # an exact tie at the K-th value
        assert set(ids[i][ids[i] >= 0].tolist()) == set(iref[i][iref[i] >= 0].tolist())


def test_padded_flashinfer_topk_wrapper(gpu):
    from loongforge_amd.dsa_fused_kernels import padded_flashinfer_topk

    g = torch.Generator().manual_seed(1)
    logits = torch.randn(10, 20, generator=g)
    vals, idx = padded_flashinfer_topk(logits.to(gpu), 5, 20)
    rv, ri = torch.topk(logits, 5)
    assert torch.equal(vals.cpu(), rv) and torch.equal(idx.cpu().long(), ri)
    vals, idx = padded_flashinfer_topk(logits.to(gpu), 25, 20)
    assert vals.shape == (10, 25) and torch.isinf(vals[:, 20:]).all() and (idx[:, 20:] == 20).all()
    assert torch.equal(vals[:, :20].cpu(), torch.sort(logits, descending=True).values)


def test_relative_layout_of_packed_logits(gpu):
    from loongforge_amd import ops

    cu = torch.tensor([0, 40, 41, 128], dtype=torch.int32)
    iq, ik, w = O.make_indexer_inputs(128, 64, 128, seed=3)
    _, _, aux = O.indexer_forward(iq, ik, w, 16, 0, cu)
    q8, qs, k8, ksc = _quant_pair(iq, ik, gpu)
    ws = (w.to(gpu) * qs * 128 ** -0.5).contiguous()
    ks, ke = aux["ks"].to(gpu), aux["ke"].to(gpu)
    dense = ops.indexer_logits(q8, ws, k8, ksc, ks, ke).cpu()
    rel = ops.indexer_logits(q8, ws, k8, ksc, ks, ke, width=87, relative=True).cpu()
    for i in range(128):
        n = int(ke[i] - ks[i])
        assert torch.equal(rel[i, :n], dense[i, int(ks[i]): int(ke[i])])
        assert torch.isinf(rel[i, n:]).all()


@pytest.mark.parametrize("kind", ["normal", "ties", "constant", "outlier", "holes", "short", "two_values", "plus_inf"])
@pytest.mark.parametrize("K,sorted_out", [(2048, True), (1000, True), (256, True), (512, False)])
def test_topk_rule_on_crafted_rows(gpu, kind, K, sorted_out):
    """The selection rule on rows that exercise every branch of the kernel: the K largest values, ties
    broken towards the smaller column, output in descending score / ascending column order.  The
    expectation is a stable sort by the library routine."""
    from loongforge_amd import ops

    n, rows = 6001, 12                                    # odd width: row starts at every 4-byte alignment
    g = torch.Generator().manual_seed(5)
    x = torch.randn(rows, n, generator=g)
    if kind == "ties":
        x = torch.round(x * 8) / 8                        # a few dozen distinct values
    elif kind == "constant":
        x = torch.full((rows, n), 1.25)
    elif kind == "outlier":
        x[:, 17] = 1e30                                   # every other value lands in the last value bins
        x[:, 99] = -1e30
    elif kind == "holes":
        x[torch.rand(rows, n, generator=g) < 0.3] = float("-inf")
    elif kind == "two_values":
        x = (x > 0.5).float()
    elif kind == "plus_inf":
        x[:, 5] = float("inf")                            # +inf is the largest value, as for torch.topk
        x[::2, 4000] = float("inf")
    end = torch.full((rows,), n, dtype=torch.int32)
    if kind == "short":
        end = torch.tensor([1, 2, 63, 64, 255, 256, 257, 999, 1000, 1001, 2047, 2049], dtype=torch.int32)
    beg = torch.zeros(rows, dtype=torch.int32) if kind == "short" else (torch.arange(rows, dtype=torch.int32) % 5)
    sc, ids = ops.topk(x.to(gpu), K, beg.to(gpu), end.to(gpu), sorted=sorted_out)
    sc, ids = sc.cpu(), ids.cpu()
    for i in range(rows):
        row = x[i, : int(end[i])].clone()
        row[: int(beg[i])] = float("-inf")                  # columns before the window cannot be selected
        order = torch.sort(-row, stable=True).indices      # descending value, ascending column among equals
        fin = row[order] > float("-inf")                    # only -inf marks a column that cannot be selected
        exp_ids = order[fin][:K]
        kk = len(exp_ids)
        if sorted_out:
            assert torch.equal(ids[i, :kk].long(), exp_ids), (kind, K, i)
            assert torch.equal(sc[i, :kk], row[exp_ids])
        else:
            got = ids[i][ids[i] >= 0].long()
            assert torch.equal(torch.sort(got).values, torch.sort(exp_ids).values), (kind, K, i)
            assert torch.equal(sc[i][ids[i] >= 0], row[got])
        assert (ids[i, kk:] == -1).all() and torch.isinf(sc[i, kk:]).all() and (sc[i, kk:] < 0).all()


def test_topk_on_full_width_rows_at_every_alignment(gpu):
    """Rows of the widest size the register-resident path takes (8192), starting 0..3 elements past a
    16-byte boundary."""
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(11)
    buf = torch.randn(4 * 8192 + 3, generator=g).to(gpu)
    for off in range(4):
        x = buf[off: off + 4 * 8192].view(4, 8192)
        assert x.data_ptr() % 16 == 4 * off
        sc, ids = ops.topk(x, 2048)
        ref = torch.sort(-x.cpu(), stable=True, dim=-1).indices[:, :2048]
        assert torch.equal(ids.cpu().long(), ref)
        assert torch.equal(sc.cpu(), torch.gather(x.cpu(), 1, ref))


@pytest.mark.parametrize("copies", [1, 80])             # at most 256 rows: 1024 threads a row; more: 256
@pytest.mark.parametrize("n,K", [(1021, 64), (1022, 1000), (2045, 64), (2046, 2048), (4090, 2048), (8189, 512)])
def test_topk_segments_of_equal_values(gpu, copies, n, K):
    """Bins that hold 1 .. 256 elements, and a bin at the K-th place with as many as the buffer has room for and one more: each
    element's place among its bin's, on both sides of the lengths at which a row takes more registers."""
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(n + K)
    rows = []
    for run in (1, 3, 4, 5, 8, 255, 256, 257, 959, 960, 961):
        x = torch.rand(n, generator=g)
        at = torch.randperm(n, generator=g)
        run = min(run, n - 2)
        first = min(max(K - run // 2, 0), n - run)                  # the K-th largest value lies in the run, or the run at the end
        order = torch.argsort(-x, stable=True)
        x[order[first: first + run]] = x[order[first]].item()
        x[at[:4]] = x[at[0]].item()
        rows.append(x)
    x = torch.stack(rows).repeat(copies, 1)
    sc, ids = ops.topk(x.to(gpu), K)
    ref = torch.sort(-x, stable=True, dim=-1).indices[:, :K]
    kk = min(n, K)
    assert torch.equal(ids.cpu().long()[:, :kk], ref[:, :kk])
    assert torch.equal(sc.cpu()[:, :kk], torch.gather(x, 1, ref)[:, :kk])
    assert (ids.cpu()[:, kk:] == -1).all()


@pytest.mark.parametrize("span", [2.0 ** -149, 1e-44, 1e-40, 1e-38, 2e-36, 1.1e-35, 1.3e-35, 1e-34])
@pytest.mark.parametrize("copies,n,K", [(1, 300, 64), (1, 6000, 2048), (300, 300, 512), (300, 2000, 64), (300, 8000, 512)])
def test_topk_of_values_close_to_one_another(gpu, copies, n, K, span):
    """Rows whose bins would be narrower than what 32 bits hold, on both sides of the line (4095.5 / span), of either sign and with one
    value beside equal ones; the general path takes them."""
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(n + K)
    a = torch.rand(n, generator=g, dtype=torch.float64)
    x = torch.stack([((a + 1) * span).float(), (-(a + 1) * span).float(), torch.zeros(n), torch.full((n,), -0.0), ((a + 1) * span).float()])
    x[2, n // 3], x[3, n // 2] = span, -span
    x[4, n // 4] = -torch.inf                            # (the form for values that are not finite)
    assert x[0].max() > x[0].min()
    sc, ids = ops.topk(x.repeat(copies, 1).to(gpu), K)
    ref = torch.sort(-x, stable=True, dim=-1).indices[:, :K]
    kk = min(n - 1, K)
    for row in (slice(0, 5), slice(5 * copies - 5, None)):
        assert torch.equal(ids[row, :kk].cpu().long(), ref[:, :kk])
        assert torch.equal(sc[row, :kk].cpu(), torch.gather(x, 1, ref)[:, :kk])


def test_fused_rotation_and_quantiser(gpu):
    """rotate_quant_e4m3 against the unfused sequence rotate_activation -> quantiser: the rotated bf16
    values agree to one bf16 step (the fp32 sums are taken in a different order), payload and scale
    are exactly the quantisation of the kernel's own rotated values, and the rotation is an involution."""
    from loongforge_amd import ops
    from loongforge_amd.dsa_fused import rotate_activation

    g = torch.Generator().manual_seed(3)
    x = torch.randn(1000, 7, 128, generator=g).to(torch.bfloat16)
    x[5] = 0
    xd = x.to(gpu)
    x8, sinv, y = ops.rotate_quant_e4m3(xd, return_rotated=True)
    ref = rotate_activation(x)                                       # fp32 product with the Hadamard matrix on the CPU
    err = (y.cpu().float() - ref.float()).abs()
    assert (err <= 2.0 ** -7 * ref.float().abs() + 1e-30).all()      # at most one bf16 step
    assert (err == 0).float().mean().item() > 0.98
    r8, rs = O.quant_rowwise_e4m3(y.cpu())
    assert torch.equal(x8.cpu().view(torch.uint8), r8.view(torch.uint8)) and torch.equal(sinv.cpu(), rs)
    x8b, sinvb = ops.rotate_quant_e4m3(xd)
    assert torch.equal(x8b.view(torch.uint8), x8.view(torch.uint8)) and torch.equal(sinvb, sinv)
    assert torch.equal(ops.rotate_bf16(xd), y)
    back = ops.rotate_bf16(y).float().cpu()                          # H.H = 128 I: rotating twice returns x
    assert (back - x.float()).abs().max().item() <= 2.0 ** -6 * x.float().abs().max().item()


def test_quantiser_with_weight_scaling_equals_the_separate_operations(gpu):
    """The quantiser kernel that also emits weights * scale_inv * factor: payload and scales are those
    of the plain kernel, the scaled weights are bit-equal to the two torch multiplications."""
    from loongforge_amd import ops

    iq, _, w = O.make_indexer_inputs(300, 64, 128, seed=3)
    x, wd = iq.to(gpu), w.to(gpu)
    for rotate in (False, True):
        plain = ops.rotate_quant_e4m3(x) if rotate else ops.quant_rowwise_e4m3(x)
        x8, si, ws = ops.quant_rowwise_e4m3_weights(x, wd, 128 ** -0.5, rotate)
        assert torch.equal(x8.view(torch.uint8), plain[0].view(torch.uint8)) and torch.equal(si, plain[1])
        assert torch.equal(ws, wd * si * 128 ** -0.5)
    with pytest.raises(ValueError):
        ops.quant_rowwise_e4m3_weights(x, wd[:, :32], 1.0)


def test_indexer_kernel_with_fused_rotation_matches_rotating_first(gpu):
    """DSAIndexerKernel(rotate=True) == DSAIndexerKernel on pre-rotated inputs: same scores and ids, and
    gradients that agree with autograd through rotate_activation."""
    from loongforge_amd.dsa_fused import rotate_activation
    from loongforge_amd.dsa_fused_kernels import DSAIndexerKernel

    S, Hi, K = 512, 64, 128
    iq, ik, w = O.make_indexer_inputs(S, Hi, 128, seed=11)
    kern = DSAIndexerKernel()
    q1, k1, w1 = (t.to(gpu).requires_grad_(True) for t in (iq, ik, w))
    sc1, id1 = kern(q1, k1, w1, K, 0, None, rotate=True)
    q2, k2, w2 = (t.to(gpu).requires_grad_(True) for t in (iq, ik, w))
    sc2, id2 = kern(rotate_activation(q2), rotate_activation(k2), w2, K, 0, None)
    fin = torch.isfinite(sc2)
    assert torch.equal(torch.isfinite(sc1), fin)
    # a bf16 step in a few rotated values moves a logit by a few 1e-3 of the row's scale
    tol = 5e-3 * sc2[fin].abs().max().item()
    assert (sc1[fin] - sc2[fin]).abs().max().item() <= tol
    same = (torch.sort(id1, 1).values == torch.sort(id2, 1).values).float().mean().item()
    assert same > 0.99
    gsc = torch.randn(S, K, generator=torch.Generator().manual_seed(12)).to(gpu)
    torch.where(fin, sc1, torch.zeros_like(sc1)).mul(gsc).sum().backward()
    torch.where(fin, sc2, torch.zeros_like(sc2)).mul(gsc).sum().backward()
    for a, b in ((q1.grad, q2.grad), (k1.grad, k2.grad), (w1.grad, w2.grad)):
        scale = b.float().abs().max().item()
        assert (a.float() - b.float()).abs().max().item() <= 3e-2 * scale


@pytest.mark.parametrize("copies", [1, 24])       # 13 rows: the 1024-thread kernel; 312 rows: the 256-thread ones
@pytest.mark.parametrize("K", [64, 1000, 2048])
def test_topk_row_lengths_at_the_edges_of_its_variants(gpu, copies, K):
    """Rows whose lengths sit at the register variants' limits, in an array wider than any of them, plus rows of one
    element, of equal values and of repeated values (ties by ascending column)."""
    from loongforge_amd import ops

    lengths = [1, 2, 255, 256, 257, 4093, 4094, 8190, 9213, 9214, 16382, 33789, 33790]
    width = 34000
    g = torch.Generator().manual_seed(K)
    x = torch.randn(len(lengths), width, generator=g)
    x[3] = 0.5
    x[4] = torch.randint(0, 9, (width,), generator=g).float()
    begin = torch.tensor([(7 * i) % 11 for i in range(len(lengths))], dtype=torch.int32)
    end = begin + torch.tensor(lengths, dtype=torch.int32)
    rep = lambda t: t.repeat(copies, *([1] * (t.ndim - 1))).to(gpu)                    # noqa: E731
    sc, ids = ops.topk(rep(x), K, rep(begin), rep(end))
    for i, n in enumerate(lengths):
        row = x[i, int(begin[i]): int(end[i])]
        v, order = torch.sort(row, descending=True, stable=True)
        k = min(K, n)
        for c in range(copies):
            got_s, got_i = sc[c * len(lengths) + i].cpu(), ids[c * len(lengths) + i].cpu()
            assert torch.equal(got_s[:k], v[:k]) and torch.equal(got_i[:k].long(), order[:k] + int(begin[i])), (n, c)
            assert (got_i[k:] == -1).all() and torch.isinf(got_s[k:]).all(), (n, c)


@pytest.mark.parametrize("copies", [1, 45])       # 6 rows: the 1024-thread kernel alone; 270 rows: behind the 256-thread one
@pytest.mark.parametrize("K", [64, 1000, 2048, 4096, 8192])
@pytest.mark.parametrize("sorted_out", [True, False])
def test_topk_of_rows_beyond_the_register_variants(gpu, copies, K, sorted_out):
    """Around the longest row held in registers and beyond it: the general path with the sorting networks, ties by ascending
    column, columns that cannot be selected, fewer of the others than slots."""
    from loongforge_amd import ops

    lengths = [36861, 36862, 41000, 41000, 41000, 41000]
    width = 41003
    g = torch.Generator().manual_seed(K)
    x = torch.randn(len(lengths), width, generator=g)
    x[3] = torch.randint(0, 5, (width,), generator=g).float()
    x[4, ::2] = float("-inf")
    x[5, 700:] = float("-inf")
    begin = torch.tensor([i % 4 for i in range(len(lengths))], dtype=torch.int32)
    end = begin + torch.tensor(lengths, dtype=torch.int32)
    rep = lambda t: t.repeat(copies, *([1] * (t.ndim - 1))).to(gpu)                    # noqa: E731
    sc, ids = ops.topk(rep(x), K, rep(begin), rep(end), sorted=sorted_out)
    sc, ids = sc.view(copies, len(lengths), K), ids.view(copies, len(lengths), K)
    assert all(torch.equal(sc[c], sc[0]) and torch.equal(ids[c], ids[0]) for c in range(copies))
    for i, n in enumerate(lengths):
        row = x[i, int(begin[i]): int(end[i])]
        v, order = torch.sort(row, descending=True, stable=True)
        k = min(K, int(torch.isfinite(row).sum()))
        got_s, got_i = sc[0, i].cpu(), ids[0, i].cpu().long()
        if sorted_out:
            assert torch.equal(got_s[:k], v[:k]) and torch.equal(got_i[:k], order[:k] + int(begin[i])), n
            assert (got_i[k:] == -1).all() and torch.isinf(got_s[k:]).all(), n
        else:                                           # in ascending column order
            want = torch.sort(order[:k])[0]
            live = got_i >= 0
            assert torch.equal(got_i[live], want + int(begin[i])) and torch.equal(got_s[live], row[want]), n
            assert torch.isinf(got_s[~live]).all(), n


@pytest.mark.parametrize("Hi", [32, 64])
def test_logits_of_few_queries_and_unrelated_windows(gpu, Hi):
    """Windows cut into parts over workgroups: shared ones (a chunk behind cached keys), unrelated ones (sequences of a
    batch, some empty), a single query, window ends off every tile boundary."""
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(Hi)
    for ks, ke, sk in (([0], [1], 5), ([3], [1999], 2000), ([0] * 9, list(range(700, 709)), 709),
                       ([0, 40, 40, 171, 900, 901, 1500, 1500, 1777, 0], [40, 40, 171, 899, 901, 1500, 1777, 1501, 1999, 3], 2000)):
        S = len(ks)
        q = torch.randn(S, Hi, 128, generator=g).to(torch.float8_e4m3fn)
        k = torch.randn(sk, 128, generator=g).to(torch.float8_e4m3fn)
        w, sc = torch.randn(S, Hi, generator=g), torch.rand(sk, generator=g)
        a, b = torch.tensor(ks, dtype=torch.int32), torch.tensor(ke, dtype=torch.int32)
        ref = O.indexer_logits(q, w, k, sc, a, b)
        for rel in (False, True):
            got = ops.indexer_logits(q.to(gpu), w.to(gpu), k.to(gpu), sc.to(gpu), a.to(gpu), b.to(gpu), relative=rel).cpu()
            for i in range(S):
                n = max(ke[i] - ks[i], 0)
                row = got[i, :n] if rel else got[i, ks[i]: ks[i] + n]
                want = ref[i, ks[i]: ks[i] + n]
                assert (row - want).abs().max().item() <= 1e-4 * max(want.abs().max().item(), 1.0) if n else True
                assert int(torch.isfinite(got[i]).sum()) == n


@pytest.mark.parametrize("relative", [False, True])
@pytest.mark.parametrize("Hi", [32, 64])
def test_logits_at_the_edges_of_tiles(gpu, Hi, relative):
    """Windows that begin and end around the sub-tiles of 32 keys, their pairs and the tiles of 128, eight related ones to a
    block, in few blocks (cut into parts) and in many; nothing outside a window is written."""
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(Hi)
    edges = [0, 1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 159, 161]
    rows = [(lo, 300 + hi) for lo in edges[::2] for hi in edges[1::2]] + [(lo, lo + n) for n in (1, 32, 33, 64, 65, 96, 128, 160) for lo in edges[::2]]
    sk = 461
    for copies in (1, 9):
        ks, ke = (torch.tensor(x, dtype=torch.int32).repeat(copies) for x in zip(*rows))
        S = ks.numel()
        q = torch.randn(S, Hi, 128, generator=g).to(torch.float8_e4m3fn)
        k = torch.randn(sk, 128, generator=g).to(torch.float8_e4m3fn)
        w, sc = torch.randn(S, Hi, generator=g), torch.rand(sk, generator=g)
        got = ops.indexer_logits(q.to(gpu), w.to(gpu), k.to(gpu), sc.to(gpu), ks.to(gpu), ke.to(gpu), relative=relative).cpu()
        want = O.indexer_logits(q, w, k, sc, ks, ke, dtype=torch.float64)
        # 128 exact products and Hi weighted terms in sums of 32 bits: an ulp each of the sum of the magnitudes
        dot = torch.einsum("ihd,jd->ihj", q.double().abs(), k.double().abs())
        bound = (128 + Hi) * 2.0 ** -24 * torch.einsum("ih,ihj->ij", w.double().abs(), dot) * sc.double()
        for i in range(S):
            lo, hi = int(ks[i]), int(ke[i])
            row = got[i, :hi - lo] if relative else got[i, lo:hi]
            assert ((row - want[i, lo:hi]).abs() <= bound[i, lo:hi]).all(), (copies, i, lo, hi)
            assert int(torch.isfinite(got[i]).sum()) == hi - lo, (copies, i)


@pytest.mark.parametrize("relative", [False, True])
@pytest.mark.parametrize("S", [3, 300])                  # unrelated and shared windows
def test_logits_in_rows_narrower_than_the_windows(gpu, relative, S):
    """Keys that have no column in the row are left out, and nothing is written behind it."""
    from loongforge_amd import _lib, ops

    g = torch.Generator().manual_seed(S)
    sk, width = 700, 333
    q = torch.randn(S, 64, 128, generator=g).to(torch.float8_e4m3fn).to(gpu)
    k = torch.randn(sk, 128, generator=g).to(torch.float8_e4m3fn).to(gpu)
    w, sc = torch.randn(S, 64, generator=g).to(gpu), torch.rand(sk, generator=g).to(gpu)
    ks = torch.tensor([(37 * i) % 400 if S < 10 else i // 8 for i in range(S)], dtype=torch.int32, device=gpu)
    ke = torch.full((S,), sk, dtype=torch.int32, device=gpu)
    full = ops.indexer_logits(q, w, k, sc, ks, ke, relative=relative)
    ld = width + 5
    out = torch.full((S + 1, ld), 7.0, device=gpu)
    _lib.check(_lib.load().dsa_indexer_logits(q.data_ptr(), w.data_ptr(), k.data_ptr(), sc.data_ptr(), ks.data_ptr(), ke.data_ptr(), S, 64, sk,
                                              out.data_ptr(), ld, width, int(relative), torch.cuda.current_stream().cuda_stream), "logits")
    assert torch.equal(out[:S, :width], full[:, :width])
    assert (out[:S, width:] == 7.0).all() and (out[S] == 7.0).all()


@pytest.mark.parametrize("cu,S,offset", [(None, 5, 3), ([0, 7], 7, 0), ([0, 3, 3, 300, 513], 256, 257), ([0, 1, 2, 700], 700, 0)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_windows_and_positions_of_packed_sequences(gpu, cu, S, offset, dtype):
    from loongforge_amd import ops

    like = torch.zeros(1, device=gpu)
    t = torch.arange(offset, offset + S)
    start = torch.zeros(S, dtype=torch.int64)
    if cu is not None:
        bounds = torch.tensor(cu)
        start = bounds[torch.searchsorted(bounds[1:].contiguous(), t, right=True)]
        pos = ops.thd_positions(bounds.to(gpu, dtype), S + 4, offset)
        inside = min(S + 4, cu[-1] - offset)
        assert torch.equal(pos[:S].cpu().long(), t - start) and not pos[inside:].any()
    ks, ke, covered = ops.indexer_window(None if cu is None else torch.tensor(cu, dtype=dtype, device=gpu), S, offset, like)
    covered.wait()
    assert torch.equal(ks.cpu().long(), start) and torch.equal(ke.cpu().long(), t + 1)
    if cu is not None:
        _, _, short = ops.indexer_window(torch.tensor(cu[:-1] + [offset + S - 1], dtype=dtype, device=gpu), S, offset, like)
        with pytest.raises(ValueError, match="inconsistent shapes"):
            short.wait()


def test_packed_sequences_that_end_before_the_queries(gpu):
    """What the windows are where nothing can raise (a launch under capture): none for the queries that no sequence holds.  What
    is refused: sequences that are too short, decreasing lengths, no sequence; no query needs none."""
    import ctypes

    from loongforge_amd import _lib, ops

    like = torch.zeros(1, device=gpu)
    for cu, offset in (([0, 3, 9], 4), ([5, 8, 14], 4), ([0], 0), ([0, 0], 0)):
        ks, ke = (torch.full((300,), 7, dtype=torch.int32, device=gpu) for _ in range(2))
        t = torch.tensor(cu, dtype=torch.int32, device=gpu)
        _lib.check(_lib.load().dsa_indexer_window(t.data_ptr(), 0, len(cu), 300, offset, ks.data_ptr(), ke.data_ptr(), None,
                                                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "window")
        held = max(cu[-1] - cu[0] - offset, 0)
        assert ke[:held].tolist() == list(range(offset + 1, offset + 1 + held)) and (ks[:held] < ke[:held] + cu[0]).all()
        assert not ks[held:].any() and not ke[held:].any()
    for bad, match in (([0, 5, 4, 20], "decrease"), ([0, 9], "9 tokens"), ([0], "no packed sequence"), ([], "no packed sequence")):
        with pytest.raises(ValueError, match=match):
            ops.indexer_window(torch.tensor(bad, dtype=torch.int64, device=gpu), 10, 3, like)[2].wait()
    long = torch.cat((torch.arange(700), torch.tensor([600])))                     # the fall lies behind the first 256 entries
    with pytest.raises(ValueError, match="decrease"):
        ops.indexer_window(long.to(gpu), 10, 3, like)[2].wait()
    ops.indexer_window(torch.tensor([0, 2], device=gpu), 0, 3, like)[2].wait()


def test_native_host_layer_equals_the_registered_ops(gpu):
    """Ordinary calls go through the C++ layer, traced ones and those under a dispatch mode through the custom op."""
    from loongforge_amd import ops
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    logits = torch.randn(3, 500, device=gpu)
    direct = ops.topk(logits, 40)
    with Seen():
        seen = ops.topk(logits, 40)
    assert any("dsa.topk" in n for n in Seen.names) and all(torch.equal(a, b) for a, b in zip(direct, seen))
    x = torch.randn(4, 128, device=gpu).to(torch.bfloat16)
    with FakeTensorMode() as mode:
        x8, scale = ops.quant_rowwise_e4m3(mode.from_tensor(x))
    assert x8.dtype == torch.float8_e4m3fn and scale.shape == (4,)
    with pytest.raises(ValueError, match="2-D fp32"):
        ops.topk(logits.double(), 4)
    with pytest.raises(ValueError, match="dsa_topk"):
        ops.topk(logits, 0)


@pytest.mark.parametrize("S,Sk,heads,rotate,bf16_weights,offset,ratio", [
    (1, 1, 32, True, False, 0, 0),
    (61, 300, 64, True, True, 239, 0),
    (255, 257, 32, False, True, 2, 0),               # windows and rows that end inside a workgroup
    (257, 64, 64, False, False, 0, 4),
    (512, 40, 32, True, True, 100, 15),              # windows beyond the last compressed key are cut there
    (9, 2, 64, False, True, 0, 1000),                # no query has a whole compressed key
])
def test_indexer_inputs_in_one_launch_are_those_of_separate_launches(gpu, S, Sk, heads, rotate, bf16_weights, offset, ratio):
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(S)
    q = torch.randn(S, heads, 128, generator=g).bfloat16().to(gpu)
    k = torch.randn(Sk, 128, generator=g).bfloat16().to(gpu)
    w = torch.randn(S, heads, generator=g).to(torch.bfloat16 if bf16_weights else torch.float32).to(gpu)
    K = min(64, Sk)
    got = ops.indexer_forward(q, k, w, rotate, 0.1, None, offset, K, True, ratio=ratio)
    q8, q_scale, scaled = ops.quant_rowwise_e4m3_weights(q, w.float(), 0.1, rotate)
    k8, k_scale = (ops.rotate_quant_e4m3 if rotate else ops.quant_rowwise_e4m3)(k)
    end = torch.arange(S, device=gpu, dtype=torch.int32) + offset + 1
    if ratio:
        end = torch.div(end, ratio, rounding_mode="floor").clamp(min=1, max=Sk)
    scores, ids = ops.indexer_topk(q8, scaled, k8, k_scale, torch.zeros_like(end), end, K, True)
    for x, y in zip(got, (scores, ids, q8, q_scale, scaled, k8, k_scale)):
        x, y = (t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t for t in (x, y))
        assert x.dtype == y.dtype and torch.equal(x, y)
    assert got[7] is None
