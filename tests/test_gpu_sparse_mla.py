"""GPU parity: sparse MLA forward / backward and the attention distribution."""
import pytest
import torch

from oracle import dsa_oracle as O
from tests.gpu_util import MLA_FORMS, REF_DKV_EXCESS_LIMIT, assert_close, assert_mla_grads, mla_bwd_with_groups, mla_form

pytestmark = pytest.mark.gpu


def _run_fwd(inp, dev, q_start=0, p_out=False, p_dtype=torch.bfloat16):
    from loongforge_amd import ops

    return ops.sparse_mla_fwd(inp.q.to(dev), inp.kv.to(dev), inp.idx.to(dev), q_start, inp.sm_scale, 512, p_out, p_dtype)


@pytest.mark.parametrize("S,H,K,q_start,skv,seed", [
    (64, 128, 64, 0, None, 0),
    (300, 128, 128, 17, None, 1),
    (256, 64, 256, 0, None, 2),
    (130, 32, 192, 5, 400, 3),
])
def test_forward_against_oracle(gpu, S, H, K, q_start, skv, seed):
    inp = O.make_mla_inputs(S, H, K, seed=seed, skv=skv, q_start=q_start)
    out, lse, _ = _run_fwd(inp, gpu, q_start)
    ro, rl, _ = O.sparse_mla_fwd(inp.q, inp.kv, inp.idx, q_start, inp.sm_scale, 512)
    assert_close(out, ro, "out")
    assert (lse.cpu() - rl).abs().max().item() < 1e-4


@pytest.mark.parametrize("K", [4096, 8192])
def test_top_k_beyond_2048(gpu, K):
    """Wider slot lists: the forward of a few queries shares them out in ranges; the backward and the recomputed attention
    distribution take 2048 / 4096 slots per call and the host walks the list in parts (the gradients are sums over the
    slots once lse and out of the whole list are given)."""
    from loongforge_amd import ops

    skv = K + 1500
    inp = O.make_mla_inputs(48, 64, K, seed=11, skv=skv, q_start=skv - 48)
    out, lse, _ = _run_fwd(inp, gpu, skv - 48)
    ro, rl, _ = O.sparse_mla_fwd(inp.q, inp.kv, inp.idx, skv - 48, inp.sm_scale, 512)
    assert_close(out, ro, "out")
    assert (lse.cpu() - rl).abs().max().item() < 1e-4
    q, kv, ids, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, ids, lse, skv - 48, inp.sm_scale)
    rdq, rdkv = O.sparse_mla_bwd(inp.q, inp.kv, inp.idx, inp.dout, skv - 48, inp.sm_scale, 512)
    assert_close(dq, rdq, "dq")
    assert_close(dkv, rdkv, "dkv")             # 48 queries: few rows per key, the bf16 rows stay inside the bound
    dist = ops.attn_dist_qk(q, kv, ids, lse, skv - 48, inp.sm_scale, 64)
    ref = O.attn_dist_from_lse(inp.q, inp.kv, inp.idx, rl, skv - 48, inp.sm_scale, 64)
    assert (dist.cpu() - ref).abs().max().item() <= 2e-5


def test_forward_p_out_and_attn_dist(gpu):
    from loongforge_amd import ops
    from loongforge_amd.dsa_fused_kernels import triton_attn_dist

    inp = O.make_mla_inputs(200, 128, 128, seed=4)
    _, _, rp = O.sparse_mla_fwd(inp.q, inp.kv, inp.idx, 0, inp.sm_scale, 512)
    for dt in (torch.float32, torch.bfloat16):
        _, _, p = _run_fwd(inp, gpu, 0, True, dt)
        assert p.dtype == dt and p.shape == (200, 128, 128)
        fin = torch.isfinite(rp)
        assert torch.equal(torch.isfinite(p.float().cpu()), fin)          # -inf exactly on invalid slots
        tol = 2e-4 if dt == torch.float32 else 0.26                         # bf16 ulp of |logit| < 64
        assert (p.float().cpu()[fin] - rp[fin]).abs().max().item() < tol
        tgt = ops.attn_dist(p, inp.sm_scale)
        ref = O.attn_dist(rp, inp.sm_scale)
        assert (tgt.cpu() - ref).abs().max().item() < (1e-5 if dt == torch.float32 else 6e-3)
        assert (tgt.sum(-1).cpu() - 1).abs().max().item() < 1e-4
        # head-sliced view (what the attention module passes when it padded the heads)
        tgt16 = ops.attn_dist(p[:, :16], inp.sm_scale)
        ref16 = O.attn_dist(rp[:, :16], inp.sm_scale)
        assert (tgt16.cpu() - ref16).abs().max().item() < (1e-5 if dt == torch.float32 else 6e-3)
        assert triton_attn_dist(p, inp.sm_scale).dtype == dt
        # leaving out leading slots changes nothing but the width of p_out
        for skip in (32, 96):
            o_s, l_s, p_s = ops.sparse_mla_fwd(inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), 0, inp.sm_scale, 512, True, dt,
                                               p_out_skip=skip)
            assert p_s.shape == (200, 128, 128 - skip) and torch.equal(p_s, p[:, :, skip:])


def test_forward_invalid_ids_and_empty_rows(gpu):
    inp = O.make_mla_inputs(96, 128, 64, seed=5, skv=120, q_start=10)
    idx = inp.idx.clone()
    idx[5, 0] = -1
    idx[6, 1] = 120            # == s_kv
    idx[7, 2] = 119            # in range but in the future of query 7
    idx[8, :] = -1             # no valid slot at all
    idx[9] = idx[9][torch.randperm(64, generator=torch.Generator().manual_seed(1))]   # padding in the middle
    inp.idx = idx
    out, lse, p = _run_fwd(inp, gpu, 10, True, torch.float32)
    ro, rl, rp = O.sparse_mla_fwd(inp.q, inp.kv, idx, 10, inp.sm_scale, 512)
    assert_close(out, ro, "out")
    assert out[8].abs().max().item() == 0 and torch.isinf(lse[8]).all() and (lse[8] > 0).all()
    m = torch.isfinite(rl)
    assert (lse.cpu()[m] - rl[m]).abs().max().item() < 1e-4
    assert torch.equal(torch.isfinite(p.cpu()), torch.isfinite(rp))


@pytest.mark.parametrize("form,ranges,S,H,K", MLA_FORMS)
@pytest.mark.parametrize("end", ["before", "last"])
def test_forward_at_the_ends_of_the_query_positions(gpu, form, ranges, S, H, K, end):
    """Queries in front of the keys (a negative position: no valid slot, a zero row, lse = +inf), and positions up to the
    largest int, in every form; with ids at and beyond the number of keys, and negative ones other than -1."""
    from loongforge_amd import ops

    assert mla_form(S, H, K) == (form, ranges)
    skv, q_start = 90, -(S + 1) // 2 if end == "before" else 2 ** 31 - S
    inp = O.make_mla_inputs(S, H, 64, seed=S + H, skv=skv, q_start=skv)
    g = torch.Generator().manual_seed(K)
    idx = torch.randint(0, skv, (S, K), generator=g).int()
    for bad in (skv, skv + 1, 1 << 20, 2 ** 31 - 1, -1, -2, -77, -2 ** 31):
        idx[torch.rand(idx.shape, generator=g) < 0.05] = bad
    ro, rl, rp = O.sparse_mla_fwd(inp.q, inp.kv, idx, q_start, inp.sm_scale, 512)
    assert torch.isinf(rl[: -q_start if end == "before" else 0]).all()
    for dt in (None, torch.float32):
        out, lse, p = ops.sparse_mla_fwd(inp.q.to(gpu), inp.kv.to(gpu), idx.to(gpu), q_start, inp.sm_scale, 512, dt is not None,
                                         dt or torch.bfloat16)
        assert_close(out, ro, "out")
        fin = torch.isfinite(rl)
        assert torch.equal(torch.isposinf(lse.cpu()), ~fin) and (out.cpu()[~fin] == 0).all()
        assert not fin.any() or (lse.cpu() - rl)[fin].abs().max().item() < 1e-4
        if dt is not None:
            assert torch.equal(torch.isneginf(p.cpu()), torch.isneginf(rp))


@pytest.mark.parametrize("form,ranges,S,H,K", MLA_FORMS)
def test_forward_of_logits_that_are_minus_infinity(gpu, form, ranges, S, H, K):
    """Logits beyond the range of fp32 on the lower side count for nothing in every form: a row that has no others is like one
    without a valid slot, and where they come first the others decide, in the same tile or a later one."""
    from loongforge_amd import ops

    assert mla_form(S, H, K) == (form, ranges)
    skv = 2 * K
    inp = O.make_mla_inputs(S, H, 64, seed=S + H, skv=skv, q_start=skv)
    q, kv = inp.q.clone(), inp.kv.clone()
    q[:, :, 0], kv[:, 0] = 0, 0
    kv[:K, 0] = 8                                         # times -2^127: keys 0 .. K - 1 have a logit of -inf
    idx = torch.stack([torch.randperm(K)[:K] + K for _ in range(S)]).int()
    for i in range(S):                                    # none, all, those in front of a tile's middle, of all tiles but one, of half
        idx[i, :[0, K, 16, K - 32, K // 2][(i + 1) % 5]] -= K
        q[i, ::2 if i % 2 else 1, 0] = -2.0 ** 127        # odd rows: half of the heads
    sink = torch.linspace(-2, 2, H)
    for sk in (None, sink):
        ro, rl, rp = O.sparse_mla_fwd(q, kv, idx, skv, inp.sm_scale, 512, attn_sink=sk)
        assert torch.isneginf(rp).any() and not torch.isnan(ro).any()
        for dt in (None, torch.float32):
            out, lse, p = ops.sparse_mla_fwd(q.to(gpu), kv.to(gpu), idx.to(gpu), skv, inp.sm_scale, 512, dt is not None,
                                             dt or torch.bfloat16, attn_sink=None if sk is None else sk.to(gpu))
            assert_close(out, ro, "out")
            fin = torch.isfinite(rl)
            assert torch.equal(torch.isposinf(lse.cpu()), ~fin) and (out.cpu()[~fin] == 0).all()
            assert not fin.any() or (lse.cpu() - rl)[fin].abs().max().item() < 1e-4
            if dt is not None:
                assert torch.equal(torch.isneginf(p.cpu()), torch.isneginf(rp))


def test_backward_of_queries_in_front_of_the_keys(gpu):
    """The backward has the same rule: their dQ is zero and they add nothing to dKV."""
    from loongforge_amd import ops

    inp = O.make_mla_inputs(100, 64, 64, seed=3, skv=70, q_start=70)
    q_start = -41
    q, kv, idx, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, q_start, inp.sm_scale)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, q_start, inp.sm_scale)
    assert_mla_grads(dq, dkv, inp.q, inp.kv, inp.idx, inp.dout, q_start, inp.sm_scale, out=out, lse=lse)
    assert (dq[:41] == 0).all()


def test_forward_survives_a_late_dominant_key(gpu):
    """A key whose logit exceeds everything before it by far more than 2^64 forces the exact-max
    pass; the result must still match the oracle."""
    inp = O.make_mla_inputs(80, 128, 64, seed=6)
    kv = inp.kv.clone().float()
    kv[70] = inp.q[79, 0].float() * 40.0          # q.k ~ 40 * |q|^2 for query 79, head 0
    inp.kv = kv.to(torch.bfloat16)
    inp.idx[79, 63] = 70                            # visited in the last tile position
    out, lse, _ = _run_fwd(inp, gpu)
    ro, rl, _ = O.sparse_mla_fwd(inp.q, inp.kv, inp.idx, 0, inp.sm_scale, 512)
    assert_close(out, ro, "out", atol=4e-2)         # |kv[70]| is ~40x larger than the other rows
    assert (lse.cpu() - rl).abs().max().item() < 2e-2 * rl.abs().max().item() * 1e-2 + 1e-2


@pytest.mark.parametrize("S,H,K,q_start,skv", [
    (1, 128, 512, 900, None),         # one query: 32-head workgroups, a range per pair of tiles
    (3, 64, 320, 500, 700),           # five pairs of tiles per query
    (5, 96, 192, 300, None),          # the last 64-head workgroup holds 32 heads
    (2, 32, 128, 400, None),
    (300, 64, 192, 0, None),          # two workgroups on a unit, odd tile counts in the early rows
    (300, 32, 256, 0, None),
    (140, 64, 320, 0, None),          # two tiles at a time without ranges, odd tile counts in the early rows
    (140, 32, 256, 0, None),
    (2, 128, 4096, 5000, None),       # ranges that fit the two-tile ring though the whole list does not
])
def test_forward_shares_a_query_among_workgroups(gpu, S, H, K, q_start, skv):
    """Few queries or few heads: heads and slots of a query are spread over workgroups and streams.  Slot lists with
    holes, ranges without a valid slot, an empty row, sinks, logits, and a key that moves the softmax reference late."""
    from loongforge_amd import ops

    inp = O.make_mla_inputs(S, H, K, seed=S + H, skv=skv, q_start=q_start)
    g = torch.Generator().manual_seed(K)
    idx = inp.idx.clone()
    idx[torch.rand(idx.shape, generator=g) < 0.3] = -1
    idx[0, : K // 2] = -1
    if S > 2:
        idx[1] = -1
        idx[2, 33:] = -1
    sink = torch.linspace(-2, 2, H)
    for name, sk in (("plain", None), ("sink", sink)):
        if name == "sink" and (idx[0] >= 0).any():      # the last tile of a query beats those before it by far more than 2^64
            last = int((idx[0] >= 0).nonzero()[-1])
            kv = inp.kv.clone()
            kv[idx[0, last].long()] = (inp.q[0, H - 1].float() * 40.0).to(torch.bfloat16)
            inp.kv = kv
        ro, rl, rp = O.sparse_mla_fwd(inp.q, inp.kv, idx, q_start, inp.sm_scale, 512, attn_sink=sk)
        for dt in (None, torch.bfloat16, torch.float32):
            out, lse, p = ops.sparse_mla_fwd(inp.q.to(gpu), inp.kv.to(gpu), idx.to(gpu), q_start, inp.sm_scale, 512, dt is not None,
                                             dt or torch.bfloat16, attn_sink=None if sk is None else sk.to(gpu))
            assert_close(out, ro, name + " out", atol=4e-2 if sk is not None else 2e-2)
            fin = torch.isfinite(rl)
            assert torch.equal(torch.isfinite(lse.cpu()), fin)
            assert ((lse.cpu() - rl)[fin].abs() / rl[fin].abs().clamp_min(1)).max().item() < 1e-3
            if dt is not None:
                assert torch.equal(torch.isfinite(p.float().cpu()), torch.isfinite(rp))
            if dt == torch.float32:
                assert ((p.cpu() - rp)[torch.isfinite(rp)].abs() / rp[torch.isfinite(rp)].abs().clamp_min(1)).max().item() < 1e-3


@pytest.mark.parametrize("S,H,K,q_start,skv", [
    (3, 128, 64, 0, None),            # one pair of tiles, whatever the heads: one tile, then none
    (40, 96, 64, 30, None),           # one and two tiles, the fourth 32-head block is not there
    (5, 32, 64, 60, None),
    (260, 128, 192, 0, None),         # up to six tiles, fewer than the ring in the early rows; a second round of workgroups
    (170, 96, 320, 400, 500),         # the fourth 32-head block is not there
    (300, 128, 768, 0, None),         # from one tile in the early rows to 24
    (110, 128, 512, 900, None),       # two tiles at a time by 64 heads, without ranges: the blocks done again are the second group's
    (110, 96, 512, 900, None),
    (48, 96, 2048, 3000, None),       # in ranges of slots, by 64 heads
    (88, 96, 2048, 3000, None),       # in ranges, in two roles
    (70, 128, 2048, 0, 2100),         # the same; ranges without a tile in the early rows
])
def test_forward_of_many_heads(gpu, S, H, K, q_start, skv):
    """The two-role kernel, and the one for a pair of tiles, at the edges of their rings and heads; slot lists and bounds as above."""
    test_forward_shares_a_query_among_workgroups(gpu, S, H, K, q_start, skv)


@pytest.mark.parametrize("H", [64, 32])
@pytest.mark.parametrize("S,K,q_start,skv", [
    (300, 64 * 3, 0, None),           # one tile in the early rows: the other half of the ring stays empty
    (257, 128, 700, None),            # just more than there are compute units
    (530, 320, 900, None),
])
def test_forward_two_workgroups_to_a_unit(gpu, S, K, q_start, skv, H):
    """More queries than compute units: the forms and bounds of the tests above, and bf16 logits that are the fp32 ones rounded."""
    from loongforge_amd import ops

    test_forward_shares_a_query_among_workgroups(gpu, S, H, K, q_start, skv)
    inp = O.make_mla_inputs(S, H, K, seed=5, skv=skv, q_start=q_start)
    inp.idx[:, ::7] += S + q_start    # beyond the keys: no valid slots
    ro, rl, _ = O.sparse_mla_fwd(inp.q, inp.kv, inp.idx, q_start, inp.sm_scale, 512)
    out, lse, _ = _run_fwd(inp, gpu, q_start)
    assert_close(out, ro, "out")
    fin = torch.isfinite(rl)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and (lse.cpu() - rl)[fin].abs().max().item() < 1e-4
    for skip in (0, 64):
        p16, p32 = (ops.sparse_mla_fwd(inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), q_start, inp.sm_scale, 512, True, dt, p_out_skip=skip)[2]
                    for dt in (torch.bfloat16, torch.float32))
        assert p32.shape[2] == K - skip and torch.equal(p16, p32.to(torch.bfloat16))


@pytest.mark.parametrize("form,ranges,S,H,K", [
    (3, 1, 270, 64, 2112),            # more slots than one sweep of the masks takes, more tiles than a wave has lanes
    (4, 1, 258, 32, 2112),
    (3, 1, 350, 64, 8192),            # the longest list, which a block done again holds beside a tile
    (4, 1, 258, 32, 8192),
    (0, 1, 130, 128, 4096),
    (0, 5, 45, 128, 4096),
    (0, 2, 90, 96, 8192),
])
def test_forward_of_long_lists_in_every_form_for_many_queries(gpu, form, ranges, S, H, K):
    """The forms that own a query's slots with lists of more than 2048, in some of the rows: holes, tiles without a valid slot, an
    empty row, causal bounds, sinks, logits, and for one row a key in the last slot that beats all others by far more than 2^64."""
    from loongforge_amd import ops

    assert mla_form(S, H, K) == (form, ranges)
    skv = K + 900
    q_start = skv - S // 2                                # half of the queries have keys behind them
    g = torch.Generator().manual_seed(S + K)
    q = torch.randn(S, H, 576, generator=g).to(torch.bfloat16)
    kv = torch.randn(skv, 576, generator=g).to(torch.bfloat16)
    idx = torch.stack([torch.randperm(skv, generator=g)[:K] for _ in range(S)]).int()
    idx[torch.rand(idx.shape, generator=g) < 0.3] = -1
    idx[1, 32:K - 64] = -1                                # the first tile and the last two
    idx[2] = -1
    idx[S - 2, :2080] = -1
    idx[: S - 2][idx[: S - 2] == skv - 1] = -1
    idx[S - 3, K - 1] = skv - 1
    kv[skv - 1] = (q[S - 3, H - 1].float() * 40.0).to(torch.bfloat16)
    rows = [0, 1, 2, 3, S // 2, S - 3, S - 2, S - 1]
    sink = torch.linspace(-2, 2, H)
    for sk in (None, sink):
        ref = [O.sparse_mla_fwd(q[i:i + 1], kv, idx[i:i + 1], q_start + i, 192 ** -0.5, 512, attn_sink=sk) for i in rows]
        ro, rl, rp = (torch.cat(x) for x in zip(*ref))
        for dt in (None, torch.bfloat16, torch.float32):
            out, lse, p = ops.sparse_mla_fwd(q.to(gpu), kv.to(gpu), idx.to(gpu), q_start, 192 ** -0.5, 512, dt is not None,
                                             dt or torch.bfloat16, attn_sink=None if sk is None else sk.to(gpu))
            assert_close(out[rows], ro, "out", atol=4e-2)
            lse, fin = lse[rows].cpu(), torch.isfinite(rl)
            assert torch.equal(torch.isposinf(lse), ~fin)
            assert ((lse - rl)[fin].abs() / rl[fin].abs().clamp_min(1)).max().item() < 1e-3
            assert torch.isfinite(out.float()).all()
            if dt is not None:
                p = p[rows].cpu()
                assert torch.equal(torch.isfinite(p), torch.isfinite(rp))
            if dt == torch.bfloat16:
                p16 = p
            if dt == torch.float32:
                assert ((p - rp)[torch.isfinite(rp)].abs() / rp[torch.isfinite(rp)].abs().clamp_min(1)).max().item() < 1e-3
                assert torch.equal(p.to(torch.bfloat16), p16)


@pytest.mark.parametrize("form,S,H,K", [(2, 128, 32, 1024), (2, 61, 64, 1024), (2, 40, 96, 1024), (1, 115, 64, 2048), (1, 61, 96, 2048), (1, 55, 128, 2048)])
def test_two_ranges_of_slots_that_meet(gpu, form, S, H, K):
    """Two ranges whose second workgroup puts both together: keys that beat all before them by far more than 2^64 in the first range, in
    the second, in both; rows with nothing in one range or in either; sinks; whatever the workspace held; replays of a captured call."""
    from loongforge_amd import _lib, ops

    assert mla_form(S, H, K) == (form, 2)
    lib, skv, g = _lib.load(), K + 900, torch.Generator().manual_seed(S + H)
    q, kv = (torch.randn(*shape, generator=g).to(torch.bfloat16) for shape in ((S, H, 576), (skv, 576)))
    idx = torch.stack([torch.randperm(skv - 4, generator=g)[:K] for _ in range(S)]).int()
    idx[3] = -1
    idx[4, :K // 2] = -1
    idx[5, K // 2:] = -1
    for n, (row, slots) in enumerate([(6, [K // 2 - 1]), (7, [K - 1]), (8, [K // 2 - 1, K - 1])]):
        idx[row, slots[-1]] = skv - 1 - n
        idx[row, slots[0]] = skv - 1 - n if len(slots) == 1 else skv - 4
        kv[skv - 1 - n] = (q[row, H - 1].float() * 40.0).to(torch.bfloat16)
    kv[skv - 4] = kv[skv - 3] * 1.5
    rows, sm = list(range(12)) + [S - 1], 192 ** -0.5
    qg, kvg, ig = q.to(gpu), kv.to(gpu), idx.to(gpu)
    for sk in (None, torch.linspace(-2, 2, H)):
        sg = None if sk is None else sk.to(gpu)
        out, lse, _ = ops.sparse_mla_fwd(qg, kvg, ig, skv, sm, attn_sink=sg)
        ref = [O.sparse_mla_fwd(q[i:i + 1], kv, idx[i:i + 1], skv, sm, 512, attn_sink=sk) for i in rows]
        ro, rl = (torch.cat(x) for x in list(zip(*ref))[:2])
        assert_close(out[rows], ro, "out", atol=4e-2)
        got, fin = lse[rows].cpu(), torch.isfinite(rl)
        assert torch.equal(torch.isposinf(got), ~fin) and ((got - rl)[fin].abs() / rl[fin].abs().clamp_min(1)).max().item() < 1e-3
        nbytes = lib.dsa_sparse_mla_fwd_workspace_bytes(S, H, skv, K)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
        for fill in (0, 255, 85, None, None):
            if fill is not None:
                ws.fill_(fill)
            o2, l2 = torch.full_like(out, 7.0), torch.full_like(lse, 7.0)
            rc = lib.dsa_sparse_mla_fwd_ws(qg.data_ptr(), kvg.data_ptr(), ig.data_ptr(), S, H, skv, K, skv, sm, 512, o2.data_ptr(), l2.data_ptr(),
                                           None, 0, None if sg is None else sg.data_ptr(), 0, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
            assert rc == 0, lib.dsa_last_error()
            assert torch.equal(o2, out) and torch.equal(l2, lse)
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    plain = ops.sparse_mla_fwd(qg, kvg, ig, skv, sm)[0]
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        ops.sparse_mla_fwd(qg, kvg, ig, skv, sm)
    torch.cuda.current_stream().wait_stream(stream)
    with torch.cuda.graph(graph):
        captured = ops.sparse_mla_fwd(qg, kvg, ig, skv, sm)[0]
    for _ in range(4):
        captured.zero_()
        graph.replay()
        assert torch.equal(captured, plain)
        assert torch.equal(ops.sparse_mla_fwd(qg, kvg, ig, skv, sm)[0], plain)


def test_forward_slot_permutation_invariance(gpu):
    inp = O.make_mla_inputs(100, 128, 128, seed=7)
    out1, lse1, _ = _run_fwd(inp, gpu)
    perm = torch.randperm(128, generator=torch.Generator().manual_seed(2))
    inp.idx = inp.idx[:, perm].contiguous()
    out2, lse2, _ = _run_fwd(inp, gpu)
    assert (out1.float() - out2.float()).abs().max().item() < 2e-2
    assert (lse1 - lse2).abs().max().item() < 1e-4


@pytest.mark.parametrize("S,H,K,q_start,skv,seed", [
    (64, 128, 64, 0, None, 0),
    (200, 128, 128, 40, 300, 3),
    (160, 64, 64, 0, None, 5),
    (130, 32, 192, 5, 400, 7),           # 16 heads and half a tile's keys for each of four waves
    (90, 96, 320, 0, None, 9),           # six of eight 16-head waves hold real heads; ten tiles per query
])
def test_backward_against_oracle_and_deterministic(gpu, S, H, K, q_start, skv, seed):
    from loongforge_amd import ops

    inp = O.make_mla_inputs(S, H, K, seed=seed, skv=skv, q_start=q_start)
    q, kv, idx, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, q_start, inp.sm_scale)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, q_start, inp.sm_scale)
    assert_mla_grads(dq, dkv, inp.q, inp.kv, inp.idx, inp.dout, q_start, inp.sm_scale, out=out, lse=lse)
    dq2, dkv2 = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, q_start, inp.sm_scale)
    assert torch.equal(dq, dq2) and torch.equal(dkv, dkv2)          # bit-identical


@pytest.mark.parametrize("H", [32, 64])
@pytest.mark.parametrize("S,K,q_start,skv", [
    (1, 64, 0, None),                 # one valid slot
    (67, 64, 0, None),                # one and two tiles per query
    (70, 320, 0, None),               # up to ten tiles: odd and even counts, more than the rings hold
    (9, 2048, 3000, None),            # the longest lists
])
def test_backward_of_few_heads(gpu, H, S, K, q_start, skv):
    """Up to 64 heads the passes share tiles, k-steps and compute units differently; one workspace sweep and several give the
    sums of the oracle, and an empty row or a tile without valid slots adds nothing."""
    from loongforge_amd import ops

    inp = O.make_mla_inputs(S, H, K, seed=S + H, skv=skv, q_start=q_start)
    inp.idx = inp.idx.clone()
    inp.idx[:, 40:50] = -1
    if S > 2:
        inp.idx[2] = -1
    q, kv, idx, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, q_start, inp.sm_scale)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, q_start, inp.sm_scale)
    assert_mla_grads(dq, dkv, inp.q, inp.kv, inp.idx, inp.dout, q_start, inp.sm_scale, out=out, lse=lse)
    dq2, dkv2 = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, q_start, inp.sm_scale)
    assert torch.equal(dq, dq2) and torch.equal(dkv, dkv2)
    if S > 2:
        assert (dq[2] == 0).all()


@pytest.mark.parametrize("S,H,K,q_start", [
    (1, 128, 64, 0),                  # one valid slot
    (68, 96, 64, 0),                  # heads that repeat the last one; one and two tiles per query
    (70, 128, 320, 0),                # up to ten tiles
    (5, 128, 2048, 3000),             # the longest lists
])
def test_backward_of_many_heads_in_one_pass(gpu, S, H, K, q_start):
    """P, dS and the rows of the pairs in one kernel: the first and the last tiles of a query, empty rows, the end of the order's
    list, against the oracle, with the bounds of the other backward tests."""
    test_backward_of_few_heads(gpu, H, S, K, q_start, None)


@pytest.mark.parametrize("S,H,K", [(511, 128, 64), (512, 96, 64), (770, 128, 64), (1301, 128, 192)])
def test_every_query_of_several_rounds_is_worked_on(gpu, S, H, K):
    """The first 256 workgroups take queries from the whole range, the others what is left: each query once, whatever the sizes."""
    from loongforge_amd import ops

    inp = O.make_mla_inputs(S, H, K, seed=S)
    q, kv, ids, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
    torch.full((3 * S, H, 576), float("nan"), dtype=torch.bfloat16, device=gpu)        # (what is left unwritten is likely to show)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, ids, 0, inp.sm_scale)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, ids, lse, 0, inp.sm_scale)
    ro, rl, _ = O.sparse_mla_fwd(inp.q, inp.kv, inp.idx, 0, inp.sm_scale, 512)
    assert_close(out, ro, "out")
    assert (lse.cpu() - rl).abs().max().item() < 1e-4
    assert_mla_grads(dq, dkv, inp.q, inp.kv, inp.idx, inp.dout, 0, inp.sm_scale, name="rounds", out=out, lse=lse)


def _overlapping_ids(S, K, skv, turn, far, seed):
    """Causal ids of queries at positions skv - S + i: K of the K + K / 8 keys behind a place that moves by a key every ``turn``
    queries (0: never), and for every ``far``-th run of 16 queries ids at random, which neighbours hardly share."""
    g = torch.Generator().manual_seed(seed)
    ids = torch.full((S, K), -1, dtype=torch.int32)
    for i in range(S):
        last = skv - S + i
        if far and i // 16 % far == far - 1:
            pool = torch.arange(last + 1)
        else:
            pool = torch.arange(max(0, i // turn - 8) if turn else 0, last + 1)[:K + K // 8]
        pick = pool[torch.randperm(len(pool), generator=g)[:K]]
        ids[i, :len(pick)] = pick.int()
    return ids


def _assert_rounded_rows(dkv, inp, units, q_start, sm, out, lse):
    """dKV against the oracle with the same rounding points - bf16 P and dS, a row per query in bf16 or per group of queries worked as one
    in its 11 bits - within the bound of assert_mla_grads: a step of the grid of the largest row on top of 2e-2 + 1e-2 |ref|.
    Returns dQ and dKV of the oracle without rounded rows."""
    kw = dict(out=out.cpu(), lse=lse.cpu(), dtype=torch.float64)
    dq_b, dkv_b = O.sparse_mla_bwd_kernel_rounding(inp.q, inp.kv, inp.idx, inp.dout, q_start, sm, 512, **kw)
    _, ref, _, largest = O.sparse_mla_bwd_kernel_rounding(inp.q, inp.kv, inp.idx, inp.dout, q_start, sm, 512, round_rows_bf16=True,
                                                          return_abs_sum=True, units=units, **kw)
    over = ((dkv.cpu().double() - ref).abs() - (2e-2 + 1e-2 * ref.abs() + 2.0 ** -7 * largest)).max().item()
    assert over <= 0, "dKV exceeds the bound by %.3e" % over
    return dq_b, dkv_b


@pytest.mark.parametrize("H,S,K,skv,turn,far", [
    (64, 515, 128, 900, 1, 0),        # pairs of queries as one, one query left over
    (64, 520, 192, 1400, 1, 3),       # both kinds of groups
    (64, 513, 128, 520, 2, 0),        # lists that begin short
    (64, 520, 192, 40_000, 1, 3),     # long key arrays
    (32, 1030, 64, 33_000, 2, 2),
    (32, 768, 64, 1100, 1, 0),        # four queries as one
    (32, 771, 64, 1500, 1, 2),        # three queries left over, both kinds
])
def test_backward_of_joint_queries(gpu, H, S, K, skv, turn, far):
    """Consecutive queries of 64 or 32 heads that share most of their keys are worked as one query of 128 heads: holes, empty
    rows and groups of either kind against the oracle with the same rounding points."""
    from loongforge_amd import ops

    q_start = skv - S
    inp = O.make_mla_inputs(S, H, K, seed=S + H, skv=skv, q_start=q_start)
    inp.idx = _overlapping_ids(S, K, skv, turn, far, S)
    inp.idx[2] = -1
    inp.idx[8:12] = -1
    inp.idx[20:40, 10:13] = -1
    q, kv, idx, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, q_start, inp.sm_scale)
    dq, dkv, G, joint = mla_bwd_with_groups(q, kv, out, do, idx, lse, q_start, inp.sm_scale)
    assert G == 128 // H and len(joint) // 4 < sum(joint) < len(joint) - len(joint) // 8 * (far > 0)
    dq_b, dkv_b = _assert_rounded_rows(dkv, inp, (G, joint), q_start, inp.sm_scale, out, lse)
    assert_close(dq, dq_b, "dQ")
    assert ((dkv.double().cpu() - dkv_b).abs() - 2e-2 - 1e-2 * dkv_b.abs()).max().item() <= REF_DKV_EXCESS_LIMIT
    dq2, dkv2 = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, q_start, inp.sm_scale)
    assert torch.equal(dq, dq2) and torch.equal(dkv, dkv2)
    assert (dq[2] == 0).all() and (dq[8:12] == 0).all()
    # a repeated id in one query of a group: NaN everywhere, as ever
    dup = idx.clone()
    dup[S // 2, 5] = dup[S // 2, 9]
    dq3, dkv3 = ops.sparse_mla_bwd(q, kv, out, do, dup, lse, q_start, inp.sm_scale)
    assert torch.isnan(dq3.float()).all() and torch.isnan(dkv3.float()).all()


@pytest.mark.parametrize("H,S,K,skv", [(64, 512, 128, 300), (64, 1024, 64, 72), (64, 520, 64, 64), (32, 800, 128, 300), (32, 768, 64, 200),
                                       (32, 800, 64, 64)])
@pytest.mark.parametrize("alike,steep", [(0.0, 1.0), (0.9, 1.0), (0.99, 1.0), (0.9, 2.0)])
def test_backward_of_joint_queries_is_no_less_accurate_than_one_by_one(gpu, H, S, K, skv, alike, steep):
    """Neighbouring queries with most of their keys, and of their values (``alike``: correlation of Q and dO), in common: dKV is no
    further from bf16 P and dS with unrounded rows than the sums of one bf16 row per query are, the result's own rounding on
    both sides."""
    from loongforge_amd import ops

    inp = O.make_mla_inputs(S, H, K, seed=S + H, skv=skv, q_start=skv)
    g = torch.Generator().manual_seed(S)
    mix = lambda t: (alike ** 0.5 * torch.randn((S + 7) // 8, 1, *t.shape[1:], generator=g).expand(-1, 8, -1, -1).flatten(0, 1)[:S]    # noqa: E731
                     + (1 - alike) ** 0.5 * torch.randn(t.shape, generator=g)).to(torch.bfloat16)
    inp.q, inp.dout = mix(inp.q), mix(inp.dout)
    some = min(K + K // 8, skv)
    pool = torch.stack([torch.randperm(skv, generator=g)[:some] for _ in range((S + 7) // 8)])
    inp.idx = torch.stack([pool[i // 8][torch.randperm(some, generator=g)[:K]] for i in range(S)]).int()
    q, kv, idx, do, sm = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu), steep * inp.sm_scale
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, skv, sm)
    dq, dkv, G, joint = mla_bwd_with_groups(q, kv, out, do, idx, lse, skv, sm)
    assert sum(joint) > len(joint) // 2
    dq_b, ref = _assert_rounded_rows(dkv, inp, (G, joint), skv, sm, out, lse)
    _, rows = O.sparse_mla_bwd_kernel_rounding(inp.q, inp.kv, inp.idx, inp.dout, skv, sm, 512, round_rows_bf16=True, out=out.cpu(),
                                               lse=lse.cpu(), dtype=torch.float64)
    assert_close(dq, dq_b, "dQ")
    off, one_by_one = dkv.cpu().double() - ref, rows.to(torch.bfloat16).double() - ref
    assert off.norm() <= one_by_one.norm()
    assert off.abs().max() <= 1.1 * one_by_one.abs().max()                 # (the largest of many roundings, of other values)


@pytest.mark.parametrize("H,S,K,skv,causal", [
    (64, 700, 2048, 2300, False),
    (32, 1100, 2048, 3110, False),    # unions beyond the longest list of a unit, and within it
    (64, 1030, 512, 1200, True),
    (32, 1537, 192, 1537, True),      # from one key on
    (32, 1540, 256, 6000, False),     # little in common: no units
    (32, 2103, 128, 400, False),      # more than two rounds of groups
])
def test_backward_of_joint_queries_is_that_of_wider_queries(gpu, H, S, K, skv, causal):
    """The same gradients as through the kernels for 128 heads with heads of zeros beside the queries' own, in one sweep and in
    several.  dQ: the order of its fp32 sums, rounded to bf16 - 2**-8 of an element, or an fp32 step of the largest ones where terms
    cancel.  dKV: rows rounded to bf16 per query on one side and to 11 bits per unit on the other, and either result to bf16: a
    rounding to bf16 is 1.66e-3 of the norm (2**-7 / sqrt(12) over the root mean square of a significand), 3 of them 2.9e-3."""
    from loongforge_amd import _lib, ops

    g = torch.Generator(device=gpu).manual_seed(S + H)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu).to(torch.bfloat16)                     # noqa: E731
    q, kv, do = rnd(S, H, 576), rnd(skv, 576), rnd(S, H, 512)
    score = torch.rand(S, skv, generator=g, device=gpu)
    q_start = skv - S if causal else skv
    if causal:
        score.masked_fill_(torch.arange(skv, device=gpu)[None] > (q_start + torch.arange(S, device=gpu))[:, None], -1.0)
    val, idx = score.topk(K, -1)
    idx = torch.where(val >= 0, idx, -1).int()
    sm = 192 ** -0.5
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, q_start, sm)
    dq, dkv, G, joint = mla_bwd_with_groups(q, kv, out, do, idx, lse, q_start, sm)
    assert G == 128 // H and (sum(joint) == 0 if skv == 6000 else sum(joint) > len(joint) // 4)
    wide = lambda t: torch.cat([t, torch.zeros(S, 128 - H, *t.shape[2:], dtype=t.dtype, device=gpu)], 1).contiguous()      # noqa: E731
    dq_w, dkv_w = ops.sparse_mla_bwd(wide(q), kv, wide(out), wide(do), idx, wide(lse), q_start, sm)
    a, b = dq.float(), dq_w[:, :H].float()
    assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 2.0 ** -14 * b.abs().max()).all()
    a, b = dkv.float(), dkv_w.float()
    assert (a - b).norm() <= 3.3e-3 * b.norm()
    part = _lib.load().dsa_sparse_mla_bwd_workspace_bytes((S + 1) // 2, H, skv, K)
    dq2, dkv2, G2, joint2 = mla_bwd_with_groups(q, kv, out, do, idx, lse, q_start, sm, part)
    assert torch.equal(dq2, dq) and G2 == G and joint2 == joint
    a, b = dkv2.float(), dkv_w.float()
    assert (a - b).norm() <= 3.3e-3 * b.norm()


@pytest.mark.parametrize("H,S", [(64, 700), (32, 1103)])
def test_dq_of_joint_queries_does_not_depend_on_the_workspace(gpu, H, S):
    """Which queries are worked as one follows from the whole call and not from the chunks that a smaller workspace allows: the same
    bits of dQ in one sweep, in two, in chunks of 64 or less, and dKV to the order of its sums.  Less than the smallest documented
    workspace is still taken if it holds 64 queries one by one."""
    from loongforge_amd import _lib, ops

    K, skv = 192, 1200
    inp = O.make_mla_inputs(S, H, K, seed=S, skv=skv, q_start=skv)
    inp.idx = _overlapping_ids(S, K, skv + S, 0, 3, S)
    q, kv, idx, do, sm = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu), inp.sm_scale
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, skv, sm)
    dq, dkv, G, joint = mla_bwd_with_groups(q, kv, out, do, idx, lse, skv, sm)
    assert len(joint) // 4 < sum(joint) < len(joint)
    lib = _lib.load()
    least, one_by_one = lib.dsa_sparse_mla_bwd_workspace_bytes_min(S, H, skv, K), lib.dsa_sparse_mla_bwd_workspace_bytes(64, H, skv, K)
    assert one_by_one <= least
    for nbytes in (lib.dsa_sparse_mla_bwd_workspace_bytes((S + 3) // 2, H, skv, K) + 2 ** 20, least, one_by_one):
        dq2, dkv2, G2, joint2 = mla_bwd_with_groups(q, kv, out, do, idx, lse, skv, sm, nbytes)
        assert G2 == G and joint2 == joint and torch.equal(dq, dq2) or nbytes < least and G2 == 1
        a, b = dkv2.float(), dkv.float()
        assert (a - b).norm() <= 3e-3 * b.norm()
        assert_close(dq2, dq, "dQ")


@pytest.mark.parametrize("H,S", [(64, 520), (32, 800)])
@pytest.mark.parametrize("where,value", [("dout", float("nan")), ("dout", float("inf")), ("q", float("nan")), ("q_rope", float("inf")),
                                         ("kv", float("nan"))])
def test_backward_of_joint_queries_keeps_nonfinite_values_apart(gpu, H, S, where, value):
    """A value that is not finite in one query's row reaches that query's dQ and the keys it selected and nothing else, as if
    the queries it is worked with were not there; in a key row, the queries that selected the key."""
    from loongforge_amd import ops

    K, skv = 128, 700
    inp = O.make_mla_inputs(S, H, K, seed=S, skv=skv, q_start=skv)
    idx = _overlapping_ids(S, K, skv + S, 0, 0, 5)        # K of 144 keys
    q, kv, do = inp.q.to(gpu), inp.kv.to(gpu), inp.dout.to(gpu)
    ids, sm = idx.to(gpu), inp.sm_scale
    out, lse, _ = ops.sparse_mla_fwd(q, kv, ids, skv, sm)
    dq0, dkv0, G, joint = mla_bwd_with_groups(q, kv, out, do, ids, lse, skv, sm)
    assert torch.isfinite(dq0.float()).all() and torch.isfinite(dkv0.float()).all()
    bad = 101
    assert joint[bad // G]
    if where == "dout":
        do[bad, H // 2, 77] = value
    elif where == "kv":
        kv[int(idx[bad, 3]), 5] = value
    else:
        q[bad, 3, 40 if where == "q" else 570] = value
    out, lse, _ = ops.sparse_mla_fwd(q, kv, ids, skv, sm)
    dq, dkv, _, joint = mla_bwd_with_groups(q, kv, out, do, ids, lse, skv, sm)
    assert joint[bad // G] == (where != "kv")
    hit = torch.zeros(S, dtype=torch.bool)
    if where == "kv":
        hit = (idx == int(idx[bad, 3])).any(1)
        keys = torch.unique(idx[hit]).long()
    else:
        hit[bad] = True
        keys = idx[bad].long()
    assert 0 < hit.sum() < S
    touched = torch.zeros(skv, dtype=torch.bool)
    touched[keys] = True
    dq, dkv = dq.float().cpu(), dkv.float().cpu()
    assert torch.isfinite(dq[~hit]).all()
    assert (~torch.isfinite(dq[hit])).flatten(1).any(1).all()
    assert torch.isfinite(dkv[~touched]).all()
    if where != "kv":                          # (every pair of the query has a non-finite row)
        assert (~torch.isfinite(dkv[touched])).any(1).all() and torch.equal(dkv[~touched], dkv0.float().cpu()[~touched])


@pytest.mark.parametrize("H,S", [(64, 520), (32, 800)])
@pytest.mark.parametrize("factor", [2.0 ** -12, 2.0 ** -20])
def test_backward_of_joint_queries_with_columns_of_unlike_size(gpu, H, S, factor):
    """Every other column of Q, dO and the keys smaller: those columns of dKV share their power of two with the large ones and are no
    less accurate for it than one bf16 row per query makes them."""
    from loongforge_amd import ops

    K, skv = 128, 700
    inp = O.make_mla_inputs(S, H, K, seed=S, skv=skv, q_start=skv)
    inp.idx = _overlapping_ids(S, K, skv + S, 0, 0, 5)
    for t in (inp.q, inp.kv, inp.dout):
        t[..., 1::2] *= factor
    q, kv, do, ids, sm = inp.q.to(gpu), inp.kv.to(gpu), inp.dout.to(gpu), inp.idx.to(gpu), inp.sm_scale
    out, lse, _ = ops.sparse_mla_fwd(q, kv, ids, skv, sm)
    _, dkv, G, joint = mla_bwd_with_groups(q, kv, out, do, ids, lse, skv, sm)
    assert sum(joint) > len(joint) // 2
    kw = dict(out=out.cpu(), lse=lse.cpu(), dtype=torch.float64)
    _, ref = O.sparse_mla_bwd_kernel_rounding(inp.q, inp.kv, inp.idx, inp.dout, skv, sm, 512, **kw)
    _, rows = O.sparse_mla_bwd_kernel_rounding(inp.q, inp.kv, inp.idx, inp.dout, skv, sm, 512, round_rows_bf16=True, **kw)
    off, one_by_one = dkv.cpu().double() - ref, rows.to(torch.bfloat16).double() - ref
    for c in (slice(0, None, 2), slice(1, None, 2)):
        assert off[:, c].norm() <= one_by_one[:, c].norm()


@pytest.mark.parametrize("H,S", [(64, 520), (32, 800)])
def test_backward_of_joint_queries_with_a_column_that_overflows(gpu, H, S):
    """A sum over the heads beyond the range of fp32 in one column of a pair row leaves the row's other columns as they are."""
    from loongforge_amd import ops

    K, skv, bad, col = 128, 700, 101, 77
    inp = O.make_mla_inputs(S, H, K, seed=S, skv=skv, q_start=skv)
    idx = _overlapping_ids(S, K, skv + S, 0, 0, 5)
    key = int(idx[bad, 3])
    q, kv, do, ids, sm = inp.q.to(gpu), inp.kv.to(gpu), inp.dout.to(gpu), idx.to(gpu), inp.sm_scale
    kv[:, col] = 0                             # (else dP and delta overflow as well)
    kv[key] *= 4
    q[bad] = kv[key]                           # every head's probability is on this key
    do[bad, :, col] = 0
    out, lse, _ = ops.sparse_mla_fwd(q, kv, ids, skv, sm)
    dq0, dkv0 = ops.sparse_mla_bwd(q, kv, out, do, ids, lse, skv, sm)
    do[bad, :, col] = 3e38
    dq, dkv, G, joint = mla_bwd_with_groups(q, kv, out, do, ids, lse, skv, sm)
    assert joint[bad // G]
    assert torch.isposinf(dkv[key, col])
    rest = torch.arange(576, device=gpu) != col
    assert torch.isfinite(dkv0.float()).all() and torch.equal(dq, dq0) and torch.equal(dkv[:, rest], dkv0[:, rest])


@pytest.mark.parametrize("H", [32, 128])
def test_backward_of_keys_with_few_and_many_rows(gpu, H):
    """Keys with numbers of rows around one row per thread group (7) and one batch of loads (56), and with none, in any
    neighbourhood."""
    from loongforge_amd import ops

    counts = [0, 1, 6, 7, 0, 0, 0, 0, 8, 55, 56, 57, 111, 112, 113, 180, 168, 0, 63, 5, 0]
    S, K, skv = 180, 64, len(counts)
    inp = O.make_mla_inputs(S, H, K, seed=H, skv=skv, q_start=skv)
    idx = torch.full((S, K), -1, dtype=torch.int32)
    for i in range(S):
        mine = [j for j, c in enumerate(counts) if i < c]
        idx[i, :len(mine)] = torch.tensor(mine, dtype=torch.int32)
    q, kv, do, ids = inp.q.to(gpu), inp.kv.to(gpu), inp.dout.to(gpu), idx.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, ids, skv, inp.sm_scale)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, ids, lse, skv, inp.sm_scale)
    # Against the same rounding points (bf16 P, dS and rows), within the bound that assert_mla_grads derives for them: one step of the
    # bf16 grid at the largest row that enters.  (Its further limits against plain fp32 are for selections of many keys; with a
    # dozen P is of order 0.1 and so are the errors that its rounding to bf16 puts into sums of 180 rows.)
    _, ref, _, largest = O.sparse_mla_bwd_kernel_rounding(inp.q, inp.kv, idx, inp.dout, skv, inp.sm_scale, 512, out=out.cpu(), lse=lse.cpu(),
                                                          dtype=torch.float64, round_rows_bf16=True, return_abs_sum=True)
    dkv = dkv.float().cpu()
    assert ((dkv - ref).abs() <= 2e-2 + 1e-2 * ref.abs() + 2.0 ** -7 * largest).all()
    assert (dkv[torch.tensor(counts) == 0] == 0).all()


def test_backward_does_not_depend_on_the_slot_order(gpu):
    """The backward walks each query's ids in ascending key order whatever order they arrive in, so
    permuting the slots (independently per query) and scattering unused slots between the used ones
    gives bit-identical gradients."""
    from loongforge_amd import ops

    S, K = 150, 128
    inp = O.make_mla_inputs(S, 128, 96, seed=9)                       # 96 used slots ...
    idx = torch.cat([inp.idx, torch.full((S, K - 96), -1, dtype=torch.int32)], dim=1)
    g = torch.Generator().manual_seed(3)
    shuffled = torch.stack([idx[i][torch.randperm(K, generator=g)] for i in range(S)])      # ... anywhere among 128
    q, kv, do = inp.q.to(gpu), inp.kv.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx.to(gpu), 0, inp.sm_scale)
    dq1, dkv1 = ops.sparse_mla_bwd(q, kv, out, do, idx.to(gpu), lse, 0, inp.sm_scale)
    dq2, dkv2 = ops.sparse_mla_bwd(q, kv, out, do, shuffled.to(gpu), lse, 0, inp.sm_scale)
    assert torch.equal(dq1, dq2) and torch.equal(dkv1, dkv2)
    assert_mla_grads(dq2, dkv2, inp.q, inp.kv, inp.idx, inp.dout, 0, inp.sm_scale, out=out, lse=lse)


def test_backward_with_more_keys_than_the_key_bitmap_in_lds_holds(gpu):
    """Beyond about 600 000 keys the per-query key bitmap (and with it the key-sorted id list) no longer
    fits LDS and the passes walk the caller's slot order; results must not care.  The oracle runs on the
    selected keys only (compacted), everything else must get a zero gradient."""
    from loongforge_amd import ops

    S, H, K, skv = 64, 128, 64, 620_000
    g = torch.Generator().manual_seed(17)
    q = torch.randn(S, H, 576, generator=g).to(torch.bfloat16)
    dout = torch.randn(S, H, 512, generator=g).to(torch.bfloat16)
    picked = torch.randperm(skv, generator=g)[:1500]                       # the keys any query may select
    kv_small = torch.randn(1500, 576, generator=g).to(torch.bfloat16)
    idx_small = torch.stack([torch.randperm(1500, generator=g)[:K] for _ in range(S)]).to(torch.int32)
    idx_small[3, 10:] = -1
    idx = torch.where(idx_small >= 0, picked[idx_small.clamp(min=0).long()].to(torch.int32), idx_small)
    kv = torch.zeros(skv, 576, dtype=torch.bfloat16)
    kv[picked] = kv_small
    sm = 192 ** -0.5
    qd, kd, dd, ids = q.to(gpu), kv.to(gpu), dout.to(gpu), idx.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(qd, kd, ids, skv, sm)                 # q_start = skv: no causal test
    dq, dkv = ops.sparse_mla_bwd(qd, kd, out, dd, ids, lse, skv, sm)
    ro, _, _ = O.sparse_mla_fwd(q, kv_small, idx_small, 1500, sm, 512)
    assert_close(out, ro, "out")
    assert_mla_grads(dq, dkv, q, kv_small, idx_small, dout, 1500, sm, out=out, lse=lse, dkv_rows=picked)
    rest = torch.ones(skv, dtype=torch.bool)
    rest[picked] = False
    assert (dkv.cpu()[rest] == 0).all()


def test_backward_with_a_repeated_id_returns_nan_not_a_wrong_sum(gpu):
    """The backward keeps one bit and one row per (query, key): a row of ids that names a key twice
    cannot be summed correctly, and the call says so by returning NaN everywhere."""
    from loongforge_amd import ops

    inp = O.make_mla_inputs(96, 128, 64, seed=4)
    idx = inp.idx.clone()
    idx[70, 5] = idx[70, 9]
    q, kv, do = inp.q.to(gpu), inp.kv.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx.to(gpu), 0, inp.sm_scale)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, idx.to(gpu), lse, 0, inp.sm_scale)
    assert torch.isnan(dq.float()).all() and torch.isnan(dkv.float()).all()
    # the same workspace-free call with distinct ids is clean again (the flag is cleared per call)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, inp.idx.to(gpu), 0, inp.sm_scale)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, inp.idx.to(gpu), lse, 0, inp.sm_scale)
    assert torch.isfinite(dq.float()).all() and torch.isfinite(dkv.float()).all()
    # a repeated id that is not valid (in the future of the query) does not count
    idx = inp.idx.clone()
    idx[3, 5] = idx[3, 9] = 50
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx.to(gpu), 0, inp.sm_scale)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, idx.to(gpu), lse, 0, inp.sm_scale)
    assert torch.isfinite(dq.float()).all() and torch.isfinite(dkv.float()).all()


def test_forward_and_backward_with_attention_sink(gpu):
    from loongforge_amd import ops

    S, H, K, q_start = 200, 128, 128, 40
    inp = O.make_mla_inputs(S, H, K, seed=7, skv=300, q_start=q_start)
    idx = inp.idx.clone()
    idx[9, :] = -1                                                  # a row with only the sink
    g = torch.Generator().manual_seed(3)
    sink = torch.randn(H, generator=g) * 3.0
    sink[0], sink[1], sink[2] = 60.0, -60.0, 0.0                    # dominant, negligible, neutral
    q, kv, ids, do = inp.q.to(gpu), inp.kv.to(gpu), idx.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, ids, q_start, inp.sm_scale, attn_sink=sink.to(gpu))
    ro, rl, _ = O.sparse_mla_fwd(inp.q, inp.kv, idx, q_start, inp.sm_scale, 512, attn_sink=sink)
    assert_close(out, ro, "out")
    assert torch.isfinite(lse).all()
    assert (lse.cpu() - rl).abs().max().item() < 1e-4
    assert (lse[9].cpu() - sink).abs().max().item() < 1e-5 and out[9].abs().max().item() == 0
    # without a sink the same call is unchanged by the extra argument
    o0, l0, _ = ops.sparse_mla_fwd(q, kv, ids, q_start, inp.sm_scale)
    o1, l1, _ = ops.sparse_mla_fwd(q, kv, ids, q_start, inp.sm_scale, attn_sink=None)
    assert torch.equal(o0, o1) and torch.equal(l0, l1)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, ids, lse, q_start, inp.sm_scale)
    assert_mla_grads(dq, dkv, inp.q, inp.kv, idx, inp.dout, q_start, inp.sm_scale, attn_sink=sink, out=out, lse=lse)


def test_sink_survives_the_exact_pass(gpu):
    # a late dominant key sends the query through the second (exact-maximum) pass; the sink term
    # must be applied there as well
    from loongforge_amd import ops

    inp = O.make_mla_inputs(80, 128, 64, seed=6)
    kv = inp.kv.clone().float()
    kv[70] = inp.q[79, 0].float() * 40.0
    kv = kv.to(torch.bfloat16)
    idx = inp.idx.clone()
    idx[79, 63] = 70
    sink = torch.linspace(-4, 4, 128)
    sink[0] = 1567.0                                 # comparable with the dominant logit of head 0 (about 1568)
    out, lse, _ = ops.sparse_mla_fwd(inp.q.to(gpu), kv.to(gpu), idx.to(gpu), 0, inp.sm_scale, attn_sink=sink.to(gpu))
    ro, rl, _ = O.sparse_mla_fwd(inp.q, kv, idx, 0, inp.sm_scale, 512, attn_sink=sink)
    assert_close(out, ro, "out", atol=4e-2)
    assert ((lse.cpu() - rl).abs() / rl.abs().clamp_min(1)).max().item() < 1e-3


@pytest.mark.parametrize("S,H,K", [(3073, 32, 2048), (1537, 64, 2048)])          # dS of the sweep 384 MiB and 128 or 256 KiB more
def test_backward_on_both_sides_of_the_way_that_ds_is_read(gpu, monkeypatch, S, H, K):
    """One sweep whose dS is just above the size from which it is read through the caches, against sweeps of less: the same dQ."""
    from loongforge_amd import _lib, ops

    g = torch.Generator(device=gpu).manual_seed(S)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=gpu, dtype=torch.bfloat16)      # noqa: E731
    q, kv, do = rnd(S, H, 576), rnd(S + 500, 576), rnd(S, H, 512)
    ids = ops.topk(torch.randn(S, S + 500, generator=g, device=gpu), K)[1]
    out, lse, _ = ops.sparse_mla_fwd(q, kv, ids, S + 500)
    dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, ids, lse, S + 500)
    half = _lib.load().dsa_sparse_mla_bwd_workspace_bytes((S + 1) // 2 + 4, H, S + 500, K)
    monkeypatch.setenv("DSA_BWD_WORKSPACE_GIB", repr(half / 2 ** 30))
    dq2, dkv2 = ops.sparse_mla_bwd(q, kv, out, do, ids, lse, S + 500)
    ops.release_bwd_workspace()
    assert torch.equal(dq, dq2) and torch.isfinite(dq.float()).all()
    assert (dkv.float() - dkv2.float()).abs().max().item() <= 2 * 2.0 ** -8 * dkv.float().abs().max().item()


def test_backward_chunked_workspace_through_the_c_abi(gpu):
    """A workspace too small for all queries at once makes the library walk the queries in chunks;
    the result must not change."""
    from loongforge_amd import _lib, ops

    inp = O.make_mla_inputs(300, 128, 128, seed=7)
    q, kv, idx, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, 0, inp.sm_scale)
    dq1, dkv1 = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, 0, inp.sm_scale)
    lib = _lib.load()
    small = lib.dsa_sparse_mla_bwd_workspace_bytes(100, 128, 300, 128)
    ws = torch.empty(small, dtype=torch.uint8, device=gpu)
    dq2, dkv2 = torch.empty_like(q), torch.empty_like(kv)
    rc = lib.dsa_sparse_mla_bwd(q.data_ptr(), kv.data_ptr(), out.data_ptr(), do.data_ptr(), idx.data_ptr(),
                                lse.data_ptr(), 300, 128, 300, 128, 0, inp.sm_scale, 512, dq2.data_ptr(),
                                dkv2.data_ptr(), ws.data_ptr(), small, None)
    assert rc == 0, lib.dsa_last_error()
    torch.cuda.synchronize()
    assert torch.equal(dq1, dq2)
    assert (dkv1.float() - dkv2.float()).abs().max().item() <= 2 * 2.0 ** -8 * dkv1.float().abs().max().item()
    # the smallest accepted workspace, and a repeated id in the last chunk: every chunk's dQ is NaN, not only the last's
    least = lib.dsa_sparse_mla_bwd_workspace_bytes_min(300, 128, 300, 128)
    assert 0 < least <= small
    idx_dup = inp.idx.clone()
    idx_dup[299, 5] = idx_dup[299, 9]
    idx_dup = idx_dup.to(gpu)
    wl = torch.empty(least, dtype=torch.uint8, device=gpu)
    rc = lib.dsa_sparse_mla_bwd(q.data_ptr(), kv.data_ptr(), out.data_ptr(), do.data_ptr(), idx_dup.data_ptr(),
                                lse.data_ptr(), 300, 128, 300, 128, 0, inp.sm_scale, 512, dq2.data_ptr(),
                                dkv2.data_ptr(), wl.data_ptr(), least, None)
    assert rc == 0, lib.dsa_last_error()
    torch.cuda.synchronize()
    assert torch.isnan(dq2.float()).all() and torch.isnan(dkv2.float()).all()
    tiny = torch.empty(1024, dtype=torch.uint8, device=gpu)
    rc = lib.dsa_sparse_mla_bwd(q.data_ptr(), kv.data_ptr(), out.data_ptr(), do.data_ptr(), idx.data_ptr(),
                                lse.data_ptr(), 300, 128, 300, 128, 0, inp.sm_scale, 512, dq2.data_ptr(),
                                dkv2.data_ptr(), tiny.data_ptr(), 1024, None)
    assert rc == -3 and b"workspace" in lib.dsa_last_error()


def test_backward_op_workspace_is_capped_and_kept(gpu, monkeypatch):
    """ops.sparse_mla_bwd keeps its workspace between calls (one allocation per device, not one per call) and
    honours DSA_BWD_WORKSPACE_GIB: a cap below the full size makes the library walk the queries in chunks."""
    from loongforge_amd import _lib, ops

    inp = O.make_mla_inputs(300, 128, 128, seed=8)
    q, kv, idx, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, 0, inp.sm_scale)
    ops._BWD_WS.clear()
    dq1, dkv1 = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, 0, inp.sm_scale)
    kept = ops._BWD_WS[gpu.index or 0]
    full = _lib.load().dsa_sparse_mla_bwd_workspace_bytes(300, 128, 300, 128)
    assert kept.numel() == full
    ops.sparse_mla_bwd(q, kv, out, do, idx, lse, 0, inp.sm_scale)
    assert ops._BWD_WS[gpu.index or 0] is kept                      # reused, not reallocated
    ops._BWD_WS.clear()
    small = _lib.load().dsa_sparse_mla_bwd_workspace_bytes(100, 128, 300, 128)
    monkeypatch.setenv("DSA_BWD_WORKSPACE_GIB", repr(small / 2 ** 30))
    dq2, dkv2 = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, 0, inp.sm_scale)
    assert ops._BWD_WS[gpu.index or 0].numel() <= small + 256 < full
    assert torch.equal(dq1, dq2)
    assert (dkv1.float() - dkv2.float()).abs().max().item() <= 2 * 2.0 ** -8 * dkv1.float().abs().max().item()
    ops._BWD_WS.clear()


def test_backward_on_two_streams_at_once(gpu):
    """Backward passes that overlap on two streams do not share a workspace: the results are those of passes one by one."""
    from loongforge_amd import ops

    inp = [O.make_mla_inputs(300, 64, 128, seed=s) for s in (1, 2)]
    args = []
    for i in inp:
        q, kv, idx, do = i.q.to(gpu), i.kv.to(gpu), i.idx.to(gpu), i.dout.to(gpu)
        out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, 0, i.sm_scale)
        args.append((q, kv, out, do, idx, lse, 0, i.sm_scale))
    want = [ops.sparse_mla_bwd(*a) for a in args]
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream(), torch.cuda.Stream()], [[], []]
    for _ in range(4):
        for n, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[n].append(ops.sparse_mla_bwd(*args[n]))
    torch.cuda.synchronize()
    for n in range(2):
        assert all(torch.equal(g, w) for pair in got[n] for g, w in zip(pair, want[n]))
    ops._BWD_WS.clear()


def test_argument_errors(gpu):
    from loongforge_amd import ops

    q = torch.zeros(8, 128, 576, dtype=torch.bfloat16, device=gpu)
    kv = torch.zeros(8, 576, dtype=torch.bfloat16, device=gpu)
    with pytest.raises(ValueError, match="multiple of 64"):
        ops.sparse_mla_fwd(q, kv, torch.zeros(8, 48, dtype=torch.int32, device=gpu))
    with pytest.raises(ValueError, match="576"):
        ops.sparse_mla_fwd(q[..., :512].contiguous(), kv, torch.zeros(8, 64, dtype=torch.int32, device=gpu))
    with pytest.raises(ValueError, match="head count"):
        ops.sparse_mla_fwd(q[:, :16].contiguous(), kv, torch.zeros(8, 64, dtype=torch.int32, device=gpu))
    with pytest.raises(ValueError, match="d_v"):
        ops.sparse_mla_fwd(q, kv, torch.zeros(8, 64, dtype=torch.int32, device=gpu), d_v=256)
    # the backward keeps one bit per key in LDS: more than 1 228 800 keys are turned down with a message
    big = torch.zeros(1_300_000, 576, dtype=torch.bfloat16, device=gpu)
    ids = torch.zeros(8, 64, dtype=torch.int32, device=gpu)
    out, lse, _ = ops.sparse_mla_fwd(q, big, ids, 1_300_000)
    with pytest.raises(ValueError, match="at most"):
        ops.sparse_mla_bwd(q, big, out, torch.zeros_like(out), ids, lse, 1_300_000)


@pytest.mark.parametrize("S,H,K,heads,q_start,skv,seed", [
    (200, 128, 128, 128, 40, 300, 3),
    (96, 128, 64, 16, 0, None, 5),          # 16 real heads padded to 128: only they count
    (70, 64, 192, 64, 0, None, 8),
])
def test_attn_dist_from_q_kv_lse_matches_oracle_and_the_logits_path(gpu, S, H, K, heads, q_start, skv, seed):
    from loongforge_amd import ops

    inp = O.make_mla_inputs(S, H, K, seed=seed, skv=skv, q_start=q_start)
    idx = inp.idx.clone()
    idx[5, 3] = -1
    q, kv, ids = inp.q.to(gpu), inp.kv.to(gpu), idx.to(gpu)
    out, lse, p_out = ops.sparse_mla_fwd(q, kv, ids, q_start, inp.sm_scale, 512, True, torch.float32)
    got = ops.attn_dist_qk(q, kv, ids, lse, q_start, inp.sm_scale, heads)
    _, rl, rp = O.sparse_mla_fwd(inp.q, inp.kv, idx, q_start, inp.sm_scale, 512)
    ref = O.attn_dist_from_lse(inp.q, inp.kv, idx, rl, q_start, inp.sm_scale, heads)
    assert (got.cpu() - ref).abs().max().item() <= 2e-5
    assert (got.cpu() - O.attn_dist(rp[:, :heads], inp.sm_scale)).abs().max().item() <= 2e-5
    # the route through the materialised logits gives the same distribution
    via_logits = ops.attn_dist(p_out[:, :heads], inp.sm_scale)
    assert (got - via_logits).abs().max().item() <= 2e-5
    assert ((got.sum(-1) - 1.0).abs() <= 1e-4).all() and (got[5, 3] == 0).all()


@pytest.mark.parametrize("S,H,K,block", [
    (300, 64, 192, 100),              # the whole: two workgroups to a unit; a block by itself would share its queries' heads out
    (300, 64, 192, 256),              # the last block of 44 alone
    (300, 32, 128, 200),
    (200, 128, 256, 64),
    (140, 128, 320, 96),              # two roles; blocks of 96 and 44
    (40, 64, 2048, 16),               # in four ranges of slots; a block alone in eight
    (20, 32, 2048, 9),                # the same, and the ranges' sums of few queries are put together another way
    (10, 128, 512, 3),                # one workgroup for a query's slots; a block alone in ranges
])
def test_forward_with_distribution_in_blocks_is_that_of_the_whole(gpu, S, H, K, block):
    from loongforge_amd import ops

    heads = H - 5
    q_start = K + 50
    inp = O.make_mla_inputs(S, H, K, seed=S + H, q_start=q_start)
    q, kv, ids, sink = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), torch.linspace(-2, 2, H).to(gpu)
    assert any(mla_form(n, H, K) != mla_form(S, H, K) for n in (block, S % block))          # by themselves
    for sk in (None, sink):
        out, lse, p_out = ops.sparse_mla_fwd(q, kv, ids, q_start, inp.sm_scale, 512, True, attn_sink=sk)
        want = out, lse, ops.attn_dist(p_out[:, :heads], inp.sm_scale)
        for n in (block, S):
            got = ops.sparse_mla_fwd_dist(q, kv, ids, q_start, inp.sm_scale, 512, heads, n, sk)
            assert all(torch.equal(g, w) for g, w in zip(got, want)), n


@pytest.mark.parametrize("form,ranges,S,H,K", MLA_FORMS)
@pytest.mark.parametrize("misaligned", [False, True])
def test_distribution_of_short_rows_reads_only_what_the_forward_wrote(gpu, form, ranges, S, H, K, misaligned):
    """The passing logits of tiles without a valid slot are neither written nor read: with NaN in their place, rows that end early,
    have holes of whole tiles or no slot at all give the distribution of the logits that the caller can ask for, bit for bit.
    (A buffer that starts between two 32-byte pieces is written and read whole.)"""
    from loongforge_amd import _lib, ops

    assert mla_form(S, H, K) == (form, ranges)
    inp = O.make_mla_inputs(S, H, K, seed=S, skv=K + S, q_start=K)
    idx = inp.idx.clone()
    for i in range(0, S, 2):
        idx[i, (37 * i) % K:] = -1
    idx[S // 2, :32] = -1
    idx[S // 3] = K + S + 5                     # behind the keys
    if S > 2:
        idx[1, 32:] = K + 2                     # behind the query
        idx[2, 5:] = -1
    q, kv, ids = inp.q.to(gpu), inp.kv.to(gpu), idx.to(gpu)
    out, lse, p_out = ops.sparse_mla_fwd(q, kv, ids, K, inp.sm_scale, 512, True)
    heads = H - 3
    want = ops.attn_dist(p_out[:, :heads], inp.sm_scale)
    got = ops.sparse_mla_fwd_dist(q, kv, ids, K, inp.sm_scale, 512, heads, S)
    assert torch.equal(got[0], out) and torch.equal(got[1], lse) and torch.equal(got[2], want)
    lib = _lib.load()
    off = 8 if misaligned else 0
    logits = torch.full((S * H * K + 16,), float("nan"), dtype=torch.bfloat16, device=gpu)[off:]
    out2, lse2, dist2 = torch.empty_like(out), torch.empty_like(lse), torch.full_like(want, float("nan"))
    n = lib.dsa_sparse_mla_fwd_workspace_bytes(S, H, K + S, K)
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device=gpu)
    rc = lib.dsa_sparse_mla_fwd_dist(q.data_ptr(), kv.data_ptr(), ids.data_ptr(), S, S, H, K + S, K, K, inp.sm_scale, 512, out2.data_ptr(),
                                     lse2.data_ptr(), None, heads, dist2.data_ptr(), logits.data_ptr(), ws.data_ptr(), n,
                                     torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.dsa_last_error()
    assert torch.equal(out2, out) and torch.equal(lse2, lse)
    # (element by element the sums of a head are grouped differently: a few roundings of 2**-24 of values of one sign)
    assert torch.equal(dist2, want) if not misaligned else torch.allclose(dist2, want, rtol=2e-6, atol=0)


def test_attn_dist_from_q_kv_lse_with_sink_is_the_softmax_over_the_slots(gpu):
    from loongforge_amd import ops

    inp = O.make_mla_inputs(120, 128, 64, seed=12)
    sink = torch.linspace(-3, 3, 128)
    q, kv, ids = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu)
    out, lse, p_out = ops.sparse_mla_fwd(q, kv, ids, 0, inp.sm_scale, 512, True, torch.float32, attn_sink=sink.to(gpu))
    got = ops.attn_dist_qk(q, kv, ids, lse, 0, inp.sm_scale, 128, attn_sink=sink.to(gpu))
    _, _, rp = O.sparse_mla_fwd(inp.q, inp.kv, inp.idx, 0, inp.sm_scale, 512)
    assert (got.cpu() - O.attn_dist(rp, inp.sm_scale)).abs().max().item() <= 5e-5


def test_random_shapes_forward_backward_distribution(gpu):
    """Sixteen seeded random shapes (32 - 128 heads, 1 - 8 tiles per query, chunk offsets, longer key arrays, slot
    lists with holes): forward, backward by the parity rule, bit-equal reruns, recomputed attention distribution."""
    import random

    from loongforge_amd import ops

    rng = random.Random(1234)
    for case in range(16):
        H = rng.choice([32, 64, 96, 128])
        K = 64 * rng.randint(1, 8)
        S = rng.randint(1, 160)
        q_start = rng.choice([0, 0, rng.randint(1, 300)])
        skv = q_start + S + rng.choice([0, 0, rng.randint(1, 100)])
        seed = rng.randint(0, 10 ** 6)
        name = "case %d S=%d H=%d K=%d q_start=%d skv=%d seed=%d" % (case, S, H, K, q_start, skv, seed)
        print(name, flush=True)
        inp = O.make_mla_inputs(S, H, K, seed=seed, skv=skv, q_start=q_start)
        if rng.random() < 0.3:
            holes = torch.rand(inp.idx.shape, generator=torch.Generator().manual_seed(seed)) < 0.3
            inp.idx[holes] = -1
        q, kv, idx, do = inp.q.to(gpu), inp.kv.to(gpu), inp.idx.to(gpu), inp.dout.to(gpu)
        out, lse, _ = ops.sparse_mla_fwd(q, kv, idx, q_start, inp.sm_scale)
        ro, rl, _ = O.sparse_mla_fwd(inp.q, inp.kv, inp.idx, q_start, inp.sm_scale)
        assert_close(out, ro, name + " out", atol=2e-2, rtol=0)
        fin = torch.isfinite(rl)
        assert torch.equal(torch.isfinite(lse.cpu()), fin), name
        assert_close(lse.cpu()[fin], rl[fin], name + " lse", atol=1e-3, rtol=0)
        dq, dkv = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, q_start, inp.sm_scale)
        dq2, dkv2 = ops.sparse_mla_bwd(q, kv, out, do, idx, lse, q_start, inp.sm_scale)
        assert torch.equal(dq, dq2) and torch.equal(dkv, dkv2), name
        assert_mla_grads(dq, dkv, inp.q, inp.kv, inp.idx, inp.dout, q_start, inp.sm_scale, name=name, out=out, lse=lse)
        target = ops.attn_dist_qk(q, kv, idx, lse, q_start, inp.sm_scale, H)
        ref = O.attn_dist_from_lse(inp.q, inp.kv, inp.idx, lse.cpu(), q_start, inp.sm_scale, H)
        assert_close(target, ref, name + " attn_dist", atol=1e-3, rtol=1e-2)


def test_recomputed_distribution_refuses_host_tensors(gpu):
    """Keys, ids and statistics are read by the kernel as well as the queries: none of them may be host memory."""
    from loongforge_amd import ops

    args = [torch.zeros(4, 32, 576, dtype=torch.bfloat16), torch.zeros(9, 576, dtype=torch.bfloat16), torch.zeros(4, 64, dtype=torch.int32),
            torch.zeros(4, 32)]
    for host in range(4):
        with pytest.raises(RuntimeError, match="HIP device"):
            ops.attn_dist_qk(*[t if i == host else t.to(gpu) for i, t in enumerate(args)], 0, 0.1)


@pytest.mark.parametrize("H", [7, 8, 9, 33, 64, 128])
@pytest.mark.parametrize("K", [8, 64, 200, 256, 264, 512])
def test_attn_dist_of_short_lists(gpu, H, K):
    """Rows of up to 512 slots, four heads of a wave together and up to 256 slots two side by side: against 64 bits, with heads and slots of
    -inf, a head far above the others, strided rows; NaN and +inf reach their query alone."""
    from loongforge_amd import ops

    g = torch.Generator().manual_seed(H * K)
    S, scale = 37, 192 ** -0.5
    wide = (torch.randn(S, H + 2, K + 8, generator=g) * 30).to(torch.bfloat16)
    p = wide[:, 1:H + 1, :K]
    p[torch.rand(S, H, K, generator=g) < 0.2] = -float("inf")
    p[3, : H // 2] = -float("inf")
    p[4] = -float("inf")
    p[5, :, K // 2:] = -float("inf")
    p[6, H - 1] *= 100
    pd = wide.to(gpu)[:, 1:H + 1, :K]
    got = ops.attn_dist(pd.contiguous(), scale)
    z = p.double() * scale
    ref = torch.nan_to_num(torch.softmax(z, -1), 0.0).sum(1) / H        # a head without a slot adds nothing
    # a term's exponent and product in 32 bits, sums of K and H of them
    assert (got.double().cpu() - ref).abs().max().item() <= 2.0 ** -23 * (8 + 64)
    assert ((got.double().cpu() - ref).abs() <= 2e-5 * ref + 1e-30).all()
    assert (got[4] == 0).all()
    bad = pd.contiguous().clone()
    bad[7, H - 1, K - 1] = float("nan")
    bad[8, 0, 0] = float("inf")
    mixed = ops.attn_dist(bad, scale)
    keep = torch.ones(S, dtype=torch.bool)
    keep[7:9] = False
    assert torch.equal(mixed[keep.to(gpu)], got[keep.to(gpu)]) and torch.isnan(mixed[7]).any() and torch.isnan(mixed[8]).any()
