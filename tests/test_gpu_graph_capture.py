"""The kernels record into a HIP graph: the library allocates nothing, clears nothing with memset
nodes and never synchronises, so indexer -> top-k -> attention forward -> backward -> attention
distribution can be captured once and replayed.  Every replay is compared bit for bit with the
eager result on the same inputs (all kernels are deterministic), with eager work and
synchronisations between the replays."""
import pytest
import torch

from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu


def _pipeline(ops, t):
    q8, qs = ops.quant_rowwise_e4m3(t["iq"])
    k8, ksc = ops.quant_rowwise_e4m3(t["ik"])
    wsd = t["w"] * qs * 128 ** -0.5
    scores, ids = ops.indexer_topk(q8, wsd, k8, ksc, t["ks"], t["ke"], t["K"], True)
    out, lse, p_out = ops.sparse_mla_fwd(t["q"], t["kv"], ids, 0, t["sm_scale"], 512, return_p_out=True)
    dq, dkv = ops.sparse_mla_bwd(t["q"], t["kv"], out, t["dout"], ids, lse, 0, t["sm_scale"])
    target = ops.attn_dist(p_out, t["sm_scale"])
    d_q8, d_k8, d_qw = ops.indexer_bwd(torch.where(ids >= 0, target, torch.zeros_like(target)), q8, k8, ksc, wsd, ids)
    return dict(scores=scores, ids=ids, out=out, lse=lse, dq=dq, dkv=dkv, target=target, d_q8=d_q8, d_k8=d_k8, d_qw=d_qw)


def test_pipeline_replays_from_a_graph(gpu):
    from loongforge_amd import ops

    S, H, K = 512, 128, 256
    ks, ke = O.indexer_window(S, 0, None)
    t = dict(K=K, sm_scale=192 ** -0.5, ks=ks.to(gpu), ke=ke.to(gpu))

    def fill(seed):
        inp = O.make_mla_inputs(S, H, K, seed=seed)
        iq, ik, w = O.make_indexer_inputs(S, 64, 128, seed=seed + 40)
        return dict(q=inp.q, kv=inp.kv, dout=inp.dout, iq=iq, ik=ik, w=w)

    static = {k: v.to(gpu) for k, v in fill(0).items()}
    t.update(static)
    _pipeline(ops, t)                                  # untimed first call outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = _pipeline(ops, t)
    for seed in (1, 2, 3):
        fresh = {k: v.to(gpu) for k, v in fill(seed).items()}
        eager = _pipeline(ops, dict(t, **fresh))
        torch.cuda.synchronize()
        for k, v in fresh.items():
            static[k].copy_(v)
        graph.replay()
        torch.cuda.synchronize()
        for name, ref in eager.items():
            assert torch.equal(captured[name], ref), "replay with seed %d differs from the eager run in %s" % (seed, name)


def test_packed_indexer_replays_with_other_sequences(gpu):
    """The windows of packed sequences are part of the graph: a replay follows the lengths that are in the tensor then.  Queries
    that no sequence holds, which an eager call refuses, select nothing."""
    from loongforge_amd import dsa_fused_kernels as K
    from loongforge_amd.megatron_compat import PackedSeqParams

    S, topk = 300, 64
    iq, ik, w = (t.to(gpu) for t in O.make_indexer_inputs(S, 32, 128, seed=3))
    cu = torch.tensor([0, 100, S], dtype=torch.int32, device=gpu)
    run = lambda c: K.DSAIndexerKernel()(iq, ik, w, topk, 0, PackedSeqParams(qkv_format="thd", cu_seqlens_q=c, cu_seqlens_kv=c))   # noqa: E731
    run(cu)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        scores, ids = run(cu)
    for lengths in ([0, 100, S], [0, 7, S], [0, 250, S], [0, 100, 200]):
        now = torch.tensor(lengths, dtype=torch.int32, device=gpu)
        full = now.clone()
        full[-1] = S                                   # the held queries' windows do not depend on where the last sequence ends
        want_s, want_i = run(full)
        torch.cuda.synchronize()
        cu.copy_(now)
        graph.replay()
        torch.cuda.synchronize()
        held = lengths[-1]
        assert torch.equal(ids[:held], want_i[:held]) and torch.equal(scores[:held], want_s[:held]), lengths
        assert (ids[held:] == -1).all() and (scores[held:] == float("-inf")).all(), lengths
    with pytest.raises(ValueError, match="200 tokens"):
        run(cu)
