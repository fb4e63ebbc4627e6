"""The native host layer's decisions that need no device: layouts, refusals."""
import pytest
import torch

BF = torch.bfloat16


def _views():
    r = lambda *shape: torch.arange(torch.Size(shape).numel(), dtype=torch.float32).to(BF).view(shape)             # noqa: E731
    yield "contiguous", r(5, 2, 3, 8)
    yield "packed", r(5, 3, 8)
    yield "one sequence, batch first", r(1, 5, 2, 64).transpose(0, 1)
    yield "two sequences, batch first", r(2, 5, 2, 64).transpose(0, 1)
    yield "one token, batch first", r(2, 1, 3, 8).transpose(0, 1)
    yield "one token of one sequence", r(1, 1, 3, 8).as_strided((1, 1, 3, 8), (7, 5, 8, 1))
    yield "one head, head first", r(1, 5, 2, 8).permute(1, 2, 0, 3)
    yield "heads first", r(3, 5, 2, 8).permute(1, 2, 0, 3)
    yield "leading part of a row", r(5, 2, 3, 12)[..., :8]
    yield "every other element of a row", r(5, 2, 3, 16)[..., ::2]
    yield "one sequence, batch first, leading part", r(1, 5, 2, 12).transpose(0, 1)[..., :8]
    yield "every other token", r(10, 1, 3, 8)[::2]
    yield "every other sequence", r(5, 4, 3, 8)[:, ::2]
    yield "shared by the heads", r(5, 2, 1, 8).expand(5, 2, 3, 8)
    yield "shared by the tokens", r(1, 1, 3, 8).expand(5, 1, 3, 8)


@pytest.mark.parametrize("name,t", list(_views()), ids=lambda v: v if isinstance(v, str) else "")
def test_rows_with_one_token_pitch_are_the_tensor(name, t):
    """What the kernel reads at pitch * token + head stride * head + element is the tensor, and lies inside its storage."""
    from loongforge_amd import _lib

    x, pitch = _lib.load_host().token_rows(t)
    tokens, (heads, d) = t.shape[:-2].numel(), t.shape[-2:]
    assert x.stride(-1) == 1
    last = x.storage_offset() + (tokens - 1) * pitch + (heads - 1) * x.stride(-2) + d - 1
    assert last < x.untyped_storage().nbytes() // x.element_size()
    assert torch.equal(x.as_strided((tokens, heads, d), (pitch, x.stride(-2), 1)), t.reshape(tokens, heads, d))


@pytest.mark.parametrize("shape", [(8,), (5, 8), (2, 5, 2, 3, 8)])
def test_rope_in_rounded_steps_refuses_other_dimensions(shape):
    """Two dimensions would be walked as if the tokens were heads as well, behind the storage."""
    from loongforge_amd import ops

    with pytest.raises(ValueError, match="expected"):
        ops.rope_steps(torch.zeros(shape, dtype=BF), torch.zeros(5, 1, 1, 8))


@pytest.mark.parametrize("n,k,emb", [(128, 512, 64), (512, 128, 32)])
def test_absorbed_query_leaves_other_widths_to_the_two_kernels(n, k, emb):
    from loongforge_amd import ops

    q_up, w = torch.zeros(3, 2, k + emb, dtype=BF), torch.zeros(2, n, k, dtype=BF)
    assert ops.absorbed_query(q_up, w, torch.zeros(3, emb), torch.zeros(3, emb), None, ops.ROPE_SPLIT) is None


def test_indexer_front_end_refuses_an_empty_batch():
    """The positions' default is token // batch: no batch is an error of the caller's, not a division by zero."""
    from loongforge_amd import ops

    x, table = torch.zeros(4, 128, dtype=BF), torch.zeros(4, 64)
    for batch in (0, -1):
        with pytest.raises(ValueError, match="batch must be positive"):
            ops.indexer_front_e4m3(x, cos=table, sin=table, pairing=ops.ROPE_SPLIT, batch=batch)


def test_workspace_of_an_indexer_without_keys():
    """The size is asked for before the arguments are checked: no keys must not be divided by."""
    from loongforge_amd import _lib

    lib = _lib.load()
    assert lib.dsa_indexer_topk_workspace_bytes(5, 0, 64) == 0
    with pytest.raises(ValueError, match="Sk=0"):
        _lib.check(lib.dsa_indexer_topk_fwd(None, None, None, None, None, None, 5, 64, 0, 64, 1, None, None, 256, 0, None), "no keys")


def test_tensors_of_one_call_live_on_one_device():
    """A kernel would read the other device's memory.  (Fake tensors: two devices without any.)"""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from loongforge_amd import _lib, ops

    with FakeTensorMode():
        new = lambda *shape, dtype=BF, dev=0: torch.empty(shape, dtype=dtype, device="cuda:%d" % dev)             # noqa: E731
        t, angles = new(5, 1, 2, 64), new(5, 1, 1, 64, dtype=torch.float32, dev=1)
        p, cos = new(5, 2, 64), new(5, 64, dtype=torch.float32, dev=1)
        logits, k8 = new(5, 32, 128, dtype=torch.uint8), new(9, 128, dtype=torch.uint8, dev=1)
    host = _lib.load_host()
    with pytest.raises(RuntimeError, match="on one device; got cuda:0 and cuda:1"):
        host.rope_steps(t, angles, 1.0, False, False)
    with pytest.raises(RuntimeError, match="on one device; got cuda:0 and cuda:1"):
        ops.rope_rows(p, p, cos, cos, 0, 0)
    with pytest.raises(RuntimeError, match="on one device; got cuda:0 and cuda:1"):
        ops._need_gpu(None, logits, None, k8)


def test_host_layer_is_rebuilt_for_another_torch(tmp_path, monkeypatch):
    """An extension compiled against another torch does not load; a build without --force has to notice."""
    from types import SimpleNamespace

    from loongforge_amd.csrc import build

    runs = []

    def compiler(cmd, **_):
        runs.append(cmd)
        open(cmd[cmd.index("-o") + 1], "w").close()
        return SimpleNamespace(returncode=0, stdout="", stderr="")

    monkeypatch.setattr(build, "OBJ_DIR", str(tmp_path))
    monkeypatch.setattr(build.subprocess, "run", compiler)
    for version, compiles in (("1.0", 1), ("1.0", 1), ("1.1", 2), ("1.1", 2)):
        monkeypatch.setattr(torch, "__version__", version)
        build._compile_host(False)
        assert len(runs) == compiles, version
    monkeypatch.setenv("CXX", "another")
    build._compile_host(False)
    assert len(runs) == 3
    build._compile_host(True)
    assert len(runs) == 4


@pytest.mark.parametrize("fused", [False, True])
def test_batched_products_of_the_absorption_have_contiguous_right_operands(fused, monkeypatch):
    """A bf16 batched product whose right operand is a transposed view has faulted the device; the gradients' products are
    given contiguous ones, whatever the layouts of the weights and the activations."""
    from types import SimpleNamespace

    from loongforge_amd import dsa_fused_kernels as K, ops

    seen, bmm = [], torch.bmm

    def product(a, b):
        seen.append(b.is_contiguous())
        return bmm(a, b)

    monkeypatch.setattr(torch, "bmm", product)
    monkeypatch.setattr(ops, "rope_rows", lambda *a, **k: None)
    rnd = lambda *shape: torch.randn(*shape, generator=torch.Generator().manual_seed(0), dtype=torch.float64)      # noqa: E731
    a, w, grad = rnd(5, 3, 192 if fused else 128), rnd(3, 128, 512).transpose(1, 2), rnd(5, 3, 576 if fused else 512)
    if fused:
        ctx = SimpleNamespace(saved_tensors=(a, w, None, None), args=(None, 1, 0, 128, 512, 64, a.shape), needs_input_grad=(True, True))
        d_a, d_w = K.FusedAbsorbRopeQuery.backward(ctx, grad)[:2]
    else:
        ctx = SimpleNamespace(saved_tensors=(a, w), needs_input_grad=(True, True, False))
        d_a, d_w = ops.MlaAbsorb.backward(ctx, grad)[:2]
    assert seen == [True, True]
    torch.testing.assert_close(d_a[..., :128], torch.einsum("shn,hnk->shk", grad[..., :512], w))
    torch.testing.assert_close(d_w, torch.einsum("shn,shk->hnk", grad[..., :512], a[..., :128]))


def test_backward_workspace_is_not_shared_between_streams(monkeypatch):
    """One buffer is kept per device, for the stream it was used on; another stream and a graph capture get their own."""
    from types import SimpleNamespace

    from loongforge_amd import ops

    now, empty = SimpleNamespace(stream=1, capturing=False), torch.empty
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: SimpleNamespace(cuda_stream=now.stream))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: now.capturing)
    monkeypatch.setattr(torch, "empty", lambda n, dtype, device: empty(n, dtype=dtype))
    monkeypatch.setattr(ops, "_BWD_WS", {})
    get = lambda n: ops._bwd_workspace(n, torch.device("cuda", 0))[0]                # noqa: E731
    first = get(1000)
    assert get(500) is first and get(1000) is first
    now.stream = 2
    second = get(500)
    assert second is not first and get(400) is second
    now.capturing = True
    captured = get(300)
    assert captured is not second and ops._BWD_WS[0] is second      # the graph's buffer is nobody else's, the kept one stays
    now.capturing = False
    assert get(300) is second
    now.stream = 1
    assert get(300) is not second and len(ops._BWD_WS) == 1
