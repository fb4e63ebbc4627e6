"""Shape propagation without a device: the entry points that take fake tensors."""
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

BF = torch.bfloat16


def test_indexer_and_its_front_end_take_fake_tensors():
    from loongforge_amd import dsa_fused_kernels as K, ops
    from loongforge_amd.dsa_fused import rotate_activation
    from loongforge_amd.megatron_compat import RotaryEmbedding, apply_rotary_pos_emb

    with FakeTensorMode():
        new = lambda *shape, dtype=BF: torch.empty(*shape, dtype=dtype, device="cuda")                # noqa: E731
        x = new(16, 1, 8, 64)
        assert rotate_activation(x).shape == x.shape
        assert apply_rotary_pos_emb(x, RotaryEmbedding(64, 1.0).to("cuda")(16)).shape == x.shape
        for heads, dim, hp in ((32, 128, 32), (4, 64, 32), (64, 128, 64)):
            scores, ids = K.DSAIndexerKernel()(new(48, heads, dim), new(48, dim), new(48, heads), 64, 0, None)
            assert scores.shape == ids.shape == (48, 64)
            f32 = dict(dtype=torch.float32)
            grads = ops.indexer_grads(scores, new(48, hp, 128, dtype=torch.float8_e4m3fn), new(48, 128, dtype=torch.float8_e4m3fn),
                                      new(48, **f32), new(48, hp, **f32), ids, new(48, hp, **f32), 1.0, heads, dim, (BF, BF, BF))
            assert [t.shape for t in grads[:3]] == [(48, heads, dim), (48, dim), (48, heads)]
            assert all(t.dtype == BF for t in grads[:3])
