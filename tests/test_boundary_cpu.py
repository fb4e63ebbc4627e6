"""Host-side checks that need no GPU: the C-ABI library loads and exports every symbol the header
declares, the Python binding table matches the header, and the product path refuses to run
without a HIP device instead of falling back to anything."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "dsa_hip.h")


def _declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(dsa_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    names = _declared_functions()
    for expected in ["dsa_quant_rowwise_e4m3", "dsa_indexer_logits", "dsa_topk", "dsa_indexer_topk_fwd",
                     "dsa_indexer_bwd", "dsa_sparse_mla_fwd", "dsa_sparse_mla_bwd", "dsa_attn_dist",
                     "dsa_last_error", "dsa_version"]:
        assert expected in names


def test_library_exports_every_declared_symbol():
    from loongforge_amd import _lib

    lib = ctypes.CDLL(_lib.LIB_PATH)
    for name in _declared_functions():
        assert hasattr(lib, name), name
    assert set(_lib.SIGNATURES) == set(_declared_functions())
    loaded = _lib.load()
    assert loaded.dsa_version() >= 1
    assert loaded.dsa_last_error() == b""


def test_binding_arity_matches_header():
    from loongforge_amd import _lib

    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    for name, (_, argtypes) in _lib.SIGNATURES.items():
        m = re.search(r"\b%s\s*\(([^;]*?)\)\s*;" % name, text, flags=re.S)
        assert m, name
        args = m.group(1).strip()
        n = 0 if args in ("", "void") else len([a for a in args.split(",") if a.strip()])
        assert n == len(argtypes), (name, n, len(argtypes))


def test_forms_of_the_sparse_mla_forward():
    """The sizes with which the GPU tests mean to reach every form of the forward do so."""
    from loongforge_amd import _lib
    from tests.gpu_util import MLA_FORMS, mla_form

    for form, ranges, S, H, K in MLA_FORMS:
        assert mla_form(S, H, K) == (form, ranges), (S, H, K)
    assert {f for f, _, _, _, _ in MLA_FORMS} == {0, 1, 2, 3, 4}
    # a block of a call: not of fewer queries than it has; nothing to spread, no workspace
    lib = _lib.load()
    assert lib.dsa_sparse_mla_fwd_block(None, None, None, 4, 5, 64, 9, 64, 0, 1.0, 512, None, None, None, 0, None, 0, None, 0, None) == -1
    assert lib.dsa_sparse_mla_fwd_block_workspace_bytes(4, 5, 64, 9, 2048) == 0
    assert lib.dsa_sparse_mla_fwd_block_workspace_bytes(40, 10, 64, 9, 2048) == 10 * 4 * 64 * (512 * 4 + 8) + 256
    assert lib.dsa_sparse_mla_fwd_workspace_bytes(40, 64, 9, 2048) == 40 * 4 * 64 * (512 * 4 + 8) + 256
    assert mla_form(4, 48, 64)[0] == mla_form(4, 64, 96)[0] == mla_form(4, 64, 16384)[0] == mla_form(0, 64, 64)[0] == -1


def test_no_cpu_fallback():
    from loongforge_amd import ops

    q = torch.zeros(4, 128, 576, dtype=torch.bfloat16)
    kv = torch.zeros(4, 576, dtype=torch.bfloat16)
    ids = torch.zeros(4, 64, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="HIP device"):
        ops.sparse_mla_fwd(q, kv, ids)
    with pytest.raises(RuntimeError, match="HIP device"):
        ops.quant_rowwise_e4m3(torch.zeros(2, 128, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError, match="HIP device"):
        ops.attn_dist(torch.zeros(2, 4, 64), 0.1)


def test_product_code_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "loongforge_amd")
    for base, _, files in os.walk(pkg):
        for f in files:
            if f.endswith(".py"):
                src = open(os.path.join(base, f)).read()
                assert not re.search(r"^\s*(from|import)\s+oracle", src, flags=re.M), f
                assert "dsa_oracle" not in src, f


def test_missing_library_fails_loudly(tmp_path, monkeypatch):
    from loongforge_amd import _lib

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libdsa_hip.so"))
    with pytest.raises(_lib.DsaError, match="missing"):
        _lib.load()


def test_bench_refuses_more_than_one_gpu():
    """The benchmark measures one GPU; asked for more it says so and exits without touching a device."""
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True,
                         timeout=120)
    assert res.returncode != 0
    assert "one GPU" in (res.stdout + res.stderr)


def test_groups_of_the_sparse_mla_backward():
    """Queries of 64 and 32 heads may be worked in groups of 2 and 4, from so many queries on, in every workspace from the smallest
    documented one on; queries of more heads and sizes that the backward does not take are not."""
    from loongforge_amd import _lib

    lib = _lib.load()
    at = ctypes.c_size_t(0)
    for H, G in ((64, 2), (32, 4)):
        for S in (192 * G, 1000, 1003):
            full, least = lib.dsa_sparse_mla_bwd_workspace_bytes(S, H, 500, 128), lib.dsa_sparse_mla_bwd_workspace_bytes_min(S, H, 500, 128)
            for nbytes in (full, (full + least) // 2, least):
                assert lib.dsa_sparse_mla_bwd_groups(S, H, 500, 128, nbytes, ctypes.addressof(at)) == G
                assert 0 < at.value and at.value % 256 == 0 and at.value + (S + G - 1) // G * 4 <= nbytes
        one_by_one = lib.dsa_sparse_mla_bwd_workspace_bytes(64, H, 500, 128)          # (less than `least`, and taken all the same)
        assert one_by_one < lib.dsa_sparse_mla_bwd_workspace_bytes_min(1024, H, 500, 128)
        assert lib.dsa_sparse_mla_bwd_groups(1024, H, 500, 128, one_by_one, None) == 1
        assert lib.dsa_sparse_mla_bwd_groups(192 * G - 1, H, 500, 128, full, None) == 1
    assert lib.dsa_sparse_mla_bwd_groups(1000, 128, 500, 128, 2 ** 40, None) == 1
    for S, H, Skv, K, nbytes in ((0, 64, 500, 128, 2 ** 40), (1000, 48, 500, 128, 2 ** 40), (1000, 64, 500, 100, 2 ** 40), (1000, 64, 0, 128, 2 ** 40),
                                 (1000, 64, 500, 2112, 2 ** 40), (1000, 64, 500, 128, 1 << 20)):
        assert lib.dsa_sparse_mla_bwd_groups(S, H, Skv, K, nbytes, None) == -1
