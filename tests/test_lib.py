"""The C-ABI library loads and exports every symbol include/dsv41_hip.h declares (CPU: no compute calls)."""
import ctypes
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    txt = open(os.path.join(ROOT, "include", "dsv41_hip.h")).read()
    return sorted(set(re.findall(r"^\s*(?:int|long)\s+(dsv41_\w+)\s*\(", txt, re.M)))


def test_header_declares_entry_points():
    syms = declared_symbols()
    assert "dsv41_sattn2" in syms and "dsv41_topk_indices" in syms and len(syms) >= 11


def test_library_exports_every_declared_symbol():
    from dsv41_amd import _lib
    L = ctypes.CDLL(str(_lib.LIB_PATH))
    for s in declared_symbols():
        assert hasattr(L, s), s
    assert set(declared_symbols()) == set(_lib.SIGNATURES), "python signatures out of sync with the header"


def test_shims_refuse_cpu_tensors():
    import pytest
    import torch
    import dsv41_amd
    q = torch.zeros(1, 1, 4, 64, dtype=torch.bfloat16)
    kv = torch.zeros(1, 8, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):
        dsv41_amd.sparse_attn(q, kv, torch.zeros(4), torch.zeros(1, 1, 4, dtype=torch.int32), 0.1)


def test_workspace_query_is_pure():
    from dsv41_amd._lib import lib
    L = lib()
    assert L.dsv41_attn_workspace_bytes(2048, 64, 2176, 512, 0) == 0  # many rows: one split per row
    n = L.dsv41_attn_workspace_bytes(4, 64, 2176, 512, 0)
    assert n > 0 and n % 4 == 0


def test_split_plan_of_many_rows():
    """Key splits of the 64-head kernel (16 rows x 64 heads and more; 32 keys a tile, fp32 partials of 2 + 512 a split,
    row and head): 8 at most up to 128 tiles, one round of 256 workgroups over rows padded to 8 beyond, so that a long
    list is not left to half of the card."""
    from dsv41_amd._lib import lib
    for R, H, keys, want in [(16, 64, 640, 7), (16, 64, 2176, 8), (16, 64, 4096, 8), (16, 64, 4224, 15), (16, 64, 8320, 16),
                             (20, 64, 8320, 10), (24, 64, 8320, 10), (28, 64, 8320, 8), (8, 128, 8320, 16), (9, 128, 8320, 8),
                             (48, 64, 8320, 5), (88, 64, 640, 2), (104, 64, 640, 2), (112, 64, 640, 1), (128, 64, 768, 2),
                             (256, 64, 8320, 1)]:
        n = lib().dsv41_attn_workspace_bytes(R, H, keys, 512, 0)
        assert (n // (R * H * 514 * 4) if n else 1) == want, (R, H, keys)
    for dv in (64, 128, 256):  # narrow rows, short lists: one split
        assert lib().dsv41_attn_workspace_bytes(16, 64, 384, dv, 0) == 0
        assert lib().dsv41_attn_workspace_bytes(16, 64, 416, dv, 0) > 0
