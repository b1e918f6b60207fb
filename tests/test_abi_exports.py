"""The C-ABI library loads on the CPU host, exports every symbol include/ntlowbit.h
declares, and rejects bad arguments before touching the GPU."""

from __future__ import annotations

import ctypes
import os
import re

import pytest

from conftest import PKG_PARENT, ROOT

HEADER = os.path.join(ROOT, "include", "ntlowbit.h")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    decls = re.findall(r"^(?:int64_t|int|const char\*)\s+(ntlb_\w+)\s*\(([^;]*)\);", text, flags=re.M)
    out = {}
    for name, args in decls:
        args = " ".join(args.split())
        n = 0 if args in ("", "void") else args.count(",") + 1
        out[name] = n
    return out


def test_header_declares_entry_points():
    d = _declared()
    assert "ntlb_gemm_blockscaled" in d and "ntlb_quant_tile_1x128" in d
    assert len(d) >= 8


def test_library_exports_every_declared_symbol():
    from lowbit import _lib

    L = _lib.lib()
    for name in _declared():
        assert hasattr(L, name), name


def test_python_binding_matches_header_arity():
    from lowbit import _lib

    d = _declared()
    assert set(d) == set(_lib.SIGNATURES), set(d) ^ set(_lib.SIGNATURES)
    for name, n in d.items():
        assert len(_lib.SIGNATURES[name]) == n, name


def test_abi_version_and_validation_without_gpu():
    from lowbit import _lib

    L = _lib.lib()
    assert L.ntlb_abi_version() == _lib.ABI_VERSION
    # Kp not a multiple of 128: rejected before any launch
    rc = L.ntlb_gemm_blockscaled(1, 16, 128, 16, 1, 0, 0, 16, 128, 16, 1, 0, 7, 4, 4, 100, None, 0, 16, 1, 4, None,
                                 None, None)
    assert rc == _lib.NTLB_EINVAL
    assert b"multiple of 128" in L.ntlb_last_error()
    # bad grid enum on the tile quantizer
    rc = L.ntlb_quant_tile_1x128(16, 1, 4, 128, 128, 5, 127, 0, 0, 0, 0, 16, 128, 16, 1, 1, None, 0, 0, None, None)
    assert rc == _lib.NTLB_EINVAL and b"grid" in L.ntlb_last_error()


def test_product_package_never_touches_the_oracle():
    pkg = os.path.join(PKG_PARENT, "lowbit")
    for fn in os.listdir(pkg):
        if fn.endswith(".py"):
            src = open(os.path.join(pkg, fn)).read()
            assert "oracle" not in src.replace("oracle-free", ""), fn


def test_ops_reject_cpu_tensors():
    import torch

    from lowbit import ops

    with pytest.raises(RuntimeError, match="ROCm device"):
        ops.quant_tile_1x128(torch.zeros(2, 128))


def test_ep_entry_points_validate_without_gpu():
    """The expert-parallel entry points reject bad shapes, enums and
    workspaces with NTLB_EINVAL and a message, before any launch; the record
    size follows the documented layout."""
    from lowbit import _lib

    L = _lib.lib()
    E = _lib.NTLB_EINVAL
    P = 4096  # a 16-byte aligned stand-in address: every call below returns before using it
    # record bytes: 128*ceil(H/128) codes, 4*ceil(H/128) scale bytes rounded to 16, 32 metadata bytes
    assert L.ntlb_ep_record_bytes(7168) == 7168 + 224 + 32
    assert L.ntlb_ep_record_bytes(200) == 256 + 16 + 32
    assert L.ntlb_ep_record_bytes(0) == 0
    # partition: n < 0, no buckets, too many buckets, bad key dtype / stride, short workspace
    part = L.ntlb_ep_partition
    assert part(P, 0, 4, -1, 1, 4, P, P, P, P, P, 64, None) == E
    assert part(P, 0, 4, 10, 1, 0, P, P, P, P, P, 64, None) == E
    assert part(P, 0, 4, 10, 1, 5000, P, P, P, P, P, 1 << 20, None) == E
    assert part(P, 2, 4, 10, 1, 4, P, P, P, P, P, 64, None) == E
    assert part(P, 0, 6, 10, 1, 4, P, P, P, P, P, 64, None) == E and b"key_stride" in L.ntlb_last_error()
    assert part(P, 0, 4, 1000, 1, 4, P, P, P, P, P, 8, None) == E and b"workspace" in L.ntlb_last_error()
    # unpack: ldc below the padded width; source ranks with offsets not ending at n; too many ranks
    offs = (ctypes.c_int64 * 3)(0, 2, 5)
    unpack = L.ntlb_ep_unpack_records
    assert unpack(P, 6, 200, P, 6, None, 0, P, 200, P, 1, 6, None, None, None, None, None, None) == E
    assert unpack(P, 6, 256, P, 6, ctypes.addressof(offs), 2, P, 256, P, 1, 6, None, None, None, P, None,
                  None) == E and b"recv_offsets" in L.ntlb_last_error()
    many = (ctypes.c_int64 * 258)(*([0] * 257 + [6]))
    assert unpack(P, 6, 256, P, 6, ctypes.addressof(many), 257, P, 256, P, 1, 6, None, None, None, P, None,
                  None) == E
    # combine: K above 32, H not a multiple of 8, unknown grid
    BF16 = 1  # NTLB_BF16 of include/ntlowbit.h
    comb = L.ntlb_ep_combine
    assert comb(P, 4, 256, P, 1, P, BF16, 2, 33, 1, P, BF16, 256, P, None) == E
    assert comb(P, 4, 250, P, 1, P, BF16, 2, 2, 1, P, BF16, 256, P, None) == E
    assert comb(P, 4, 256, P, 1, P, BF16, 2, 2, 7, P, BF16, 256, P, None) == E
    # return pack: a scale group that splits a 128-column tile
    ret = L.ntlb_ep_pack_return  # x bf16 (1), grid e4m3 (1), qmax 127, rounding nearest (0), rule 1
    assert ret(P, 1, 4, 256, 256, P, P, P, None, None, P, 100, 1, 127, 0, 1, 0, 0, P, None) == E
    assert b"scale group" in L.ntlb_last_error()
    # the split-K workspace size: zero for a K that is not whole 128-blocks
    assert L.ntlb_gemm_workspace_bytes(512, 1024, 1000) == 0


def test_workspace_sizes_follow_the_tile_rule():
    """split-K workspace only for products that run on 256x256 tiles: none for
    those on smaller tiles, on their own or as part of a linear call"""
    from lowbit import _lib

    L = _lib.lib()
    for m, n, kp in ((16, 4096, 4096), (512, 1024, 2304), (2048, 4096, 4096), (640, 768, 4608)):
        assert L.ntlb_gemm_workspace_bytes(m, n, kp) == 0, (m, n, kp)
    for m, n, kp in ((1500, 1600, 4608), (4100, 4000, 2304), (8192, 7168, 18432)):
        assert L.ntlb_gemm_workspace_bytes(m, n, kp) > 0, (m, n, kp)

    def plan(m, n, k):
        p = _lib.LinearPlan(M=m, N=n, K=k, ldx=k, ldw=k, x_dtype=_lib.BF16, w_dtype=_lib.BF16, grid=_lib.GRID_E4M3,
                            qmax=127)
        _lib.call("ntlb_linear_plan_init", ctypes.addressof(p))
        return p

    p = plan(16, 4096, 4096)
    assert p.forward_ws == p.recipe_ws == 0
    # dX on small tiles: workspace only for a dY of wide pitch, which the 256x256 tiles take
    p = plan(500, 1500, 4600)
    assert p.ste_free_pitch == 1536 + 8 and p.ste_ws > 0
    # 8192 x 7168 over 18432: every product fills the chip
    p = plan(8192, 18432, 7168)
    assert p.ste_free_pitch == 0 and p.ste_ws > 0 and p.recipe_ws > 0
