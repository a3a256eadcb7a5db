"""CPU checks of the C-ABI library and the host-side operator surface (no GPU needed)."""
import ctypes
import re
from pathlib import Path

import pytest
import torch

import superl8_amd
from superl8_amd import _C, _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "superl8_hip.h"


def _declared_symbols():
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(sl8_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(str(_lib.LIB_PATH))
    syms = _declared_symbols()
    assert len(syms) >= 15
    missing = [s for s in syms if not hasattr(lib, s)]
    assert not missing, f"not exported: {missing}"
    assert set(syms) == set(_lib.SIGNATURES), "ctypes table and header disagree"


def test_version_and_error_slot():
    lib = _lib.load()
    assert lib.sl8_version().startswith(b"superl8-hip")
    # argument validation runs before any device work, so it works without a GPU
    rc = lib.sl8_gemm_decode_q4k(None, None, None, None, 0, 1, 8, 100, None)
    assert rc == -1 and b"K%256" in lib.sl8_last_error()
    rc = lib.sl8_quantize_i8_rowwise(None, 7, 1, 1, None, None, None)
    assert rc == -1 and b"float16/bfloat16/float32" in lib.sl8_last_error()
    assert lib.sl8_quantize_i8_rowwise(None, 0, 0, 5, None, None, None) == 0  # empty is a no-op


def test_decode_split_heuristic_and_workspace():
    lib = _lib.load()
    # This build's auto split count: one split per ~2048 / (B * Hkv) workgroups
    # (a workgroup serves every query head of its KV head), at least 256 keys
    # per split, 1..256. The reference counts per query head (choose_n_splits,
    # attn_decode.cu:38-53) and picks 128 at config 3 where this picks 16; the
    # merged output is the same softmax either way (split invariance).
    cases = {  # (N, B, Hkv) -> splits, evaluated by hand
        (32768, 16, 8): 16,   # config 3: 2048 / 128
        (32768, 1, 8): 128,   # 2048 / 8 = 256, capped by N / 256 = 128
        (4096, 1, 1): 16,     # N / 256
        (1000, 1, 1): 4,      # ceil(1000 / 256)
        (200000, 1, 1): 256,  # 2048 -> capped at 256
        (100, 64, 64): 1,
        (1, 1, 1): 1,
        (0, 4, 4): 1,
    }
    for (n, b, hkv), want in cases.items():
        assert lib.sl8_choose_num_splits(n, b, hkv) == want, (n, b, hkv)
    assert lib.sl8_attn_int8_decode_workspace(16, 32, 128, 16) >= 16 * 16 * 32 * (128 + 2) * 4


def test_ops_reject_cpu_tensors():
    """No CPU path in the product: CPU tensors raise instead of silently falling back."""
    x = torch.randn(4, 256, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="CUDA"):
        superl8_amd.quantize_i8_rowwise(x)
    q = torch.randn(1, 2, 8, 64, dtype=torch.float16)
    with pytest.raises(RuntimeError):
        superl8_amd.attn_int8_fwd(q, q, q, internal_accuracy_gate=False)
    with pytest.raises(RuntimeError):
        superl8_amd.linear_q4k(x, torch.zeros(8, 144, dtype=torch.uint8))


class _Cuda:
    """What prologue_ok looks at in a contiguous GPU tensor."""
    is_cuda = True

    def __init__(self, *shape, device="cuda:0", dtype=torch.float16, ptr=0):
        self.shape, self.device, self.dtype, self._ptr = torch.Size(shape), torch.device(device), dtype, ptr

    def dim(self):
        return len(self.shape)

    def numel(self):
        return self.shape.numel()

    def data_ptr(self):
        return self._ptr

    def is_contiguous(self):
        return True


def test_fused_prologue_routing():
    """What the fused prologue takes: K and V of one type, shape rule and device (on two devices
    each is quantised by itself); any number of query rows and heads."""
    k = _Cuda(1, 8, 100, 128)
    assert _C.prologue_ok(k, _Cuda(1, 8, 100, 128))
    assert not _C.prologue_ok(k, _Cuda(1, 8, 100, 128, device="cuda:1"))
    assert not _C.prologue_ok(k, _Cuda(1, 8, 100, 128, dtype=torch.bfloat16))
    assert not _C.prologue_ok(k, _Cuda(1, 8, 100, 128, ptr=8))
    assert not _C.prologue_ok(_Cuda(1, 8, 100, 96)) and not _C.prologue_ok(_Cuda(1, 8, 0, 128))
    assert not _C.prologue_ok(_Cuda(1, 8, 1 << 23, 128)) and not _C.prologue_ok(_Cuda(65536, 1, 4, 128))
    assert _C.prologue_ok(k, q=_Cuda(1024, 64, 1, 128)) and _C.prologue_ok(k, q=_Cuda(1, 1, 1 << 23, 128))
    assert not _C.prologue_ok(k, q=_Cuda(1, 8, 1, 128, device="cuda:1"))
    assert not _C.prologue_ok(k, q=_Cuda(1, 8, 1, 128, ptr=2))
