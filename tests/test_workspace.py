"""Workspace sizes, as the library's host code gives them (no GPU)."""
import ctypes as C

import pytest
import torch

from tyloquant_amd import _lib as L
from tyloquant_amd import runtime as R


class _Weight:
    """What QuantLinear.reserve() reads of a weight; its workspace lands on the CPU."""
    def __init__(self, desc, out, K):
        self.desc, self.out, self.out_per_expert, self.neuron_len = desc, out, out, K
        self.data, self._ws = torch.empty(0), R._Workspace()


def _weight(fmt, out, K):
    lib = L.lib()
    if fmt == "NVQ":
        d = L.NvqDesc()
        L.check(lib.mfq_hip_nvq_plan(9, 2, out, K, C.byref(d)))
        return "nvq", d, lambda M: lib.mfq_hip_nvq_gemm_workspace_bytes(C.byref(d), M), \
            lambda M: lib.mfq_hip_nvq_gemm_copy_workspace_bytes(C.byref(d), M)
    if fmt == "NEPQ":
        d = L.NepqDesc()
        L.check(lib.mfq_hip_nepq_plan(2, 4, out, K, C.byref(d)))
        return "nepq", d, lambda M: lib.mfq_hip_nepq_gemm_workspace_bytes(C.byref(d), out, M), \
            lambda M: lib.mfq_hip_nepq_gemm_copy_workspace_bytes(C.byref(d), out, M)
    if fmt == "MX":
        return "mx", None, lambda M: lib.mfq_hip_mx_gemm_rows_workspace_bytes(K, out, M), lambda M: 0
    if fmt == "NINT8-0":
        d = L.Nint8zDesc()
        L.check(lib.mfq_hip_nint8z_plan(out, K, C.byref(d)))
        return "nint8z", d, lambda M: lib.mfq_hip_nint8z_gemm_workspace_bytes(C.byref(d), M), lambda M: 0
    d = L.NintDesc()
    L.check(lib.mfq_hip_nint_plan(*fmt, out, K, C.byref(d)))
    return "nint", d, lambda M: lib.mfq_hip_nint_gemm_workspace_bytes(C.byref(d), M), lambda M: 0


@pytest.mark.parametrize("fmt", ["NVQ", "NEPQ", "MX", "NINT8-0", (4, 6, 32), (8, 7, 48), (4, 6, 40)], ids=str)
@pytest.mark.parametrize("out,K", [(2136, 1536), (784, 4096), (4096, 3072), (1000, 768)])
@pytest.mark.parametrize("most", [700, 2048])
def test_reserve_covers_every_batch(fmt, out, K, most):
    """reserve(most) samples the batches; none in between may ask for more than it found."""
    kind, desc, need, _ = _weight(fmt, out, K)
    w = _Weight(desc, out, K)
    R.QuantLinear(kind, w).reserve(most)
    have = w._ws.buf.numel() if w._ws.buf is not None else 0
    short = [M for M in range(1, most + 1) if need(M) > have]
    assert not short, (have, short[:5], [need(M) for M in short[:5]])


@pytest.mark.parametrize("fmt", ["NVQ", "NEPQ"])
def test_the_fp16_copy_of_codebook_formats_is_asked_for_apart(fmt):
    """Two bytes per weight are no part of what a weight's own workspace is sized by."""
    out, K = 17408, 5120
    _, _, need, copy = _weight(fmt, out, K)
    assert copy(255) == 0 and copy(1) == 0
    assert copy(2048) >= 2 * out * K
    assert max(need(M) for M in (256, 300, 512, 1024, 2048)) < out * K // 2


def test_a_device_too_full_for_the_copy_is_no_error(monkeypatch):
    def full(*args, **kw):
        raise torch.OutOfMemoryError("full")
    assert R.borrow(0, "cpu") is None and R.borrow(64, "cpu").numel() == 64
    monkeypatch.setattr(torch, "empty", full)
    assert R.borrow(64, "cpu") is None


@pytest.mark.parametrize("fmt,out,K,takes,not_yet", [
    ("NVQ", 12288, 4096, 256, 255), ("NVQ", 4096, 4096, 400, 300),       # from 1.5 million outputs and 256 rows on
    ("NVQ", 17408, 5120, 400, 384), ("NEPQ", 17408, 5120, 400, 384),     # 384 rows are one round of the codebook kernel's tiles
    ("NVQ", 5120, 17408, 400, 384), ("NVQ", 32000, 4096, 2048, 512),
])
def test_rows_from_which_the_copy_is_taken(fmt, out, K, takes, not_yet):
    _, _, _, copy = _weight(fmt, out, K)
    assert copy(takes) > 2 * out * K and copy(not_yet) == 0
