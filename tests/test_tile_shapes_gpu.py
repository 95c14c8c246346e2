"""Every tile shape of the prefill tile kernel (of the widest with NINT weights, see test_tile_epilogue_gpu.py), with and without a split over K, on every kind of weights: six steps of K and
more (the ring turns several times), and remainders in rows, neurons and columns.  The shape is the library's own choice for
the sizes and compute-unit count searched out here, and is asserted through its host query."""
import ctypes as C

import numpy as np
import pytest
import torch

import synth
from oracle import mfq_oracle as O

pytestmark = pytest.mark.gpu

OUT, ROWS, CUS = (200, 392, 520, 776, 1064), (529, 545, 577, 641, 705, 769, 833, 961), tuple(range(1, 17)) + (20, 24, 32, 48, 64)
NINT = [(4, 32, 6), (4, 24, 6), (4, 16, 6), (4, 48, 6), (3, 24, 5), (2, 16, 5), (2, 32, 5), (5, 28, 7), (6, 24, 7), (8, 48, 7)]
KINDS = [("NVQ2J", "bf16", 0), ("NINT8-0", "bf16", 1), ("MXFP4", "bf16", 2), ("MXFP4", "fp16", 3), ("MXFP8", "bf16", 4), ("MXFP8", "fp16", 5)]


def _search(query, outs, shape, split):
    """(out, M, compute units) for which query(out, M) = (shape, split or not); leaves the override set."""
    from tyloquant_amd import _lib as L
    for out in outs:
        for M in ROWS:
            for cu in CUS:
                L.lib().mfq_hip_set_cu_count(cu)
                got, pieces = query(out, M)
                if got == shape and (pieces > 1) == split:
                    return out, M
    pytest.fail(f"no size here takes tile shape {shape} {'with' if split else 'without'} a split over K any more")


def _wide(bits, gs):     # three row-blocks per wave need units of at most five dwords
    return gs * bits <= 160


@pytest.mark.parametrize("bits,gs,sb,shape,form", [
    (b, g, s, shape, form) for b, g, s in NINT for shape in range(5) for form in ("plain", "split", "glu")
    if shape not in (1, 3) or _wide(b, g)])
def test_nint_tile_shapes(bits, gs, sb, shape, form, cu_count):
    """Bounds as for the edges of the tiles: fp32 sums over K <= 3880 terms, 1e-5 of the sum of the magnitudes, one rounding to
    11 bits per weight of sub_scale * code from five bits on (eight bits: of sub_scale * (code - 128)).  The GLU's 16-bit result:
    2^-11 of its own and the two factors' errors."""
    from tyloquant_amd import _lib as L
    from tyloquant_amd import runtime as R
    lib, K = L.lib(), 16 * gs * 5 + 40
    desc, pieces = L.NintDesc(), C.c_int()

    def query(out, M):
        L.check(lib.mfq_hip_nint_plan(bits, sb, gs, out, K, C.byref(desc)))
        return lib.mfq_hip_nint_tile_plan(C.byref(desc), M, int(form == "glu"), C.byref(pieces)), pieces.value
    out, M = _search(query, [o if form != "glu" else (o + 31) // 32 * 32 for o in OUT], shape, form == "split")
    rng = np.random.default_rng(bits * 100 + gs + shape)
    t = synth.nint_random(rng, out, K, bits, gs, sb)
    lin = R.load_quant_linear(*O.pack_tensor(t))
    deq = O.dequantize_nint(t)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
    x = (x / float(deq.std() * K ** 0.5)).to(torch.bfloat16)
    xf = x.float().numpy()
    ref = O.linear_forward_f64(deq, xf)
    if form == "glu":
        need = lib.mfq_hip_nint_gemm_workspace_bytes(C.byref(desc), M)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        xd, hidden = x.cuda(), torch.empty((M, out // 2), dtype=torch.float16, device="cuda")
        L.check(lib.mfq_hip_nint_gemm_glu(C.byref(desc), lin.weight.data.data_ptr(), xd.data_ptr(), L.X_BF16, K, M, L.GLU_SILU,
                                          hidden.data_ptr(), L.X_F16, out // 2, ws.data_ptr(), need, None))
        torch.cuda.synchronize()
        g, u = ref[:, :out // 2], ref[:, out // 2:]
        want = g / (1 + np.exp(-g)) * u
        err = np.linalg.norm(hidden.float().cpu().numpy() - want) / np.linalg.norm(want)
        assert err < (5e-4 if bits < 5 else 1.5e-3), err
        return
    y = lin(x.cuda()).cpu().numpy()
    codes = np.abs(t.q.astype(np.float64) - 128) if bits == 8 else t.q
    scale_part = (t.neuron_scale[:, None, None] * t.sub_scale[:, :, None] * t.q).reshape(out, -1)[:, :K]
    rounded = (t.neuron_scale[:, None, None] * t.sub_scale[:, :, None] * codes).reshape(out, -1)[:, :K]
    per_weight = 1e-5 * (scale_part + np.abs(deq - scale_part)) + (2.0 ** -11 if bits >= 5 else 0.0) * rounded
    assert np.all(np.abs(y - ref) <= np.abs(xf) @ per_weight.T + 1e-30)


# row-blocks a wave: two of NINT8-0, four (shape 5) of fp16 fragments only
@pytest.mark.parametrize("fmt,xd,kind,shape,split", [
    (*k, shape, split) for k in KINDS for shape in range(6) for split in (False, True)
    if (k[2] != 1 or shape not in (1, 3)) and (shape != 5 or k[2] == 0)])
def test_row_tile_shapes(fmt, xd, kind, shape, split, cu_count):
    """Bounds: fp32 sums over K <= 2688 terms, and one rounding to 11 bits per weight for NINT8-0 and NVQ2J."""
    from tyloquant_amd import _lib as L
    from tyloquant_amd import runtime as R
    lib, K, pieces = L.lib(), 2592 if fmt != "MXFP8" else 2688, C.c_int()
    out, M = _search(lambda out, M: (lib.mfq_hip_row_tile_plan(kind, out, K, M, C.byref(pieces)), pieces.value), OUT, shape, split)
    rng = np.random.default_rng(kind * 100 + shape)
    if fmt.startswith("MX"):
        t = synth.mx_random(rng, fmt, out, K)
        dtype, blob, deq = fmt, O.pack_mx(t), O.dequantize_mx(t)
    else:
        t = (O.quantize_nint8_zero((rng.standard_normal((out, K)) * 0.02).astype(np.float32)) if fmt == "NINT8-0"
             else synth.nvq_jsc_random(rng, out, K, "e8_256", 4))
        dtype, blob = O.pack_tensor(t)
        deq = O.dequantize_tensor(O.unpack_tensor(dtype, blob))
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16 if xd == "bf16" else torch.float16)
    ref = O.linear_forward_f64(deq, x.float().numpy())
    y = R.load_quant_linear(dtype, blob)(x.cuda()).cpu().numpy()
    per_weight = (1e-5 + (0.0 if fmt.startswith("MX") else 2.0 ** -11)) * np.abs(deq) + 2.0 ** -36 * np.abs(deq).max(axis=1, keepdims=True)
    assert np.all(np.abs(y - ref) <= np.abs(x.float().numpy()) @ per_weight.T + 1e-30)
