"""The widest tile shape of the prefill kernel, and results that leave it in rows off 16 bytes or with columns that end inside a piece."""
import ctypes as C

import numpy as np
import pytest
import torch

import synth
from oracle import mfq_oracle as O
from test_tile_shapes_gpu import OUT, _search

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,gs,sb", [(4, 32, 6), (4, 24, 6), (4, 16, 6), (2, 16, 5), (2, 32, 5)])
@pytest.mark.parametrize("form", ["plain", "split", "glu"])
def test_four_row_blocks_a_wave(bits, gs, sb, form, cu_count):
    """Bounds as in test_tile_shapes_gpu.py: fp32 sums over K <= 2600 terms, 1e-5 of the sum of the magnitudes; the GLU's result adds
    its own rounding to 11 bits."""
    from tyloquant_amd import _lib as L
    from tyloquant_amd import runtime as R
    lib, K = L.lib(), 16 * gs * 5 + 40
    desc, pieces = L.NintDesc(), C.c_int()

    def query(out, M):
        L.check(lib.mfq_hip_nint_plan(bits, sb, gs, out, K, C.byref(desc)))
        return lib.mfq_hip_nint_tile_plan(C.byref(desc), M, int(form == "glu"), C.byref(pieces)), pieces.value
    out, M = _search(query, [o if form != "glu" else (o + 31) // 32 * 32 for o in OUT], 5, form == "split")
    rng = np.random.default_rng(bits * 100 + gs)
    t = synth.nint_random(rng, out, K, bits, gs, sb)
    lin = R.load_quant_linear(*O.pack_tensor(t))
    deq = O.dequantize_nint(t)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
    x = (x / float(deq.std() * K ** 0.5)).to(torch.bfloat16)
    ref = O.linear_forward_f64(deq, x.float().numpy())
    if form != "glu":
        y = lin(x.cuda()).cpu().numpy()
        part = (t.neuron_scale[:, None, None] * t.sub_scale[:, :, None] * t.q).reshape(out, -1)[:, :K]
        assert np.all(np.abs(y - ref) <= np.abs(x.float().numpy()) @ (1e-5 * (part + np.abs(deq - part))).T + 1e-30)
        return
    _check_glu(lin, desc, x, ref, out // 2)


def _check_glu(lin, desc, x, ref, ldh):
    """act(gate) * up through the C entry point into rows of ldh halves; what lies behind a row's columns stays."""
    from tyloquant_amd import _lib as L
    lib, (M, K), half = L.lib(), x.shape, ref.shape[1] // 2
    need = lib.mfq_hip_nint_gemm_workspace_bytes(C.byref(desc), M)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    xd, hidden = x.cuda(), torch.full((M, ldh), 7.0, dtype=torch.float16, device="cuda")
    L.check(lib.mfq_hip_nint_gemm_glu(C.byref(desc), lin.weight.data.data_ptr(), xd.data_ptr(), L.X_BF16, K, M, L.GLU_SILU,
                                      hidden.data_ptr(), L.X_F16, ldh, ws.data_ptr(), need, None))
    got = hidden.float().cpu().numpy()
    g, u = ref[:, :half], ref[:, half:]
    want = g / (1 + np.exp(-g)) * u
    assert np.linalg.norm(got[:, :half] - want) < 5e-4 * np.linalg.norm(want)
    assert np.all(got[:, half:] == 7.0)


@pytest.mark.parametrize("extra", [0, 1, 4])
def test_gated_rows_off_16_bytes(extra, cu_count):
    """Rows of hidden values 0, 2 and 8 bytes off a multiple of 16; 80 columns, so the last wave's pieces end inside the tile."""
    from tyloquant_amd import _lib as L
    from tyloquant_amd import runtime as R
    cu_count(4)
    rng = np.random.default_rng(11)
    out, K, M, desc = 160, 552, 777, L.NintDesc()
    t = synth.nint_random(rng, out, K, 4, 32, 6)
    L.check(L.lib().mfq_hip_nint_plan(4, 6, 32, out, K, C.byref(desc)))
    lin = R.load_quant_linear(*O.pack_tensor(t))
    deq = O.dequantize_nint(t)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
    x = (x / float(deq.std() * K ** 0.5)).to(torch.bfloat16)
    _check_glu(lin, desc, x, O.linear_forward_f64(deq, x.float().numpy()), out // 2 + extra)


@pytest.mark.parametrize("rows", [5, 6, 11, 12, 17, 22, 30])
@pytest.mark.parametrize("out,K", [(48, 1000), (4 * 16 * 3 - 7, 7000)])
@pytest.mark.parametrize("fmt", ["NVQ3J-512", "NEPQ1-S", "NVQ2J"])
def test_activations_turned_in_lds(fmt, out, K, rows, cu_count):
    """Batches on either side of the rows from which small-batch kernels sort the activations in LDS, with K inside a step and with
    several steps a wave, rows at 16 bytes and not.  Bound: fp32 sums of K <= 7000 terms, and the activations' own bf16 is exact."""
    from tyloquant_amd import runtime as R
    from tyloquant_amd.runtime_vq import NepqWeight, nepq_matmul
    cu_count(4)
    rng = np.random.default_rng(out + K + rows)
    x = torch.from_numpy(rng.standard_normal((rows, K)).astype(np.float32)).to(torch.bfloat16)
    wide = torch.zeros((rows, K + 3), dtype=torch.bfloat16)
    wide[:, :K] = x
    if fmt == "NEPQ1-S":
        out16 = (out + 15) // 16 * 16
        t = synth.nepq_random(rng, fmt, 1, out16, K, 3)
        deq, w = O.dequantize_nepq(t)[0], NepqWeight.from_blob(O.pack_nepq(t))
        run = lambda v: nepq_matmul(w, v, 0)
    else:
        t = synth.nvq_jsc_random(rng, out, K, "d4_512" if fmt == "NVQ3J-512" else "e8_256", 2 if fmt == "NVQ3J-512" else 4)
        dtype, blob = O.pack_tensor(t)
        deq = O.dequantize_tensor(O.unpack_tensor(dtype, blob))
        lin = R.load_quant_linear(dtype, blob)
        run = lambda v: lin(v)
    ref = O.linear_forward_f64(deq, x.float().numpy())
    # NVQ3J-512: magnitude * scale is rounded to fp16, 2^-11 of each weight.  NEPQ1-S: a weight is state * (digit + bias - 1) with the
    # digit (0 .. 2) and the rest (up to 37 / 32) summed apart, and at least 5 / 32 state: parts of up to (1 + 2 * 37 / 5) weights.
    per_weight = {"NVQ3J-512": 1e-5 + 2.0 ** -11, "NEPQ1-S": 1e-5 * (1 + 2 * 37 / 5), "NVQ2J": 1e-5}[fmt]
    bound = per_weight * (np.abs(x.float().numpy()) @ np.abs(deq).T) + 1e-30
    for v in (x.cuda(), wide.cuda()[:, :K]):
        y = run(v).float().cpu().numpy().reshape(ref.shape)
        assert np.all(np.abs(y - ref) <= bound), np.max(np.abs(y - ref) / bound)


@pytest.mark.parametrize("rows", [17, 21, 22, 64, 65, 85, 86, 128])
@pytest.mark.parametrize("out,K", [(48, 1000), (16 * 5 - 7, 6000)])
def test_last_rows_of_a_batch_turned_or_not(out, K, rows, cu_count):
    """NVQ2J: full tiles of 32 or 64 rows, whose activations are turned in LDS, and last ones on either side of the rows from which they
    are.  Bound: fp32 sums of K <= 6000 terms."""
    from tyloquant_amd import runtime as R
    cu_count(16)
    rng = np.random.default_rng(out + K + rows)
    x = torch.from_numpy(rng.standard_normal((rows, K)).astype(np.float32)).to(torch.bfloat16)
    dtype, blob = O.pack_tensor(synth.nvq_jsc_random(rng, out, K, "e8_256", 4))
    deq = O.dequantize_tensor(O.unpack_tensor(dtype, blob))
    lin = R.load_quant_linear(dtype, blob)
    ref = O.linear_forward_f64(deq, x.float().numpy())
    bound = 1e-5 * (np.abs(x.float().numpy()) @ np.abs(deq).T) + 1e-30
    for dt in (torch.bfloat16, torch.float16):
        y = lin(x.to(dt).cuda()).cpu().numpy()
        r = ref if dt is torch.bfloat16 else O.linear_forward_f64(deq, x.to(dt).float().numpy())
        assert np.all(np.abs(y - r) <= bound), np.max(np.abs(y - r) / bound)


@pytest.mark.parametrize("rows", [7, 8, 9, 10, 13, 14, 22, 23, 24, 26, 27, 30])
@pytest.mark.parametrize("out", [48, 112, 169])
@pytest.mark.parametrize("K", [3000, 7000])
def test_tiles_of_the_signed_kernel_turned_or_not(K, out, rows, cu_count):
    """NVQ3J-512 with one, two and three row-blocks a block and one and several steps a wave: rows on either side of those from which a
    tile's activations are turned in LDS, in the first tile and in the second.  Bound: fp32 sums of K <= 7000 terms, and magnitude *
    scale rounded to fp16, 2^-11 of each weight."""
    from tyloquant_amd import runtime as R
    cu_count(4)
    rng = np.random.default_rng(out + K + rows)
    x = torch.from_numpy(rng.standard_normal((rows, K)).astype(np.float32)).to(torch.bfloat16)
    dtype, blob = O.pack_tensor(synth.nvq_jsc_random(rng, out, K, "d4_512", 2))
    deq = O.dequantize_tensor(O.unpack_tensor(dtype, blob))
    ref = O.linear_forward_f64(deq, x.float().numpy())
    bound = (1e-5 + 2.0 ** -11) * (np.abs(x.float().numpy()) @ np.abs(deq).T) + 1e-30
    y = R.load_quant_linear(dtype, blob)(x.cuda()).cpu().numpy()
    assert np.all(np.abs(y - ref) <= bound), np.max(np.abs(y - ref) / bound)
