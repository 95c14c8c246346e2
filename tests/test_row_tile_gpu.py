"""The prefill tile kernel on row-major weights: MX payloads, NINT8-0 blocks, and formats dequantized to fp16 rows first."""
import numpy as np
import pytest
import torch

import synth
from oracle import mfq_oracle as O

pytestmark = pytest.mark.gpu


def _tensor(rng, fmt, out, K):
    if fmt in ("MXFP4", "MXFP8"):
        t = synth.mx_random(rng, fmt, out, K)
        return fmt, O.pack_mx(t), O.dequantize_mx(t)
    if fmt == "NINT8-0":
        w = (rng.standard_normal((out, K)) * 0.02).astype(np.float32)
        w[0, :32] = 0.0
        w[1] *= 1e3                               # scales of a row far above the others
        w[2, 32:] *= 1e-4                         # and of a block inside a row
        t = O.quantize_nint8_zero(w)
        dtype, blob = O.pack_tensor(t)
        return dtype, blob, O.dequantize_nint8_zero(t)
    dtype, blob = O.pack_tensor(synth.nvq_jsc_random(rng, out, K, "e8_256", 4))
    return dtype, blob, O.dequantize_tensor(O.unpack_tensor(dtype, blob))


@pytest.mark.parametrize("xd", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fmt", ["MXFP4", "MXFP8", "NINT8-0", "NVQ2J"])
@pytest.mark.parametrize("out,K,M,cus", [
    (200, 1568, 529, 0),     # row-blocks that end inside a wave, K inside a step, one 16-row block in the last tile; split over K
    (200, 1568, 600, 1),     # the same tensor in one pass over K (every tile shape: test_tile_shapes_gpu.py)
    (195, 2656, 577, 2),     # neurons that end inside a row-block, output rows off 16 bytes
    (16, 64, 520, 0),        # one row-block, K inside the first step
    (130, 512, 260, 3),      # whole steps, neurons of two 128-row bands
])
def test_tile_kernel_on_row_major_weights(fmt, out, K, M, cus, xd, cu_count):
    """Bound per element: fp32 sums over K <= 2656 terms, 1e-5 of the sum of the magnitudes, and one rounding to fp16's eleven
    bits per weight (2^-11) where a format has one: NINT8-0 and NVQ2J, not MX (its elements have at most four bits).  Weights
    2^-24 below their row's largest drop out of fp16 (half its smallest step, 2^-25 of a range of 2^12 and more)."""
    from tyloquant_amd import runtime as R
    cu_count(cus)
    if fmt == "MXFP8":
        K = (K + 127) // 128 * 128
    rng = np.random.default_rng(out + K + M + len(fmt))
    dtype, blob, deq = _tensor(rng, fmt, out, K)
    lin = R.load_quant_linear(dtype, blob)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
    x[1] *= 1e3 if xd is torch.float16 else 1e6
    x[2] *= 1e-2 if xd is torch.float16 else 1e-6
    x = x.to(xd)
    wide = torch.zeros((M, K + 5), dtype=xd)
    wide[:, 3:K + 3] = x
    ref = O.linear_forward_f64(deq, x.float().numpy())
    ax = np.abs(x.float().numpy())
    per_weight = (1e-5 + (0.0 if fmt.startswith("MX") else 2.0 ** -11)) * np.abs(deq) + 2.0 ** -36 * np.abs(deq).max(axis=1, keepdims=True)
    bound = ax @ per_weight.T + 1e-30
    for view in (x.cuda(), wide.cuda()[:, 3:K + 3]):        # rows at 16 bytes, and at neither 16 bytes nor an even stride
        y = lin(view).cpu().numpy()
        assert y.shape == ref.shape and np.all(np.abs(y - ref) <= bound), np.max(np.abs(y - ref) / bound)


@pytest.mark.parametrize("dtype", ["MXFP4", "MXFP8"])
def test_mx_tiles_keep_special_scales_and_payloads_off_16_bytes(dtype):
    """E8M0 0 and 255 on the tile kernel (255: that neuron NaN, no other), and a payload at an odd address, which goes by way of
    an fp16 copy, through the C entry point."""
    from tyloquant_amd import _lib as L
    from tyloquant_amd import runtime as R
    rng = np.random.default_rng(78)
    rows, cols, M = 256, 512, 300
    t = synth.mx_random(rng, dtype, rows, cols)
    t.scales[0, 0] = 255
    t.scales[-1, -1] = 0
    want = O.dequantize_mx(t)
    nan_rows = np.isnan(want).any(axis=1)
    lin = R.load_quant_linear(dtype, O.pack_mx(t))
    lib = L.lib()
    for xd, code in ((torch.bfloat16, L.X_BF16), (torch.float16, L.X_F16)):
        x = torch.from_numpy(rng.standard_normal((M, cols)).astype(np.float32)).to(xd).cuda()
        ref = O.linear_forward_f64(want[~nan_rows], x.float().cpu().numpy())
        ax = np.abs(x.float().cpu().numpy())
        bound = 1e-5 * (ax @ np.abs(want[~nan_rows]).T) + 1e-30
        odd = torch.zeros(t.values.nbytes + 1, dtype=torch.uint8, device="cuda")
        odd[1:] = torch.from_numpy(np.ascontiguousarray(t.values).view(np.uint8).reshape(-1).copy()).cuda()
        sc = torch.from_numpy(np.ascontiguousarray(t.scales).copy()).cuda()
        need = lib.mfq_hip_mx_gemm_rows_workspace_bytes(cols, rows, M)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        y = torch.empty((M, rows), dtype=torch.float32, device="cuda")
        rc = lib.mfq_hip_mx_gemm_rows(4 if dtype == "MXFP4" else 8, odd.data_ptr() + 1, sc.data_ptr(), rows, cols, 0, rows, x.data_ptr(),
                                      code, cols, M,
                                      y.data_ptr(), rows, ws.data_ptr(), need, None)
        assert rc == 0
        torch.cuda.synchronize()
        for got in (lin(x).cpu().numpy(), y.cpu().numpy()):
            assert np.isnan(got[:, nan_rows]).all()
            assert np.all(np.abs(got[:, ~nan_rows] - ref) <= bound)


@pytest.mark.parametrize("xd", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fmt,banks,out,K,M", [
    ("d4_512", 2, 2005, 1003, 750),      # neurons inside a row-block, K inside a group, a slice and a piece of eight columns
    ("d4_512", 4, 5900, 1000, 256),      # the fewest rows, four codebooks
    ("d4_512", 2, 5900, 1000, 255),      # one row less: the kernel that looks every weight up
    ("d4_256", 1, 1000, 400, 1501),      # 256 entries, built-in grid
    ("NEPQ1-S", 5, 2000, 1000, 750),
    ("NEPQ1-L", 40, 2000, 1000, 751),    # tables beyond the LDS
    ("NEPQ1-S", 1, 5904, 96, 255),
])
def test_codebook_formats_by_fp16_copy(fmt, banks, out, K, M, xd):
    """Bound per element as above: the NVQ weights are rounded once to fp16 (2^-11 of each), the NEPQ ones are whole numbers times
    the anchor.  NEPQ: the second of two experts, rows that start inside the tensor."""
    from tyloquant_amd import runtime as R
    from tyloquant_amd.runtime_vq import NepqWeight, nepq_matmul
    rng = np.random.default_rng(out + K + M + banks)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
    x[1] *= 1e3
    x = x.to(xd)
    nepq = fmt.startswith("NEPQ")
    if nepq:
        t = synth.nepq_random(rng, fmt, 2, out, K, banks)
        deq = O.dequantize_nepq(t)[1]
        y = nepq_matmul(NepqWeight.from_blob(O.pack_nepq(t)), x.cuda(), 1)
    else:
        t = synth.nvq_plain_random(rng, out, K) if fmt == "d4_256" else synth.nvq_jsc_random(rng, out, K, fmt, banks)
        dtype, blob = O.pack_tensor(t)
        deq = O.dequantize_tensor(O.unpack_tensor(dtype, blob))
        y = R.load_quant_linear(dtype, blob)(x.cuda())
    y, xf = y.cpu().numpy(), x.float().numpy()
    ref = O.linear_forward_f64(deq, xf)
    per_weight = (1e-5 + (0.0 if nepq else 2.0 ** -11)) * np.abs(deq) + 2.0 ** -36 * np.abs(deq).max(axis=1, keepdims=True)
    bound = np.abs(xf) @ per_weight.T + 1e-30
    assert y.shape == ref.shape and np.all(np.abs(y - ref) <= bound), np.max(np.abs(y - ref) / bound)


@pytest.mark.parametrize("fmt", ["NINT4", "NINT8-0", "d4_512"])
def test_prefill_of_rows_near_the_smallest_bf16_magnitudes(fmt):
    """Rows whose largest magnitude is 2^-120, 2^-127 (subnormal) and zero, next to ordinary ones, on the tile kernel's and the
    codebook kernel's activation prep: finite, and as accurate as fp32 results of that size can be.  Bound: as above, fp16's
    step below 2^-7 for a row scaled by 2^126 at most (half of 2^-24 of it), and eight steps of the subnormal result."""
    from tyloquant_amd import runtime as R
    rng = np.random.default_rng(92)
    out, K, M = 200, 512, 600
    if fmt == "NINT4":
        t = synth.nint_random(rng, out, K, 4, 32, 6)
    elif fmt == "NINT8-0":
        t = O.quantize_nint8_zero((rng.standard_normal((out, K)) * 0.02).astype(np.float32))
    else:
        t = synth.nvq_jsc_random(rng, out, K, fmt, 2)
    dtype, blob = O.pack_tensor(t)
    deq = O.dequantize_tensor(O.unpack_tensor(dtype, blob))
    x = rng.standard_normal((M, K))
    x[3] *= 2.0 ** -120 / np.abs(x[3]).max()
    x[4] *= 2.0 ** -127 / np.abs(x[4]).max()
    x[5] = 0.0
    x = torch.from_numpy(x.astype(np.float32)).to(torch.bfloat16)
    ref = O.linear_forward_f64(deq, x.float().numpy())
    y = R.load_quant_linear(dtype, blob)(x.cuda()).cpu().numpy()
    bound = np.abs(x.float().numpy()) @ ((2e-5 + 2.0 ** -11) * np.abs(deq)).T + 2.0 ** -151 * np.abs(deq).sum(axis=1) + 2.0 ** -146
    assert np.isfinite(y).all() and np.all(y[5] == 0.0)
    assert np.all(np.abs(y - ref)[3:5] <= bound[3:5]), np.max(np.abs(y - ref) / bound)


def test_small_block_scales_of_a_q8_row_keep_their_bits():
    """NINT8-0 blocks whose scale lies 2^-24 and 2^-28 below the row's largest still round once, to fp16's eleven bits: each
    activation row meets one weight, so the result is that weight times the activation within 2^-11, or within half of fp16's
    smallest step (2^-25 of the row's power of two, 4 for a largest scale of 1000) where the product is subnormal."""
    from tyloquant_amd import runtime as R
    rng = np.random.default_rng(94)
    out, K, M = 160, 256, 300
    t = O.quantize_nint8_zero(rng.standard_normal((out, K)).astype(np.float32))
    t.scale[:, 0] = np.float16(1000.0)
    t.scale[:, 1:4] = rng.uniform(6.2e-5, 1.2e-4, (out, 3)).astype(np.float16)     # 2^-14: 2^-24 of the largest
    t.scale[:, 4:] = np.float16(2.0 ** -18)                                        # a power of two, 2^-28 of the largest
    t.q[:, :, :] = rng.choice(np.array([-128, -127, -61, 3, 77, 127], dtype=np.int8), t.q.shape)
    x = np.zeros((M, K), dtype=np.float32)
    cols = 32 + rng.integers(0, K - 32, M)
    x[np.arange(M), cols] = 1.5
    deq = O.dequantize_nint8_zero(t)
    y = R.load_quant_linear(*O.pack_tensor(t))(torch.from_numpy(x).to(torch.bfloat16).cuda()).cpu().numpy()
    want = 1.5 * deq[:, cols].T.astype(np.float64)
    assert np.all(np.abs(y - want) <= (2.0 ** -11 + 2.0 ** -23) * np.abs(want) + 1.5 * 2.0 ** -23), np.max(np.abs(y / want - 1))


@pytest.mark.parametrize("out,K,M", [(4105, 64, 33), (9000, 128, 48), (40, 1024, 600), (4105, 6176, 33), (2100, 6176, 170), (16384, 32, 129), (16390, 32, 129), (16390, 32, 128)])
def test_neurons_of_every_range_get_their_power_of_two(out, K, M):
    """NINT8-0: the power of two of a neuron is found in the launch that lays the activations out, by blocks behind and between theirs:
    more neurons than waves of a launch, one and several blocks a row-block of activations, activations with a scale launch of their
    own, and on 256 compute units both sides of where the neurons get one.
    Neurons' scales lie between 2^-20 and 2^10, one scale is NaN.  Bound as in test_tile_kernel_on_row_major_weights: 1e-5 of the
    sum of the magnitudes, a rounding to 11 bits a weight, 2^-36 of the neuron's largest where fp16 is subnormal."""
    from tyloquant_amd import runtime as R
    rng = np.random.default_rng(out + K + M)
    q = rng.integers(-127, 128, (out, K // 32, 32), dtype=np.int8)
    scale = (rng.uniform(0.5, 1.0, (out, K // 32)) * 2.0 ** rng.integers(-19, 11, (out, 1))).astype(np.float16)
    t = O.quantize_nint8_zero(np.zeros((out, K), dtype=np.float32))
    t.q[...], t.scale[...] = q.reshape(t.q.shape), scale.reshape(t.scale.shape)
    t.scale.reshape(out, -1)[7, 0] = np.float16("nan")
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16)
    y = R.load_quant_linear(*O.pack_tensor(t))(x.cuda()).cpu().numpy()
    deq = O.dequantize_nint8_zero(t)
    ok = np.arange(out) != 7
    ref, deq = O.linear_forward_f64(deq[ok], x.float().numpy()), np.abs(deq[ok])
    bound = np.abs(x.float().numpy()) @ ((1e-5 + 2.0 ** -11) * deq + 2.0 ** -36 * deq.max(axis=1, keepdims=True)).T + 1e-30
    assert np.all(np.abs(y[:, ok] - ref) <= bound), np.max(np.abs(y[:, ok] - ref) / bound)
    assert np.isnan(y[:, 7]).all()


@pytest.mark.parametrize("fmt,out,K,M", [("MXFP4", 4096, 4096, 100), ("MXFP8", 4096, 1024, 160), ("NINT4", 8192, 4096, 64),
                                         ("NINT8", 4096, 1056, 160)])
def test_streaming_batches_need_no_workspace(fmt, out, K, M):
    """Batches the streaming kernels can serve run without the workspace that the faster tile kernel would use (asked for by the
    query), and give what a call with it gives up to the bounds above."""
    from tyloquant_amd import _lib as L
    from tyloquant_amd import runtime as R
    import ctypes as C
    rng = np.random.default_rng(95)
    if fmt.startswith("MX"):
        dtype, blob, deq = _tensor(rng, fmt, out, K)
    else:
        t = synth.nint_random(rng, out, K, *((4, 32, 6) if fmt == "NINT4" else (8, 48, 7)))
        dtype, blob = O.pack_tensor(t)
        deq = O.dequantize_nint(t)
    lin = R.load_quant_linear(dtype, blob)
    lib, w = L.lib(), lin.weight
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    y = torch.empty((M, out), dtype=torch.float32, device="cuda")
    if fmt.startswith("MX"):
        assert lib.mfq_hip_mx_gemm_rows_workspace_bytes(K, out, M) > 0
        rc = lib.mfq_hip_mx_gemm_rows(w.kind, w.values.data_ptr(), w.scales.data_ptr(), out, K, 0, out, x.data_ptr(), L.X_BF16, K, M,
                                      y.data_ptr(), out, None, 0, None)
    else:
        assert lib.mfq_hip_nint_gemm_workspace_bytes(C.byref(w.desc), M) > 0
        rc = lib.mfq_hip_nint_gemm(C.byref(w.desc), w.data.data_ptr(), x.data_ptr(), L.X_BF16, K, M, y.data_ptr(), out, None, 0, None)
    assert rc == L.OK
    torch.cuda.synchronize()
    xf = x.float().cpu().numpy()
    ref = O.linear_forward_f64(deq, xf)
    limit = 1e-5 if fmt != "NINT8" else 3e-4
    for got in (y.cpu().numpy(), lin(x).cpu().numpy()):
        assert np.linalg.norm(got - ref) <= limit * np.linalg.norm(ref)


def _gemm(lin, x, ws_bytes):
    """The C entry of a linear with a workspace of that many bytes: (status, y)."""
    from tyloquant_amd import _lib as L
    import ctypes as C
    lib, w, (M, K) = L.lib(), lin.weight, x.shape
    ws = torch.full((max(ws_bytes, 1),), 0xA5, dtype=torch.uint8, device="cuda")
    y = torch.empty((M, w.out), dtype=torch.float32, device="cuda")
    tail = (x.data_ptr(), L.X_BF16, K, M, y.data_ptr(), w.out, ws.data_ptr(), ws_bytes, None)
    if lin.kind == "mx":
        rc = lib.mfq_hip_mx_gemm_rows(w.kind, w.values.data_ptr(), w.scales.data_ptr(), w.out, K, 0, w.out, *tail)
    else:
        name = {"nint": "nint", "nint8z": "nint8z", "nvq": "nvqs" if type(w).__name__ == "NvqsWeight" else "nvq"}[lin.kind]
        rc = getattr(lib, f"mfq_hip_{name}_gemm")(C.byref(w.desc), w.data.data_ptr(), *tail)
    torch.cuda.synchronize()
    return rc, y.cpu().numpy()


def _workspace(lin, M):
    from tyloquant_amd import _lib as L
    import ctypes as C
    lib, w = L.lib(), lin.weight
    if lin.kind == "mx":
        return lib.mfq_hip_mx_gemm_rows_workspace_bytes(w.neuron_len, w.out, M)
    name = {"nint": "nint", "nint8z": "nint8z", "nvq": "nvqs" if type(w).__name__ == "NvqsWeight" else "nvq"}[lin.kind]
    return getattr(lib, f"mfq_hip_{name}_gemm_workspace_bytes")(C.byref(w.desc), M)


@pytest.mark.parametrize("fmt", ["NINT4", "NINT8-0", "MXFP4", "NVQ2J"])
def test_a_workspace_without_room_for_the_split_is_enough(fmt, cu_count):
    """A split over K belongs to small batches, so a workspace sized for the largest batch can be smaller than the query of a
    smaller one: the call then splits into the pieces that fit.  Sizes: all pieces, two of them, none; one byte less than that
    is refused.  The results differ by the order of 32-bit sums."""
    from tyloquant_amd import _lib as L
    from tyloquant_amd import runtime as R
    rng = np.random.default_rng(96)
    out, K, M = 256, 4096, 300
    dtype, blob, deq = (None, None, None) if fmt == "NINT4" else _tensor(rng, fmt, out, K)
    if fmt == "NINT4":
        t = synth.nint_random(rng, out, K, 4, 32, 6)
        dtype, blob = O.pack_tensor(t)
        deq = O.dequantize_nint(t)
    lin = R.load_quant_linear(dtype, blob)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    ref = O.linear_forward_f64(deq, x.float().cpu().numpy())
    all_pieces = _workspace(lin, M)
    cu_count(1)
    least = _workspace(lin, M)
    cu_count(0)
    assert all_pieces >= least + 3 * M * out * 4
    for nbytes in (all_pieces, least + 2 * M * out * 4, least):
        rc, y = _gemm(lin, x, nbytes)
        assert rc == L.OK
        assert np.linalg.norm(y - ref) <= (1e-5 if fmt in ("NINT4", "MXFP4") else 4e-4) * np.linalg.norm(ref)
    if fmt == "MXFP4":       # its query also covers MXFP8, which keeps more
        least = 0
    assert _gemm(lin, x, max(least - 1, 0))[0] == L.ERR_WORKSPACE


def test_fp16_copies_are_borrowed_per_call():
    """Prefill of NVQ3J-512 by way of the fp16 copy: nothing stays with the weight, two weights take turns in the same scratch,
    with less memory the call takes the codebook kernel, and a captured pair of calls replays with eager work in between."""
    from tyloquant_amd import runtime as R
    rng = np.random.default_rng(97)
    out, K, M = 2000, 1000, 800
    lins = [R.load_quant_linear(*O.pack_tensor(synth.nvq_jsc_random(rng, out, K, "d4_512", 2))) for _ in range(2)]
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16).cuda()
    refs = [x.double() @ lin.dequantize().double().t() for lin in lins]
    close = lambda y, ref: float((y.double() - ref).norm() / ref.norm()) < 4e-4      # one rounding of the weight to 11 bits
    eager = [lin(x) for lin in lins]
    assert all(close(y, ref) for y, ref in zip(eager, refs))
    assert all(lin.weight._ws.buf is None for lin in lins)
    small = _workspace(lins[0], M)
    assert small < 2 * out * K + 2 * M * K
    rc, y = _gemm(lins[0], x, small)
    assert rc == 0 and close(torch.from_numpy(y).cuda(), refs[0])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for lin in lins:
            lin(x)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ys = [lin(x) for lin in lins]
    for rep in range(3):
        for y in ys:
            y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(y, e) for y, e in zip(ys, eager)), rep
        lins[1](x[:300])
        torch.cuda.synchronize()


@pytest.mark.parametrize("xd", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fmt,K,M", [("NINT4", 6160, 600), ("NINT4", 6144, 600), ("NINT4", 17416, 600), ("NINT5", 12308, 600),
                                     ("NINT8-0", 6176, 64), ("NINT8-0", 6144, 64), ("NINT8-0", 17408, 33), ("NINT8-0", 12320, 672),
                                     ("NINT8-0", 12320, 673)])
def test_activations_of_long_rows(fmt, K, M, xd):
    """Rows of more than 6144 values in batches of up to 672 get their scale from a launch of its own (sizes on both sides of
    either limit, pieces that end inside a round), with infinities, NaN, zero rows and rows off 16 bytes.  Bound: fp32 sums
    over K <= 17416 terms, 1e-5 of the sum of the magnitudes, and one rounding to 11 bits of a weight (its scale part)."""
    from tyloquant_amd import runtime as R
    rng = np.random.default_rng(K + M)
    out = 48
    if fmt == "NINT8-0":
        t = O.quantize_nint8_zero((rng.standard_normal((out, K)) * 0.02).astype(np.float32))
        deq = O.dequantize_nint8_zero(t)
        per_weight = (1e-5 + 2.0 ** -11) * np.abs(deq)
    else:
        t = synth.nint_random(rng, out, K, *((4, 24, 6) if fmt == "NINT4" else (5, 28, 7)))
        deq = O.dequantize_nint(t)
        scale_part = (t.neuron_scale[:, None, None] * t.sub_scale[:, :, None] * t.q).reshape(out, -1)[:, :K]
        per_weight = (1e-5 + (2.0 ** -11 if fmt == "NINT5" else 0.0)) * scale_part + 1e-5 * np.abs(deq - scale_part)
    lin = R.load_quant_linear(*O.pack_tensor(t))
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
    x[1] *= 1e3 if xd is torch.float16 else 1e6
    x[2] = 0.0
    x[3, K - 1] = 300.0                          # the largest value is the row's last
    x[4, 5] = float("inf")
    x[5, K - 2] = float("nan")
    x = x.to(xd)
    wide = torch.zeros((M, K + 3), dtype=xd)
    wide[:, 1:K + 1] = x
    ok = np.ones(M, dtype=bool)
    ok[4:6] = False
    xf = x.float().numpy()[ok]
    ref = O.linear_forward_f64(deq, xf)
    bound = np.abs(xf) @ per_weight.T + 1e-30
    for view in (x.cuda(), wide.cuda()[:, 1:K + 1]):
        y = lin(view).cpu().numpy()
        assert np.all(np.abs(y[ok] - ref) <= bound), np.max(np.abs(y[ok] - ref) / bound)
        assert not np.isfinite(y[4:6]).any()
