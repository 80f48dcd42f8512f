"""GPU parity: the HIP path (through the C ABI) against the CPU oracle.

Bars: dequant and quantize bit-exact; qmm bf16 outputs within relative
Frobenius 1e-3 and max-abs 4 bf16 ulp of each row's max |y| (oracle rounds its
double sum once to bf16); f32 outputs within the same bound.
"""
import ctypes
import functools
import re
from math import ceil

import numpy as np
import pytest
import torch

import oracle as O
import gemm_shapes as G
import qmm as Q

pytestmark = pytest.mark.gpu

TOL = dict(rel_fro=1e-3, ulps=4.0)


def bf16(a):
    return O.f32_to_bf16_bits(np.asarray(a, np.float32))


def f32(bits):
    return O.bf16_bits_to_f32(bits)


def rand_w(rng, mode, N, K, scale=0.02):
    W = f32(bf16(rng.standard_normal((N, K)) * scale))
    return O.quantize(mode, W)


def run_qmm(mode, xb, wq, s, *, x_f32=False, **kw):
    x = Q.Array.from_numpy(xb, Q.FLOAT32 if x_f32 else Q.BFLOAT16)
    w = Q.Array.from_numpy(wq, Q.UINT32)
    sc = Q.Array.from_numpy(s, Q.UINT8)
    y = Q.quantized_matmul(x, w, sc, mode, **kw)
    return y.numpy()


def test_device_is_gfx950():
    import ctypes

    buf = ctypes.create_string_buffer(512)
    Q.check(Q.lib.qmm_device_info(buf, 512), "device_info")
    info = buf.value.decode()
    print(info)
    assert "gfx950" in info


@pytest.mark.parametrize("out_dtype", [Q.FLOAT32, Q.BFLOAT16])
def test_dequant_mxfp8_exhaustive_bit_exact(out_dtype):
    K = 256
    codes = np.arange(256, dtype=np.uint8)
    w = np.tile(codes.view(np.uint32), (256, 1))
    s = np.repeat(np.arange(256, dtype=np.uint8)[:, None], K // 32, axis=1)
    d = Q.dequantize(Q.Array.from_numpy(w, Q.UINT32), Q.Array.from_numpy(s, Q.UINT8), "mxfp8", dtype=out_dtype).numpy()
    if out_dtype == Q.FLOAT32:
        ref = O.dequant("mxfp8", w, s, K)
        assert np.array_equal(np.isnan(d), np.isnan(ref))
        assert np.array_equal(np.nan_to_num(d).view(np.uint32), np.nan_to_num(ref).view(np.uint32))
    else:
        ref = O.dequant_bf16("mxfp8", w, s, K)
        nan = (ref & 0x7FFF) > 0x7F80
        assert np.array_equal((d & 0x7FFF) > 0x7F80, nan)
        assert np.array_equal(d[~nan], ref[~nan])


@pytest.mark.parametrize("out_dtype", [Q.FLOAT32, Q.BFLOAT16])
def test_dequant_nvfp4_exhaustive_bit_exact(out_dtype):
    K = 256
    row = np.array([0x76543210, 0xFEDCBA98] * (K // 16), np.uint32)
    w = np.tile(row, (256, 1))
    s = np.repeat(np.arange(256, dtype=np.uint8)[:, None], K // 16, axis=1)
    d = Q.dequantize(Q.Array.from_numpy(w, Q.UINT32), Q.Array.from_numpy(s, Q.UINT8), "nvfp4", dtype=out_dtype).numpy()
    if out_dtype == Q.FLOAT32:
        ref = O.dequant("nvfp4", w, s, K)
        assert np.array_equal(np.isnan(d), np.isnan(ref))
        assert np.array_equal(np.nan_to_num(d).view(np.uint32), np.nan_to_num(ref).view(np.uint32))
    else:
        ref = O.dequant_bf16("nvfp4", w, s, K)
        nan = (ref & 0x7FFF) > 0x7F80
        assert np.array_equal((d & 0x7FFF) > 0x7F80, nan)
        assert np.array_equal(d[~nan], ref[~nan])


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
@pytest.mark.parametrize("src", ["bf16", "f32"])
def test_quantize_bit_exact(mode, src):
    rng = np.random.default_rng(21)
    N, K = 96, 512
    W = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    W[0, :64] = 0.0
    W[1, 3] = 3e3
    W[2, 32:48] = [6, .25, .75, 1.25, 1.75, 2.5, 3.5, 5, -.25, -.75, -2.5, -5, 0, 1, 2, 3]
    W[3] *= 1e-30  # tiny groups
    if src == "bf16":
        W = f32(bf16(W))
        wa = Q.Array.from_numpy(bf16(W), Q.BFLOAT16)
    else:
        wa = Q.Array.from_numpy(W, Q.FLOAT32)
    wq, s = Q.quantize(wa, mode)
    rq, rs = O.quantize(mode, W)
    assert np.array_equal(s.numpy(), rs)
    assert np.array_equal(wq.numpy(), rq)


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
@pytest.mark.parametrize("src", ["bf16", "f32"])
@pytest.mark.parametrize("N,K", [(1, 32), (3, 96), (33, 992), (65, 4128)])
def test_convert_ragged_bit_exact(mode, src, N, K):
    """Chunks of 8 elements: sizes that end inside a block's last pass, every magnitude of
    group (largest scales, subnormal scales, zeros of both signs), values on the midpoints of
    their scale; and back, on a buffer of 2-byte alignment."""
    rng = np.random.default_rng(N + K)
    W = rng.standard_normal((N, K)).astype(np.float32)
    W *= np.exp2(rng.integers(-40, 40, (N, K // 16))).astype(np.float32).repeat(16, 1)
    mids = np.array([.25, .75, 1.25, 1.75, 2.5, 3.5, 5, 6, -.25, -.75, -2.5, -5, 0, -0., 1e-3, -1e-3], np.float32)
    for r in range(0, N, 2):
        W[r, 16:32] = mids * np.float32(2.0 ** rng.integers(-6, 6)) * np.float32(1 + rng.integers(0, 8) / 8)
    if src == "bf16":
        W = f32(bf16(W))
    wa = Q.Array.from_numpy(bf16(W), Q.BFLOAT16) if src == "bf16" else Q.Array.from_numpy(W, Q.FLOAT32)
    wq, s = Q.quantize(wa, mode)
    rq, rs = O.quantize(mode, W)
    assert np.array_equal(s.numpy(), rs)
    assert np.array_equal(wq.numpy(), rq)
    buf = torch.zeros(N * K + 1, dtype=torch.bfloat16, device="cuda")
    out, stream = Q.Array.from_torch(buf[1:].view(N, K)), Q.Stream()
    Q.check(Q.lib.qmm_dequantize(ctypes.byref(out.h), wq.h, s.h, Q.qmm_array(None), Q.opt_int(), Q.opt_int(),
                                 mode.encode(), Q.qmm_array(None), Q.qmm_optional_dtype(0, False), stream.h))
    stream.sync()
    d, ref = out.numpy(), O.dequant_bf16(mode, rq, rs, K)
    assert np.array_equal(d, ref)


def test_freed_results_are_reused_in_stream_order():
    """Results freed on the null stream are handed to its next allocations of their size:
    live results never share memory, and a reused buffer holds the new result whatever the
    earlier one still queued."""
    rng = np.random.default_rng(5)
    ws = [O.quantize("nvfp4", f32(bf16(rng.standard_normal((n, 512)) * 0.02))) for n in (64, 64, 96, 2048)]
    refs = [O.dequant_bf16("nvfp4", w, s, 512) for w, s in ws]
    arrs = [(Q.Array.from_numpy(w, Q.UINT32), Q.Array.from_numpy(s, Q.UINT8)) for w, s in ws]
    for _ in range(3):
        live = [Q.dequantize(*a, "nvfp4") for a in arrs]
        spans = sorted((d.ptr, d.ptr + r.nbytes) for d, r in zip(live, refs))
        assert all(x[1] <= y[0] for x, y in zip(spans, spans[1:]))
        first = live[0].ptr
        live[0].free()
        again = Q.dequantize(*arrs[1], "nvfp4")  # the size just freed
        assert again.ptr == first
        for d, r in zip([again] + live[1:], [refs[1]] + refs[1:]):
            assert np.array_equal(d.numpy(), r)
    for n in range(1, 200):  # more sizes than are kept
        d = Q.dequantize(Q.Array.from_numpy(ws[3][0][:n], Q.UINT32), Q.Array.from_numpy(ws[3][1][:n], Q.UINT8), "nvfp4")
        if n % 50 == 0:
            assert np.array_equal(d.numpy(), refs[3][:n])


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
def test_reference_qmm_case_exact(mode):
    """src/model.zig:1561-1609 restated: integer W, x -> closed-form integer y (tighter than tol 0.05)."""
    W = np.array([(i % 7) - 3 for i in range(8 * 32)], np.float32).reshape(8, 32)
    x = np.array([(i % 5) - 2 for i in range(2 * 32)], np.float32).reshape(2, 32)
    wq, s = Q.quantize(Q.Array.from_numpy(W, Q.FLOAT32), mode)
    yexp = (x.astype(np.int64) @ W.astype(np.int64).T).astype(np.float32)
    y32 = Q.quantized_matmul(Q.Array.from_numpy(x, Q.FLOAT32), wq, s, mode).numpy()
    assert np.array_equal(y32, yexp)
    yb = Q.quantized_matmul(Q.Array.from_numpy(bf16(x), Q.BFLOAT16), wq, s, mode,
                            group_size=O.GROUP[mode], bits=O.BITS[mode]).numpy()
    assert np.array_equal(f32(yb), yexp)
    dq = Q.dequantize(wq, s, mode, dtype=Q.FLOAT32).numpy()
    assert np.array_equal(dq, W)


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
def test_reference_qmm_case_golden(mode):
    """The committed fixture of the same case: packed words and scales from the
    format definitions; the GPU quantizer, dequant and qmm must reproduce them."""
    import json
    from pathlib import Path

    g = json.loads((Path(__file__).resolve().parent / "golden" / "reference_qmm_case.json").read_text())
    gm = g["modes"][mode]
    W, x, y = (np.array(g[k], np.float32) for k in ("W", "x", "y"))
    wq, s = Q.quantize(Q.Array.from_numpy(W, Q.FLOAT32), mode)
    assert np.array_equal(wq.numpy(), np.array(gm["w"], np.uint32))
    assert np.array_equal(s.numpy(), np.array(gm["scales"], np.uint8))
    wg = Q.Array.from_numpy(np.array(gm["w"], np.uint32), Q.UINT32)
    sg = Q.Array.from_numpy(np.array(gm["scales"], np.uint8), Q.UINT8)
    assert np.array_equal(Q.dequantize(wg, sg, mode, dtype=Q.FLOAT32).numpy(), W)
    assert np.array_equal(Q.quantized_matmul(Q.Array.from_numpy(x, Q.FLOAT32), wg, sg, mode).numpy(), y)
    yb = Q.quantized_matmul(Q.Array.from_numpy(bf16(x), Q.BFLOAT16), wg, sg, mode).numpy()
    assert np.array_equal(f32(yb), y)


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K", [(256, 512), (61, 1536), (48, 5120), (37, 96)])
def test_decode_matches_oracle(mode, M, N, K):
    rng = np.random.default_rng(M * 1000 + N + K)
    wq, s = rand_w(rng, mode, N, K)
    xb = bf16(rng.standard_normal((M, K)))
    y = run_qmm(mode, xb, wq, s)
    ref = O.qmm(mode, xb, wq, s)
    ok, fro, worst = O.check_tolerance(f32(y), f32(ref), **TOL)
    assert ok, (fro, worst)
    # determinism: a second call gives identical bits
    assert np.array_equal(run_qmm(mode, xb, wq, s), y)


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("mode,N,K", [("nvfp4", 13, 17408), ("nvfp4", 37, 10752), ("nvfp4", 5, 33792),
                                      ("mxfp8", 11, 17408), ("mxfp8", 29, 5632)])
def test_decode_long_k_matches_oracle(mode, M, N, K):
    """Rows too long for the register-staged x (the down projection, K = 17408): x
    staged in LDS by DMA, rows streamed per wave; N not a multiple of the grid's
    waves, chunk counts not a multiple of the segment; K = 33792 at M >= 3 does not
    fit LDS and takes the looping kernel."""
    rng = np.random.default_rng(M * 7 + N + K)
    wq, s = rand_w(rng, mode, N, K)
    xb = bf16(rng.standard_normal((M, K)) * 0.5)
    y = run_qmm(mode, xb, wq, s)
    ref = O.qmm(mode, xb, wq, s)
    ok, fro, worst = O.check_tolerance(f32(y), f32(ref), **TOL)
    assert ok, (fro, worst)
    assert np.array_equal(run_qmm(mode, xb, wq, s), y)


@pytest.mark.parametrize("K", [128, 256, 384, 512])
def test_prefill_mxfp8_partial_last_round(K):
    """x rows 300 (ragged against every tile), W rows 33180: several rounds of tiles, the last
    one partial; the last columns are checked (plus a sample of the rest), all rows, at
    K = 128 to 512 (1 to 4 stages of W, around the ring's depth of 2 or 3), and a second call
    must return the same bits."""
    mode, M, N = "mxfp8", 300, 33180
    rng = np.random.default_rng(11)
    wq, s = rand_w(rng, mode, N, K)
    xb = bf16(rng.standard_normal((M, K)))
    y = run_qmm(mode, xb, wq, s)
    cols = np.unique(np.concatenate([np.arange(32768 - 40, N), rng.choice(N, size=64, replace=False)]))
    ref = O.qmm(mode, xb, wq, s, cols=cols)
    ok, fro, worst = O.check_tolerance(f32(y[:, cols]), f32(ref), **TOL)
    assert ok, (fro, worst)
    assert np.array_equal(run_qmm(mode, xb, wq, s), y)


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
@pytest.mark.parametrize("M", [1, 3, 20])
def test_f32_x_matches_oracle(mode, M):
    rng = np.random.default_rng(5 + M)
    N, K = 130, 1024
    wq, s = rand_w(rng, mode, N, K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    y = run_qmm(mode, x, wq, s, x_f32=True)
    ref = O.qmm(mode, x, wq, s, x_is_bf16=False, out="f32")
    rel = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    assert rel < 1e-5, rel


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
def test_one_hot_x_reads_back_dequantized_rows(mode):
    """In-kernel unpack is bit-exact: x = e_k returns deq(W)[:, k] exactly (f32 out)."""
    rng = np.random.default_rng(3)
    N, K = 64, 256
    w = rng.integers(0, 2 ** 32, size=(N, K * O.BITS[mode] // 32), dtype=np.uint32)
    if mode == "mxfp8":  # keep away from NaN codes and overflow
        b = w.view(np.uint8)
        b[(b & 0x7F) == 0x7F] = 0x10
        s = rng.integers(100, 150, size=(N, K // 32), dtype=np.uint8)
    else:
        s = rng.integers(0, 0x7F, size=(N, K // 16), dtype=np.uint8)
    ks = [0, 1, 7, 8, 31, 32, 100, 255]
    x = np.zeros((len(ks), K), np.float32)
    for i, k in enumerate(ks):
        x[i, k] = 1.0
    ref = O.dequant(mode, w, s, K)[:, ks].T
    y = run_qmm(mode, x[:8], w, s, x_f32=True)
    assert np.array_equal(y, ref)
    yb = run_qmm(mode, bf16(x[:8]), w, s)
    # compare values: a dequantized -0 sums to +0 in any matmul (-0 + +0 = +0)
    assert np.array_equal(f32(yb), f32(bf16(ref)))


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
@pytest.mark.parametrize("M,N,K", [(64, 256, 512), (300, 200, 1024), (129, 96, 5120), (17, 1000, 160),
                                   (40, 200, 384), (33, 130, 1152)])
def test_prefill_matches_oracle(mode, M, N, K):
    if mode == "mxfp8" and K % 32:
        pytest.skip("mxfp8 needs K % 32 == 0")
    rng = np.random.default_rng(M + N + K)
    wq, s = rand_w(rng, mode, N, K)
    xb = bf16(rng.standard_normal((M, K)))
    y = run_qmm(mode, xb, wq, s)
    ref = O.qmm(mode, xb, wq, s)
    ok, fro, worst = O.check_tolerance(f32(y), f32(ref), **TOL)
    assert ok, (fro, worst)


# K of one to three 64-element steps: the pipelined GEMMs' ring prologue issues fewer
# steps than it has stages, in tiles of 32 to 128 rows.
@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
@pytest.mark.parametrize("M,N,K", [(300, 300, 64), (300, 300, 128), (300, 300, 192), (40, 600, 128), (100, 520, 192)])
def test_prefill_short_k(mode, M, N, K):
    rng = np.random.default_rng(7 * M + N + K)
    wq, s = rand_w(rng, mode, N, K)
    xb = bf16(rng.standard_normal((M, K)))
    y = run_qmm(mode, xb, wq, s)
    ref = O.qmm(mode, xb, wq, s)
    ok, fro, worst = O.check_tolerance(f32(y), f32(ref), **TOL)
    assert ok, (fro, worst)


# The pipelined prefill GEMMs on weights over every code (all E2M1 nibbles / every
# finite E4M3 byte) and x with the edge groups: ragged N and M, several K steps,
# and the down projection's K = 17408 (checked on a column sample).
@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
@pytest.mark.parametrize("M,N,K", [(257, 1000, 1024), (40, 4099, 5120), (520, 384, 17408)])
def test_prefill_pipe_edge_values(mode, M, N, K):
    rng = np.random.default_rng(3 * M + N + K)
    wq, s = rand_packed(rng, mode, N, K)
    xb = make_x(rng, M, K, "edge")
    y = run_qmm(mode, xb, wq, s)
    cols = np.unique(np.concatenate([np.arange(0, N, max(1, N // 97)), np.arange(N - 9, N)]))
    ref = O.qmm(mode, xb, wq, s, cols=cols)
    ok, fro, worst = O.check_tolerance(f32(y[:, cols]), f32(ref), **TOL)
    assert ok, (fro, worst)
    assert np.array_equal(run_qmm(mode, xb, wq, s), y)


def test_rank3_x_and_inplace_output():
    """x [1, T, K] (the model's layer input, src/model.zig:1284) -> y [1, T, N]; a preallocated
    output of the exact shape is written in place."""
    rng = np.random.default_rng(8)
    mode, T, N, K = "nvfp4", 3, 64, 512
    wq, s = rand_w(rng, mode, N, K)
    xb = bf16(rng.standard_normal((1, T, K)))
    x = Q.Array.from_numpy(xb, Q.BFLOAT16)
    y = Q.quantized_matmul(x, Q.Array.from_numpy(wq, Q.UINT32), Q.Array.from_numpy(s, Q.UINT8), mode)
    assert y.shape == (1, T, N)
    ptr = y.ptr
    y2 = Q.quantized_matmul(x, Q.Array.from_numpy(wq, Q.UINT32), Q.Array.from_numpy(s, Q.UINT8), mode, out=y)
    assert y2.ptr == ptr
    ref = O.qmm(mode, xb.reshape(T, K), wq, s)
    ok, fro, worst = O.check_tolerance(f32(y.numpy().reshape(T, N)), f32(ref), **TOL)
    assert ok, (fro, worst)


@pytest.mark.parametrize("M", [1, 3, 40])
def test_dense_linear_matches_fp32_reference(M):
    """Dense bf16 fallback (linear, src/model.zig:200-211) against a float64 reference."""
    rng = np.random.default_rng(M)
    N, K = 200, 1024
    xb = bf16(rng.standard_normal((M, K)))
    wb = bf16(rng.standard_normal((N, K)) * 0.02)
    y = Q.linear(Q.Array.from_numpy(xb, Q.BFLOAT16), Q.Array.from_numpy(wb, Q.BFLOAT16)).numpy()
    ref = f32(xb).astype(np.float64) @ f32(wb).astype(np.float64).T
    refb = np.array([[O.f64_to_bf16_bits(v) for v in r] for r in ref], np.uint16)
    ok, fro, worst = O.check_tolerance(f32(y), f32(refb), **TOL)
    assert ok, (fro, worst)


@pytest.mark.parametrize("M,N,K", [
    (1, 3, 16), (2, 2049, 1040), (5, 700, 4112), (8, 2047, 2064), (3, 4100, 2064), (4, 6146, 4096),  # the GEMV's forms
    (6, 2048, 1040), (8, 5000, 528),
    (65, 129, 1040), (129, 273, 3328), (548, 256, 3584), (1030, 492, 2848), (700, 2500, 1296),
    (1000, 10240, 272), (1000, 10239, 288), (1300, 16400, 528)] + [c[:3] for c in G.DENSE])
def test_dense_linear_tiles(M, N, K):
    """The dense GEMV and GEMM at the edges of their tiles, K steps and splits (G.DENSE: every tile
    whole, split and both), against float64 on the GPU: within the one bf16 rounding (2^-8 of the value) and the fp32 sums' error, which is
    below 2^-24 K of sum |x| |w|."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen, device="cuda").to(torch.bfloat16)
    w = (torch.randn((N, K), generator=gen, device="cuda") * 0.02).to(torch.bfloat16)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    for _ in range(2):
        Q.linear(Q.Array.from_torch(x), Q.Array.from_torch(w), out=Q.Array.from_torch(y),
                 stream=Q.Stream.torch_current())
    ref = x.double() @ w.double().t()
    bound = ref.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().t()) * (K * 2.0 ** -24) + 1e-30
    assert torch.all((y.double() - ref).abs() <= bound)


class _RawStream:
    """A HIP stream of its own (torch hands out pooled ones), seen by torch and by the library."""

    def __init__(self):
        self.hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime torch and the library share
        self.ptr = ctypes.c_void_p()
        assert self.hip.hipStreamCreate(ctypes.byref(self.ptr)) == 0
        self.torch = torch.cuda.ExternalStream(self.ptr.value)

    def pool_used(self):
        """Bytes in use of the device's default memory pool, where the library's scratch lives."""
        pool, used = ctypes.c_void_p(), ctypes.c_uint64()
        assert self.hip.hipDeviceGetDefaultMemPool(ctypes.byref(pool), 0) == 0
        assert self.hip.hipMemPoolGetAttribute(pool, 7, ctypes.byref(used)) == 0  # hipMemPoolAttrUsedMemCurrent
        return used.value


def _dense(M, N, K, seed):
    """x, w, x @ w.T in float64 and its bound: one bf16 rounding and the fp32 sums' error."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    x = torch.randn((M, K), generator=gen, device="cuda").to(torch.bfloat16)
    w = (torch.randn((N, K), generator=gen, device="cuda") * 0.02).to(torch.bfloat16)
    ref = x.double() @ w.double().t()
    bound = ref.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().t()) * (K * 2.0 ** -24) + 1e-30
    return x, w, ref, bound


@pytest.mark.parametrize("M", [6, 7, 8, 16])
def test_dense_linear_takes_no_scratch_at_decode_or_in_a_graph(M):
    """x of up to 8 rows allocates nothing on a stream that has no workspace yet, and neither
    does a captured call of any size, whose tiles are then whole; replays on another stream
    beside eager calls of the capture stream, whose split tiles use that stream's workspace,
    leave both results right."""
    N, K = 10240, 5120
    x, w, ref, bound = _dense(M, N, K, M)
    x2, w2, ref2, bound2 = _dense(64, N, K, M + 100)
    y, y2 = (torch.full((m, N), float("nan"), dtype=torch.bfloat16, device="cuda") for m in (M, 64))
    xa, wa, x2a, w2a, ya, y2a = (Q.Array.from_torch(t) for t in (x, w, x2, w2, y, y2))
    s = _RawStream()
    torch.cuda.synchronize()
    used = s.pool_used()
    with torch.cuda.stream(s.torch):
        if M <= 8:
            Q.linear(xa, wa, out=ya, stream=Q.Stream.torch_current())
            torch.cuda.synchronize()
            assert s.pool_used() == used
            assert torch.all((y.double() - ref).abs() <= bound)
        Q.linear(x2a, w2a, out=y2a, stream=Q.Stream.torch_current())  # the stream's workspace is there from now on
    torch.cuda.synchronize()
    used = s.pool_used()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=s.torch):
        Q.linear(xa, wa, out=ya, stream=Q.Stream.torch_current())
    nodes = ctypes.c_size_t()
    assert s.hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(nodes)) == 0
    assert nodes.value == 1  # one kernel: no partial sums, no memory node
    graph.instantiate()
    other = torch.cuda.Stream()
    for _ in range(20):
        y.fill_(float("nan"))
        y2.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            graph.replay()
            graph.replay()
        with torch.cuda.stream(s.torch):
            for _ in range(3):
                Q.linear(x2a, w2a, out=y2a, stream=Q.Stream.torch_current())
        torch.cuda.synchronize()
        assert torch.all((y.double() - ref).abs() <= bound)
        assert torch.all((y2.double() - ref2).abs() <= bound2)
    assert s.pool_used() == used


@pytest.mark.parametrize("mode,M,N,K", [(m, *c) for m in ("nvfp4", "mxfp8") for c in [
    (17, 1, 32), (33, 129, 96), (64, 257, 224), (65, 300, 288), (33, 1000, 1056), (200, 320, 1024), (372, 328, 3456),
    (68, 2700, 3392), (383, 2416, 992), (1030, 1000, 544), (520, 5000, 256), (1691, 10240, 288), (2049, 16480, 512)]] +
    [("nvfp4", *c[:3]) for c in G.NVFP4] + [("mxfp8", *c[:3]) for c in G.MXFP8])
def test_prefill_tiles(mode, M, N, K):
    """The prefill GEMMs at the edges of their tiles, K steps, W stages and splits (G.NVFP4 and
    G.MXFP8: every tile whole, split and both), against float64 on the GPU: within the bf16 rounding (2^-8 of the value) and the fp32 sums' (and
    the mxfp8 split of x, at most 2^-12 of a block's largest) error, below 2^-12 + K 2^-24 of
    sum |x| |w| taken with each 32-block's largest |x|."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen, device="cuda").to(torch.bfloat16)
    W = (torch.randn((N, K), generator=gen, device="cuda") * 0.02).to(torch.bfloat16)
    st = Q.Stream.torch_current()
    wq, sc = Q.quantize(Q.Array.from_torch(W), mode, stream=st)
    Wd = torch.empty((N, K), dtype=torch.float32, device="cuda")
    Wd.copy_(torch.from_numpy(Q.dequantize(wq, sc, mode, dtype=Q.FLOAT32, stream=st).numpy(st)))
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    for _ in range(2):
        Q.quantized_matmul(Q.Array.from_torch(x), wq, sc, mode, out=Q.Array.from_torch(y), stream=st)
    ref = x.double() @ Wd.double().t()
    xm = x.double().abs().view(M, K // 32, 32).amax(-1, keepdim=True).expand(M, K // 32, 32).reshape(M, K)
    eps = K * 2.0 ** -24 + (2.0 ** -12 if mode == "mxfp8" else 0.0)
    bound = ref.abs() * 2.0 ** -8 + (xm @ Wd.double().abs().t()) * eps + 1e-30
    assert torch.all((y.double() - ref).abs() <= bound)


@pytest.mark.parametrize("M,N,K", [(9, 300, 96), (27, 4672, 1376), (200, 1000, 1056), (147, 2181, 8672),
                                   (5, 4672, 1344), (7, 4096, 1376), (8, 5000, 192)])
def test_mxfp8_exact_products_off_the_fp8_gemm(M, N, K):
    """mxfp8 at K % 64 = 32, and x of 5-8 rows at K % 128 != 0, multiplies x itself, not its two-part
    8-bit split: nearly every output is the exact sum's bf16.  fp32 sums of K terms are off by
    a few 2^-24 sqrt(K) of the output's rms, against a rounding step of 2^-8 of the value: at
    most 2^-14 sqrt(K) of the outputs may round the other way (K = 8672: 0.6%; a split x gives
    1.2% at every K).  The same through the MLP's projections and in a group."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + K)
    x = torch.randn((M, K), generator=gen, device="cuda").to(torch.bfloat16)
    W = (torch.randn((N, K), generator=gen, device="cuda") * 0.02).to(torch.bfloat16)
    st = Q.Stream.torch_current()
    wq, sc = Q.quantize(Q.Array.from_torch(W), "mxfp8", stream=st)
    Wd = torch.from_numpy(Q.dequantize(wq, sc, "mxfp8", dtype=Q.FLOAT32, stream=st).numpy(st)).cuda().double()
    ref = (x.double() @ Wd.t()).to(torch.bfloat16)
    xa = Q.Array.from_torch(x)
    y = Q.quantized_matmul(xa, wq, sc, "mxfp8", stream=st)
    yg = Q.quantized_matmul_group(xa, [wq], [sc], "mxfp8", stream=st)[0]
    h = Q.mlp_gate_up_silu(xa, wq, sc, wq, sc, "mxfp8", stream=st)
    assert np.array_equal(h.numpy(st), Q.silu_mul(y, y, stream=st).numpy(st))
    assert np.array_equal(yg.numpy(st), y.numpy(st))
    other = np.mean(y.numpy(st) != ref.view(torch.int16).cpu().numpy().view(np.uint16))
    assert other <= min(2.0 ** -14 * K ** 0.5, 0.006), other


# ---------------------------------------------------------------- MLP activation and the fused gate/up
def test_silu_mul_matches_oracle():
    """src/model.zig:405-415 / :451-456 on the GPU: bf16 chain within one ulp of the
    oracle's (sigmoid in f32 here, f64 there); f32 arrays against numpy."""
    rng = np.random.default_rng(31)
    g = bf16(rng.standard_normal((7, 999)) * 6)
    u = bf16(rng.standard_normal((7, 999)))
    h = Q.silu_mul(Q.Array.from_numpy(g, Q.BFLOAT16), Q.Array.from_numpy(u, Q.BFLOAT16)).numpy()
    ref = O.silu_mul_bf16(g, u)
    diff = np.abs(h.astype(np.int32) - ref.astype(np.int32))
    assert diff.max() <= 1 and (diff == 0).mean() > 0.995
    gf = (rng.standard_normal(4096) * 6).astype(np.float32)
    uf = rng.standard_normal(4096).astype(np.float32)
    hf = Q.silu_mul(Q.Array.from_numpy(gf, Q.FLOAT32), Q.Array.from_numpy(uf, Q.FLOAT32)).numpy()
    ref_f = (gf.astype(np.float64) / (1 + np.exp(-gf.astype(np.float64)))) * uf
    assert np.allclose(hf, ref_f, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
@pytest.mark.parametrize("M,N,K", [(1, 200, 512), (2, 96, 5120), (3, 61, 1536), (4, 48, 5120), (20, 72, 512),
                                   (300, 130, 384), (40, 96, 192)])
def test_mlp_gate_up_silu_matches_oracle(mode, M, N, K):
    """silu(x Wg^T) * (x Wu^T) (src/model.zig:905-913): fused decode kernels for M <= 4, one
    prefill GEMM for larger M; equal to quantized_matmul x 2 + silu_mul bit for bit, and
    within tolerance of the oracle's chain."""
    rng = np.random.default_rng(M * 100 + N + K)
    wg, sg = rand_w(rng, mode, N, K)
    wu, su = rand_w(rng, mode, N, K)
    xb = bf16(rng.standard_normal((M, K)))
    A = lambda a, d: Q.Array.from_numpy(a, d)
    x = A(xb, Q.BFLOAT16)
    h = Q.mlp_gate_up_silu(x, A(wg, Q.UINT32), A(sg, Q.UINT8), A(wu, Q.UINT32), A(su, Q.UINT8), mode).numpy()
    g = Q.quantized_matmul(x, A(wg, Q.UINT32), A(sg, Q.UINT8), mode)
    u = Q.quantized_matmul(x, A(wu, Q.UINT32), A(su, Q.UINT8), mode)
    h2 = Q.silu_mul(g, u).numpy()
    assert np.array_equal(h, h2)
    ref = O.silu_mul_bf16(O.qmm(mode, xb, wg, sg), O.qmm(mode, xb, wu, su))
    ok, fro, worst = O.check_tolerance(f32(h), f32(ref), **TOL)
    assert ok, (fro, worst)


def rand_packed(rng, mode, N, K, period=4099):
    """Random packed weights over every code: all E2M1 nibbles (nvfp4) or every finite
    E4M3 byte with |v| < 2 (mxfp8), with group scales in a moderate range.  Rows
    repeat with a period of 4099 (not a multiple of the 16-row blocks) to keep
    generation fast at large N."""
    R = min(N, period)
    if mode == "nvfp4":
        wq = np.frombuffer(rng.bytes(R * K // 2), np.uint32).reshape(R, K // 8)
        s = rng.integers(0x20, 0x48, size=(R, K // 16), dtype=np.uint8)  # E4M3 2^-4 .. 2^1
    else:
        b = np.frombuffer(rng.bytes(R * K), np.uint8) & 0xBF  # exponent field <= 7: no NaN code, |v| < 2
        wq = b.view(np.uint32).reshape(R, K // 4)
        s = rng.integers(118, 132, size=(R, K // 32), dtype=np.uint8)  # E8M0 2^-9 .. 2^4
    if N > R:
        wq = np.resize(wq, (N, wq.shape[1]))
        s = np.resize(s, (N, s.shape[1]))
    return np.ascontiguousarray(wq), np.ascontiguousarray(s)


def make_x(rng, M, K, kind):
    """bf16 x ~ N(0,1); "edge" plants groups that stress the E4M3 hi/lo split: zeros,
    one value 2^23 above the rest of its group, bf16 subnormals, a wide linear ramp,
    a group scaled by 1e-6.  Magnitudes stay O(10) so errors elsewhere stay visible."""
    x = rng.standard_normal((M, K)).astype(np.float32)
    if kind == "edge":
        x[:, 0:16] = 0.0
        x[:, 16:32] = 1e-6
        x[:, 20] = 8.0
        x[:, 32:48] = np.float32(2.0 ** -130)  # bf16 subnormal
        x[:, 48:64] = np.linspace(-12.0, 12.0, 16, dtype=np.float32)
        x[:, 96:128] *= 1e-6
    return bf16(x)


# Shapes above the MFMA decode path's thresholds (K = 5120: from N = 4096, nvfp4 M = 1
# not at 17-24 rows per workgroup): ragged row blocks (N % 16 != 0), and a row
# range per workgroup long enough (N = 70001) to need several partial-sum flushes.
# nvfp4 M = 3-4 runs the 32x32x64 form (32-row blocks, flushes every 4 blocks);
# mxfp8 M = 5-8 the 16x16x128 form with all 16 A columns (8 rows x hi|lo) live, M = 9-16
# with two A operands per chunk (their records made 8 rows at a time); nvfp4 M = 5-8 the
# dequantizing kernel (W -> bf16, all 16 x rows on the bf16 MFMA), as nvfp4 M = 9-16, down
# to N = 100 (7 workgroups of 14-15 rows).  N = 17408 (68 rows per workgroup), 10240 (40)
# and 12288 (48) end every workgroup's range with a short row block, whose units load only
# its rows; so do N = 5120 (20) and 6144 (24) with two row blocks, the second short.
@pytest.mark.parametrize("mode,M,N", [("nvfp4", 1, 16400), ("nvfp4", 1, 70001), ("nvfp4", 2, 4099),
                                      ("nvfp4", 2, 16384), ("nvfp4", 3, 4099), ("nvfp4", 3, 70001),
                                      ("nvfp4", 4, 16400), ("mxfp8", 2, 4101), ("mxfp8", 3, 8192),
                                      ("mxfp8", 4, 4096), ("mxfp8", 4, 70001), ("mxfp8", 5, 4101),
                                      ("mxfp8", 6, 8192), ("mxfp8", 7, 4096), ("mxfp8", 8, 70001),
                                      ("mxfp8", 9, 4101), ("mxfp8", 12, 8192), ("mxfp8", 15, 4096),
                                      ("mxfp8", 16, 70001), ("nvfp4", 5, 4099), ("nvfp4", 6, 70001),
                                      ("nvfp4", 7, 5120), ("nvfp4", 8, 16400), ("nvfp4", 9, 4099),
                                      ("nvfp4", 12, 70001), ("nvfp4", 16, 16400), ("nvfp4", 13, 100),
                                      ("nvfp4", 1, 17408), ("nvfp4", 2, 17408), ("nvfp4", 3, 17408),
                                      ("nvfp4", 3, 10240), ("nvfp4", 4, 12288), ("nvfp4", 2, 5120),
                                      ("nvfp4", 2, 6144), ("mxfp8", 2, 5120), ("mxfp8", 4, 6144),
                                      ("mxfp8", 8, 5120), ("mxfp8", 2, 17408), ("mxfp8", 3, 10240),
                                      ("mxfp8", 8, 17408), ("nvfp4", 1, 4096), ("nvfp4", 1, 10240),
                                      ("nvfp4", 1, 12288)])
@pytest.mark.parametrize("xkind", ["normal", "edge"])
def test_decode_mfma_shapes_match_oracle(mode, M, N, xkind):
    K = 5120
    rng = np.random.default_rng(N * 10 + M)
    wq, s = rand_packed(rng, mode, N, K)
    xb = make_x(rng, M, K, xkind)
    y = run_qmm(mode, xb, wq, s)
    cols = np.unique(np.concatenate([np.arange(0, N, 7), np.arange(N - 40, N), np.arange(40)]))
    ref = O.qmm(mode, xb, wq, s, cols=cols)
    ok, fro, worst = O.check_tolerance(f32(y[:, cols]), f32(ref), **TOL)
    assert ok, (fro, worst)
    assert np.array_equal(run_qmm(mode, xb, wq, s), y)


# K = 17408 (the MLP down projection): 34 slices of 512 walked by 12 waves in 3
# passes, the last pass with 2 slices past K.  The edge groups are planted in
# the first slice of every pass and in the last slice.
@pytest.mark.parametrize("mode,M,N", [("nvfp4", 1, 5120), ("nvfp4", 2, 4099), ("nvfp4", 3, 5120),
                                      ("nvfp4", 4, 4099), ("mxfp8", 1, 5120), ("mxfp8", 1, 4101),
                                      ("mxfp8", 2, 5120), ("mxfp8", 3, 4101), ("mxfp8", 4, 8192),
                                      ("mxfp8", 5, 5120), ("mxfp8", 6, 4101),
                                      ("mxfp8", 10, 5120), ("nvfp4", 7, 5120)])
@pytest.mark.parametrize("xkind", ["normal", "edge"])
def test_decode_mfma_down_shapes_match_oracle(mode, M, N, xkind):
    K = 17408
    rng = np.random.default_rng(N * 10 + M + 1)
    wq, s = rand_packed(rng, mode, N, K)
    xb = make_x(rng, M, K, xkind)
    if xkind == "edge":
        for off in (12 * 512, 24 * 512, K - 512):
            xb[:, off:off + 128] = xb[:, 0:128]
    y = run_qmm(mode, xb, wq, s)
    cols = np.unique(np.concatenate([np.arange(0, N, 11), np.arange(N - 40, N), np.arange(40)]))
    ref = O.qmm(mode, xb, wq, s, cols=cols)
    ok, fro, worst = O.check_tolerance(f32(y[:, cols]), f32(ref), **TOL)
    assert ok, (fro, worst)
    assert np.array_equal(run_qmm(mode, xb, wq, s), y)


# The other row lengths of the model on the MFMA kernels: K = 6144 (o_proj /
# out_proj: 12 waves, one pass) and K = 10240 (mtp.fc: 10 waves, two passes;
# nvfp4 M = 1 takes it too).  Edge groups in the first slice of every pass and in
# the last slice.
@pytest.mark.parametrize("K", [6144, 10240])
@pytest.mark.parametrize("mode,M,N", [("nvfp4", 1, 5120), ("nvfp4", 2, 4099), ("nvfp4", 3, 5120),
                                      ("nvfp4", 4, 4099), ("mxfp8", 1, 5120), ("mxfp8", 1, 4101),
                                      ("mxfp8", 2, 5120), ("mxfp8", 3, 4101), ("mxfp8", 4, 8192),
                                      ("mxfp8", 6, 5120), ("mxfp8", 8, 4101),
                                      ("mxfp8", 13, 5120), ("mxfp8", 16, 4101), ("nvfp4", 6, 4099),
                                      ("nvfp4", 10, 5120), ("nvfp4", 16, 4099)])
@pytest.mark.parametrize("xkind", ["normal", "edge"])
def test_decode_mfma_other_k_match_oracle(K, mode, M, N, xkind):
    rng = np.random.default_rng(N * 10 + M + K)
    wq, s = rand_packed(rng, mode, N, K)
    xb = make_x(rng, M, K, xkind)
    if xkind == "edge":
        for off in (5120, K - 512):
            xb[:, off:off + 128] = xb[:, 0:128]
    y = run_qmm(mode, xb, wq, s)
    cols = np.unique(np.concatenate([np.arange(0, N, 11), np.arange(N - 40, N), np.arange(40)]))
    ref = O.qmm(mode, xb, wq, s, cols=cols)
    ok, fro, worst = O.check_tolerance(f32(y[:, cols]), f32(ref), **TOL)
    assert ok, (fro, worst)
    assert np.array_equal(run_qmm(mode, xb, wq, s), y)


@pytest.mark.parametrize("M,N,K", [(3, 5120, 128), (4, 5121, 1152), (5, 4096, 4096), (6, 4111, 3968), (8, 16384, 384),
                                   (3, 8200, 2944), (4, 4097, 4224), (3, 4100, 12288), (4, 20000, 8320)])
def test_qmv_any_k(M, N, K):
    """x of 3-8 rows at row lengths of any multiple of 128: whole and half last slices, one and
    several passes, ranges that end in partial row blocks; plain, grouped and as an MLP.  A
    row's sums do not depend on the call, so grouped and fused results equal the plain ones."""
    rng = np.random.default_rng(M + N + K)
    wq, s = rand_packed(rng, "nvfp4", N, K)
    xb = make_x(rng, M, K, "edge")
    y = run_qmm("nvfp4", xb, wq, s)
    cols = np.unique(np.concatenate([np.arange(0, N, 37), np.arange(N - 20, N)]))
    ok, fro, worst = O.check_tolerance(f32(y[:, cols]), f32(O.qmm("nvfp4", xb, wq, s, cols=cols)), **TOL)
    assert ok, (fro, worst)
    x, A = Q.Array.from_numpy(xb, Q.BFLOAT16), Q.Array.from_numpy
    wu, su = rand_packed(rng, "nvfp4", N, K)
    gate, up = (A(wq, Q.UINT32), A(s, Q.UINT8)), (A(wu, Q.UINT32), A(su, Q.UINT8))
    h = Q.mlp_gate_up_silu(x, *gate, *up, "nvfp4").numpy()
    g, u = Q.quantized_matmul(x, *gate, "nvfp4"), Q.quantized_matmul(x, *up, "nvfp4")
    assert np.array_equal(h, Q.silu_mul(g, u).numpy())
    tw, ts = torch.tensor(wq.view(np.int32)).cuda(), torch.tensor(s).cuda()
    n0 = N - 1000
    outs = Q.quantized_matmul_group(x, [Q.Array.from_torch(tw[:n0]), Q.Array.from_torch(tw[n0:])],
                                    [Q.Array.from_torch(ts[:n0]), Q.Array.from_torch(ts[n0:])], "nvfp4")
    assert np.array_equal(np.concatenate([o.numpy() for o in outs], 1), y)


class _KernelNode(ctypes.Structure):
    """hipKernelNodeParams."""
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", ctypes.c_uint * 3), ("args", ctypes.c_void_p), ("lds", ctypes.c_uint)]


def kernels_of(call):
    """[(mangled name, blocks)] of the kernels that call(stream) launches, in some order."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(Q.Stream.torch_current())  # the stream's workspace and the scale copies are there after it
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=side):
        call(Q.Stream.torch_current())
    raw, n, kind, node = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t(), ctypes.c_int(), _KernelNode()
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes, out = (ctypes.c_void_p * n.value)(), []
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    for v in nodes:
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(v), ctypes.byref(kind)) == 0
        if kind.value == 0:  # hipGraphNodeTypeKernel
            assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(v), ctypes.byref(node)) == 0
            out.append((hip.hipKernelNameRefByPtr(ctypes.c_void_p(node.func), None).decode(), node.grid[0]))
    return out


def tiles_of(call, M, N, mlp=False):
    """("TM x TN", "whole", "split" or "both") of the one pipelined GEMM that call(stream) launches:
    its tiles, and whether they run whole, all split along K, or the last ones split."""
    ks = [(n, g) for n, g in kernels_of(call) if "Geom" in n]
    (name, blocks), = [k for k in ks if "reduce" not in k[0]]
    fi, fj, wm, wn = (int(v) for v in re.search(r"GeomILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E", name).groups())
    TM, TN = 32 * fi * wm, 32 * fj * wn
    total, left = -(-M // TM) * -(-N // TN) * (2 if mlp else 1), 0
    if len(ks) > 1:
        (_, rblocks), = [k for k in ks if "reduce" in k[0]]
        left = rblocks * 1024 * (2 if mlp else 1) // (TM * TN)
        assert (blocks - (total - left)) % left == 0 and blocks > total
    else:
        assert blocks == total
    return "%dx%d" % (TM, TN), "whole" if left == 0 else "split" if left == total else "both"


def _quantized(gen, mode, N, K):
    """A quantized weight, and it in float64."""
    st = Q.Stream.torch_current()
    wq, sc = Q.quantize(Q.Array.from_torch((torch.randn((N, K), generator=gen, device="cuda") * 0.02).to(torch.bfloat16)),
                        mode, stream=st)
    return (wq, sc), torch.from_numpy(Q.dequantize(wq, sc, mode, dtype=Q.FLOAT32, stream=st).numpy(st)).cuda().double()


def _random_nvfp4(gen, N, K):
    """Packed nvfp4 over every code, moderate scales, and the weight in float64."""
    w = torch.randint(0, 256, (N, K // 2), generator=gen, device="cuda", dtype=torch.uint8)
    s = torch.randint(0x20, 0x48, (N, K // 16), generator=gen, device="cuda", dtype=torch.uint8)
    v = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device="cuda")
    d = torch.stack((v[(w & 15).int()], v[(w >> 4).int()]), -1).view(N, K // 16, 16)
    return w.view(torch.int32), s, (d * s.view(torch.float8_e4m3fn).double().unsqueeze(-1)).view(N, K)


@pytest.mark.parametrize("M,N,K,flushes,mlp_flushes", [(6, 40001, 4096, 2, 3), (3, 70001, 2560, 2, 3), (4, 64500, 8192, 1, 0)])
def test_qmv_any_many_row_blocks(M, N, K, flushes, mlp_flushes):
    """Ranges of more row blocks per workgroup than the partial sums have slots for (8 in one pass):
    several flushes, the last one short; and a two-pass MLP whose row blocks do not fit the LDS
    (0 flushes: it runs as three calls).  Plain, grouped and as an MLP, every output against float64:
    within the bf16 rounding (2^-8 of the value) and K 2^-24 of sum |x| |w|."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + K)
    x = torch.randn((M, K), generator=gen, device="cuda").to(torch.bfloat16)
    st, A = Q.Stream.torch_current(), Q.Array.from_torch
    xa, new = A(x), lambda n: torch.full((M, n), float("nan"), dtype=torch.bfloat16, device="cuda")  # noqa: E731
    w, s, d = _random_nvfp4(gen, N, K)
    ref = x.double() @ d.t()
    bound = ref.abs() * 2.0 ** -8 + (x.double().abs() @ d.abs().t()) * (K * 2.0 ** -24) + 1e-30
    del d
    y, parts, h, g, u, h2 = new(N), [new(N - 12345), new(12345)], new(N), new(N), new(N), new(N)
    Q.quantized_matmul(xa, A(w), A(s), "nvfp4", out=A(y), stream=st)
    assert torch.all((y.double() - ref).abs() <= bound)
    cut = N - 12345
    Q.quantized_matmul_group(xa, [A(w[:cut]), A(w[cut:])], [A(s[:cut]), A(s[cut:])], "nvfp4",
                             outs=[A(p) for p in parts], stream=st)
    assert torch.equal(torch.cat(parts, 1), y)
    wu, su, _ = _random_nvfp4(gen, N, K)
    mlp = lambda st: Q.mlp_gate_up_silu(xa, A(w), A(s), A(wu), A(su), "nvfp4", out=A(h), stream=st)  # noqa: E731
    mlp(st)
    Q.quantized_matmul(xa, A(wu), A(su), "nvfp4", out=A(u), stream=st)
    Q.silu_mul(A(y), A(u), out=A(h2), stream=st)
    assert torch.equal(h, h2)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        return

    # the row blocks of a workgroup: those of its rows, in units of 16 (MLP: 8)
    def check(call, rows, want):
        (name, blocks), = [k for k in kernels_of(call) if "qmv_any" in k[0]]
        row_blocks = ceil(ceil(N / blocks) / rows)
        assert (ceil(row_blocks / 8) if K <= 4096 else 1) == want

    check(lambda st: Q.quantized_matmul(xa, A(w), A(s), "nvfp4", out=A(y), stream=st), 16, flushes)
    if mlp_flushes:
        check(mlp, 8, mlp_flushes)
    else:
        names = [n for n, _ in kernels_of(mlp)]
        assert sum("qmv_any" in n for n in names) == 2 and sum("silu_mul" in n for n in names) == 1


MLP_TILES = [("nvfp4", *c) for c in G.NVFP4_MLP] + [("mxfp8", *c) for c in G.MXFP8_MLP] + [
    ("mxfp8", 17, 33, 96, "none", ""), ("mxfp8", 64, 65, 224, "none", "")]  # K % 64 = 32


@pytest.mark.parametrize("mode,M,N,K,tile,split", MLP_TILES)
def test_mlp_prefill_tiles(mode, M, N, K, tile, split):
    """The one-launch prefill MLP, every tile of it whole, split along K and both, equals
    quantized_matmul x 2 + silu_mul bit for bit: it splits each column's sums as the projections
    alone do."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + K)
    (gate, _), (up, _) = _quantized(gen, mode, N, K), _quantized(gen, mode, N, K)
    x = Q.Array.from_torch(torch.randn((M, K), generator=gen, device="cuda").to(torch.bfloat16))
    h, g, u, h2 = (torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(4))
    st = Q.Stream.torch_current()
    for _ in range(2):
        Q.mlp_gate_up_silu(x, *gate, *up, mode, out=Q.Array.from_torch(h), stream=st)
        Q.quantized_matmul(x, *gate, mode, out=Q.Array.from_torch(g), stream=st)
        Q.quantized_matmul(x, *up, mode, out=Q.Array.from_torch(u), stream=st)
        Q.silu_mul(Q.Array.from_torch(g), Q.Array.from_torch(u), out=Q.Array.from_torch(h2), stream=st)
        assert not h2.isnan().any()
        assert torch.equal(h.view(torch.int16), h2.view(torch.int16))
    call = lambda s: Q.mlp_gate_up_silu(x, *gate, *up, mode, out=Q.Array.from_torch(h), stream=s)  # noqa: E731
    if tile == "none":
        assert sum("silu_mul" in n for n, _ in kernels_of(call)) == 1
    elif torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert tiles_of(call, M, N, mlp=True) == (tile, split)


@pytest.mark.parametrize("mode,M,N", [("nvfp4", 1, 16400), ("nvfp4", 2, 4099), ("nvfp4", 3, 4099),
                                      ("nvfp4", 4, 16400), ("mxfp8", 3, 4101), ("mxfp8", 4, 70001),
                                      ("mxfp8", 6, 4101), ("nvfp4", 5, 4099), ("nvfp4", 1, 17408),
                                      ("nvfp4", 2, 17408), ("nvfp4", 3, 17408), ("nvfp4", 4, 17408)])
def test_mlp_gate_up_silu_mfma_shapes(mode, M, N):
    """The fused MLP on the MFMA path: equal to two quantized_matmul + silu_mul bit for
    bit, and within tolerance of the oracle's chain on a row sample.  At N = 17408 (the
    model's MLP: 68 rows per workgroup) each range ends in a short row block."""
    K = 5120
    rng = np.random.default_rng(N + 7 * M)
    wg, sg = rand_packed(rng, mode, N, K)
    wu, su = rand_packed(rng, mode, N, K)
    xb = make_x(rng, M, K, "edge")
    A = lambda a, d: Q.Array.from_numpy(a, d)
    x = A(xb, Q.BFLOAT16)
    h = Q.mlp_gate_up_silu(x, A(wg, Q.UINT32), A(sg, Q.UINT8), A(wu, Q.UINT32), A(su, Q.UINT8), mode).numpy()
    g = Q.quantized_matmul(x, A(wg, Q.UINT32), A(sg, Q.UINT8), mode)
    u = Q.quantized_matmul(x, A(wu, Q.UINT32), A(su, Q.UINT8), mode)
    assert np.array_equal(h, Q.silu_mul(g, u).numpy())
    cols = np.unique(np.concatenate([np.arange(0, N, 5), np.arange(N - 20, N)]))
    ref = O.silu_mul_bf16(O.qmm(mode, xb, wg, sg, cols=cols), O.qmm(mode, xb, wu, su, cols=cols))
    ok, fro, worst = O.check_tolerance(f32(h[:, cols]), f32(ref), **TOL)
    assert ok, (fro, worst)


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
def test_prefill_scales_tiled_copy_kept_with_handle(mode):
    """Prefill calls read the scales in a tile-major copy the library makes once per scales
    handle (at its first eager prefill call) and keeps with it.  A call captured into a
    graph before that copy exists repacks into the stream's workspace inside the graph;
    replays of that graph, the eager call that makes the copy and later calls that reuse it
    all give identical bits, within the bar of the oracle."""
    import torch

    M, N, K = 300, 1000, 1024
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(77)
    W = (torch.randn((N, K), generator=g, device=dev) * 0.02).to(torch.bfloat16)
    x = torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16)
    wq, sc = Q.quantize(Q.Array.from_torch(W), mode)
    xa = Q.Array.from_torch(x)
    nan = lambda: torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)  # noqa: E731
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    y_graph = nan()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        Q.quantized_matmul(xa, wq, sc, mode, out=Q.Array.from_torch(y_graph), stream=Q.Stream.torch_current())
    outs = []
    for _ in range(2):
        y_graph.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        outs.append(y_graph.clone())
    for _ in range(3):  # the first makes the tile-major copy, the others reuse it
        y = nan()
        Q.quantized_matmul(xa, wq, sc, mode, out=Q.Array.from_torch(y))
        outs.append(y)
    torch.cuda.synchronize()
    for y in outs:
        assert torch.isfinite(y.float()).all()
        assert torch.equal(y.view(torch.int16), outs[0].view(torch.int16))
    ref = O.qmm(mode, x.view(torch.int16).cpu().numpy().view(np.uint16), wq.numpy(), sc.numpy())
    ok, fro, worst = O.check_tolerance(f32(outs[-1].view(torch.int16).cpu().numpy().view(np.uint16)), f32(ref), **TOL)
    assert ok, (fro, worst)


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
def test_prefill_two_streams_at_once(mode):
    """Prefill calls issued on two streams without synchronising between them: each stream
    has its own workspace (the mxfp8 x split lives there), so the interleaved calls give the
    same bits as the same calls run one after the other."""
    import torch

    M, N, K = 520, 2048, 2048
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(78)
    W = (torch.randn((N, K), generator=g, device=dev) * 0.02).to(torch.bfloat16)
    xs = [torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16) for _ in range(2)]
    wq, sc = Q.quantize(Q.Array.from_torch(W), mode)
    refs = [Q.quantized_matmul(Q.Array.from_torch(x), wq, sc, mode) for x in xs]
    torch.cuda.synchronize()
    refs = [torch.from_numpy(r.numpy().view(np.int16)) for r in refs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    for _ in range(4):
        for k in range(2):
            with torch.cuda.stream(streams[k]):
                y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
                Q.quantized_matmul(Q.Array.from_torch(xs[k]), wq, sc, mode, out=Q.Array.from_torch(y),
                                   stream=Q.Stream.torch_current())
                outs[k].append(y)
    torch.cuda.synchronize()
    for k in range(2):
        for y in outs[k]:
            assert torch.equal(y.view(torch.int16).cpu(), refs[k])
    ref = O.qmm(mode, xs[1].view(torch.int16).cpu().numpy().view(np.uint16), wq.numpy(), sc.numpy(),
                cols=np.arange(0, N, 7))
    ok, fro, worst = O.check_tolerance(f32(refs[1].numpy().view(np.uint16)[:, ::7]), f32(ref), **TOL)
    assert ok, (fro, worst)


def test_calls_from_several_host_threads():
    """Four host threads, each with its own stream, issue decode and prefill calls of both
    modes at the same time (the binding releases the GIL inside the library): every output
    equals the same call run alone, bit for bit."""
    import threading

    import torch

    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(91)
    K, N = 1024, 1536
    W = (torch.randn((N, K), generator=g, device=dev) * 0.02).to(torch.bfloat16)
    quant = {mode: Q.quantize(Q.Array.from_torch(W), mode) for mode in ("mxfp8", "nvfp4")}
    cases = [(mode, M) for mode in ("mxfp8", "nvfp4") for M in (1, 3, 300)]
    xs = {M: torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16) for M in (1, 3, 300)}
    refs = {}
    for mode, M in cases:
        wq, sc = quant[mode]
        refs[mode, M] = Q.quantized_matmul(Q.Array.from_torch(xs[M]), wq, sc, mode).numpy().view(np.int16)
    torch.cuda.synchronize()
    outs, errors = {}, []

    def worker(t):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for rep in range(3):
                    for mode, M in cases[t % 2:] + cases[:t % 2]:
                        wq, sc = quant[mode]
                        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
                        Q.quantized_matmul(Q.Array.from_torch(xs[M]), wq, sc, mode, out=Q.Array.from_torch(y),
                                           stream=Q.Stream.torch_current())
                        outs[t, rep, mode, M] = y
            s.synchronize()
        except Exception as e:  # reported by the main thread
            errors.append(repr(e))

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    torch.cuda.synchronize()
    assert not errors, errors
    assert len(outs) == 4 * 3 * len(cases)
    for (t, rep, mode, M), y in outs.items():
        assert np.array_equal(y.view(torch.int16).cpu().numpy(), refs[mode, M]), (t, rep, mode, M)
    assert Q.take_error() is None


def test_calls_from_several_host_threads_on_one_stream():
    """Four host threads issue the same calls on the null stream, each with its own x and its own
    results: calls of several launches (split tiles and their reduce, the split of x, the
    chunked recurrence) share the stream's workspace, and no thread's launches come between
    another's, so every output equals the call run alone, bit for bit."""
    import threading

    gen = torch.Generator(device="cuda")
    gen.manual_seed(92)
    rn = lambda *s: torch.randn(s, generator=gen, device="cuda")  # noqa: E731
    st, A, M, N, K, T = Q.Stream(), Q.Array.from_torch, 24, 2048, 4128, 130
    wd = (rn(N, K) * 0.02).to(torch.bfloat16)
    quant = {mode: Q.quantize(A(wd), mode) for mode in ("mxfp8", "nvfp4")}
    k = rn(1, T, 2, 128) / 128 ** 0.5
    gdn = [A(t) for t in (k.to(torch.bfloat16), torch.exp(-0.7 * torch.rand((1, T, 2), generator=gen, device="cuda")),
                          torch.sigmoid(rn(1, T, 2)).to(torch.bfloat16), rn(1, 2, 128, 128) * 0.1)]
    xs = [rn(M, K).to(torch.bfloat16) for _ in range(4)]
    vs = [rn(1, T, 2, 128).to(torch.bfloat16) for _ in range(4)]
    empty = lambda *s, dt=torch.bfloat16: torch.full(s, float("nan"), dtype=dt, device="cuda")  # noqa: E731
    outs = [dict(d=empty(M, N), q=empty(M, N), f=empty(M, N), h=empty(M, N), y=empty(1, T, 2, 128),
                 s=empty(1, 2, 128, 128, dt=torch.float32)) for _ in range(4)]

    def calls(t):
        x, o = A(xs[t]), {n: A(v) for n, v in outs[t].items()}
        Q.linear(x, A(wd), out=o["d"], stream=st)
        Q.quantized_matmul(x, *quant["nvfp4"], "nvfp4", out=o["q"], stream=st)
        Q.quantized_matmul(x, *quant["mxfp8"], "mxfp8", out=o["f"], stream=st)
        Q.mlp_gate_up_silu(x, *quant["nvfp4"], *quant["nvfp4"], "nvfp4", out=o["h"], stream=st)
        Q.gdn_recurrence(gdn[0], gdn[0], A(vs[t]), *gdn[1:], y=o["y"], state_out=o["s"], stream=st)

    refs = []
    for t in range(4):
        calls(t)
        torch.cuda.synchronize()
        refs.append({n: v.clone() for n, v in outs[t].items()})
    bad, errors = [], []

    def worker(t, barrier):
        try:
            for _ in range(10):
                barrier.wait()
                calls(t)
        except Exception as e:  # reported by the main thread
            errors.append(repr(e))

    for rep in range(20):
        barrier = threading.Barrier(4)
        threads = [threading.Thread(target=worker, args=(t, barrier)) for t in range(4)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        torch.cuda.synchronize()
        bad += [(rep, t, n) for t in range(4) for n, v in outs[t].items() if not torch.equal(v, refs[t][n])]
    assert not errors, errors
    assert not bad, bad
    assert Q.take_error() is None


@functools.lru_cache(maxsize=2)
def _nf_weights(mode, N, K):
    return rand_w(np.random.default_rng(4242), mode, N, K)


# Non-finite x: the reference multiplies dequantized weights by x in floating point, so a
# NaN in row m of x makes every output of row m NaN, and an infinity makes every output
# of the row non-finite (±inf, or NaN where the weight is zero); the other rows are
# unaffected.  Every kernel family: the unpacking GEMV, the MFMA GEMV (16x16x128 and
# 32x32x64 forms, one and several passes), the long-row GEMV and both prefill GEMMs.
@pytest.mark.parametrize("bad", ["nan", "inf", "-inf"])
@pytest.mark.parametrize("mode,M,N,K", [
    ("mxfp8", 1, 5120, 5120), ("nvfp4", 1, 5120, 5120), ("nvfp4", 1, 16400, 5120), ("nvfp4", 2, 4099, 5120),
    ("nvfp4", 3, 4099, 5120), ("mxfp8", 3, 4096, 5120), ("nvfp4", 1, 5120, 17408), ("nvfp4", 3, 5120, 17408),
    ("mxfp8", 1, 2048, 17408), ("mxfp8", 2, 5120, 17408), ("mxfp8", 300, 1000, 1024), ("nvfp4", 300, 1000, 1024)])
def test_non_finite_x_propagates_to_its_row(mode, M, N, K, bad):
    wq, s = _nf_weights(mode, N, K)
    xb = make_x(np.random.default_rng(4243), M, K, "normal")
    code = {"nan": 0x7FC0, "inf": 0x7F80, "-inf": 0xFF80}[bad]
    xb[0, 37] = code                      # one element of row 0
    if M > 1:
        xb[M - 1, K - 5] = code           # and one near the end of the last row
    y = run_qmm(mode, xb, wq, s)
    yf = f32(y)
    bad_rows = [0] + ([M - 1] if M > 1 else [])
    for m in bad_rows:
        if bad == "nan":
            assert np.isnan(yf[m]).all(), (m, int(np.isfinite(yf[m]).sum()))
        else:
            assert not np.isfinite(yf[m]).any(), (m, int(np.isfinite(yf[m]).sum()))
    good = [m for m in range(M) if m not in bad_rows]
    if good:
        cols = np.arange(0, N, 7)
        ref = O.qmm(mode, xb[good], wq, s, cols=cols)
        ok, fro, worst = O.check_tolerance(f32(y[good][:, cols]), f32(ref), **TOL)
        assert ok, (fro, worst)


def test_random_shapes_match_oracle():
    """40 seeded random (mode, M, N, K, x dtype) draws across every dispatch boundary (M in
    1..700, N in 1..6000, K any multiple of the mode's group up to 6144, x bf16 or f32),
    each against the oracle on a column sample.  A draw that fails names itself."""
    import torch

    rng = np.random.default_rng(20261202)
    draws = []
    for _ in range(40):
        mode = str(rng.choice(["mxfp8", "nvfp4"]))
        grp = 32 if mode == "mxfp8" else 16
        M = int(rng.choice([1, 2, 3, 4, 5, 7, 8, 9, 17, 64, 255, 256, 257, 700]))
        N = int(rng.integers(1, 6000))
        K = grp * int(rng.integers(1, 6144 // grp + 1))
        x_f32 = bool(rng.random() < 0.2)
        draws.append((mode, M, N, K, x_f32))
    for mode, M, N, K, x_f32 in draws:
        case = f"{mode} M={M} N={N} K={K} x_f32={x_f32}"
        print(f"[random] {case}", flush=True)
        wq, s = rand_w(rng, mode, N, K)
        xb = make_x(rng, M, K, "normal")
        xin = f32(xb) if x_f32 else xb
        y = run_qmm(mode, xin, wq, s, x_f32=x_f32)
        cols = np.unique(np.concatenate([np.arange(0, N, max(1, N // 97)), [N - 1]]))
        ref = O.qmm(mode, xb, wq, s, cols=cols, out="f32" if x_f32 else "bf16")
        got = y[:, cols] if x_f32 else f32(y[:, cols])
        want = ref if x_f32 else f32(ref)
        ok, fro, worst = O.check_tolerance(got.astype(np.float32), want.astype(np.float32), **TOL)
        assert ok, (case, fro, worst)
    torch.cuda.synchronize()


# Prefill shapes whose tiles fill rounds of the chip and part of another: M = 2000 (ragged
# against the 192- and 256-row tiles) and 2048 with N = 8448, 8348 (ragged) and 8704; one
# or two x tiles with very many of W (nvfp4 M = 100 and 200, N = 76800: 600 and 300 tiles).
@pytest.mark.parametrize("mode,M,N", [("mxfp8", 2000, 8448), ("mxfp8", 2048, 8704), ("nvfp4", 2000, 8348),
                                      ("nvfp4", 2048, 8704), ("nvfp4", 100, 76800), ("nvfp4", 200, 76800)])
def test_prefill_with_tail_tiles_in_one_launch(mode, M, N):
    K = 640
    rng = np.random.default_rng(M + N)
    wq, s = rand_w(rng, mode, N, K)
    xb = make_x(rng, M, K, "edge")
    y = run_qmm(mode, xb, wq, s)
    # every column of the last 640 (those of the last tiles), plus a sample of the rest
    cols = np.unique(np.concatenate([np.arange(N - 640, N), np.arange(0, N - 640, 37)]))
    rows = np.unique(np.concatenate([np.arange(0, M, 61), [M - 1]]))
    ref = O.qmm(mode, xb[rows], wq, s, cols=cols)
    ok, fro, worst = O.check_tolerance(f32(y[rows][:, cols]), f32(ref), **TOL)
    assert ok, (fro, worst)
    assert np.isfinite(f32(y)).all()


@pytest.mark.parametrize("mode", ["mxfp8", "nvfp4"])
def test_empty_and_one_dimensional_x(mode):
    """x with no rows ([0, K], [2, 0, K]) gives an empty result of the inferred shape and
    no error; a 1-D x [K] gives [N], the same values as x[None, :] (MLX's shape rules)."""
    rng = np.random.default_rng(77)
    N, K = 96, 512
    wq, s = rand_w(rng, mode, N, K)
    w = Q.Array.from_numpy(wq, Q.UINT32)
    sc = Q.Array.from_numpy(s, Q.UINT8)
    for shape in [(0, K), (2, 0, K)]:
        y = Q.quantized_matmul(Q.Array.from_numpy(np.zeros(shape, np.uint16), Q.BFLOAT16), w, sc, mode)
        assert tuple(y.shape) == shape[:-1] + (N,)
        assert y.numpy().size == 0
    x1 = make_x(rng, 1, K, "normal")[0]
    y1 = Q.quantized_matmul(Q.Array.from_numpy(x1, Q.BFLOAT16), w, sc, mode)
    assert tuple(y1.shape) == (N,)
    y2 = run_qmm(mode, x1[None, :], wq, s)
    assert np.array_equal(y1.numpy(), y2[0])
    assert Q.take_error() is None
