"""The small tiles (M > 32, few 128-row tiles) against the oracle: every form, the three operand types, ragged rows and columns,
a K that ends inside a 128-byte stage, fewer stages than wavefronts, K slices, gate/up pairs, every store; what lies around A
and C stays out of it; and the calls that stay with the tile kernels."""
import numpy as np
import pytest
import torch

import mm_amx_amd as mx
from gpu_util import check_float_parity, dev, dev_bf16, host_bits
from mm_amx_amd._lib import WORKSPACE_BYTES

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    mx.init(0)


def _in_nan(t, pad):
    """t inside a wider matrix of NaN (bf16) or 77 (int8): what lies behind a row must not enter the result."""
    wide = torch.full((t.shape[0], t.shape[1] + pad), float("nan") if t.dtype == torch.bfloat16 else 77, dtype=t.dtype, device="cuda")
    wide[:, :t.shape[1]] = t
    return wide[:, :t.shape[1]]


def _operands(po, kind, M, K, N):
    rng = np.random.default_rng(M + K + N)
    if kind == "i8":
        A, W = (rng.integers(-127, 128, shape).astype(np.int8) for shape in ((M, K), (K, N)))
        return dev(A), mx.repack_b(dev(W)), po.gemm_i8(A, W), {}, rng
    A = po.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
    if kind == "w8":
        W = rng.integers(-127, 128, (K, N)).astype(np.int8)
        return dev_bf16(A), mx.repack_b(dev(W)), po.gemm_bf16(A, po.f32_to_bf16(W.astype(np.float32))), {"b_dtype": mx.I8}, rng
    W = po.f32_to_bf16((rng.standard_normal((K, N)) * 0.05).astype(np.float32))
    return dev_bf16(A), mx.repack_b(dev_bf16(W)), po.gemm_bf16(A, W), {}, rng


# (bytes of K: whole stages and tails of 16 to 112 bytes, one stage to many; tiles with one live row or column in the last)
@pytest.mark.parametrize("M,kbytes,N,tile", [(33, 128, 33, "32x32"), (65, 144, 97, "32x32"), (64, 1024 + 112, 256, "32x32"), (40, 4096, 100, "32x32"),
                                             (97, 2048 + 64, 3201, "32x64"), (129, 2048, 2047, "32x64"), (250, 6000, 2150, "64x64"),
                                             (257, 9232, 3100, "64x64"), (250, 8192, 4124, "64x64")])
@pytest.mark.parametrize("kind", ["bf16", "w8", "i8"])
def test_products(po, kind, M, kbytes, N, tile):
    K = kbytes if kind == "i8" else kbytes // 2
    A, packed, ref, kw, rng = _operands(po, kind, M, K, N)
    pad = 16 + (-K) % 16
    n0, n1 = (32, N - 3) if N > 96 else (0, N)
    acc = torch.full((M, N), -7, dtype=torch.int32 if kind == "i8" else torch.float32, device="cuda")
    mx.gemm(_in_nan(A, pad), packed, N, mx.Epilogue(acc), n0=n0, n1=n1, k_splits=1, **kw)
    assert "wave_ring" in mx.last_kernel(), mx.last_kernel()
    if kind == "bf16":
        assert tile in mx.last_kernel(), mx.last_kernel()
    got = host_bits(acc)
    if kind == "i8":
        assert np.array_equal(got[:, n0:n1], ref[:, n0:n1]), mx.last_kernel()
    else:
        check_float_parity(got[:, n0:n1], ref[:, n0:n1], mx.last_kernel())
    assert np.all(got[:, :n0] == -7) and np.all(got[:, n1:] == -7)
    # the fused stores are the oracle's post-op on the GPU's own sums
    bias, deq, qs = (rng.standard_normal(N) * 0.1).astype(np.float32), rng.uniform(1e-3, 1e-2, N).astype(np.float32), rng.uniform(5, 40, N).astype(np.float32)
    opd = dict(bias=dev(bias), deq_scale_per_oc=dev(deq))
    opo = dict(bias=bias, deq_per_oc=deq)
    for dt, odt, steps, more_d, more_o in ((torch.float32, po.F32, 7, {}, {}), (torch.bfloat16, po.BF16, 3, {}, {}),
                                           (torch.int8, po.I8, 15, dict(q_scale_per_oc=dev(qs)), dict(q_per_oc=qs))):
        wide = torch.full((M, N + 5), 3, dtype=dt, device="cuda")
        mx.gemm(A, packed, N, mx.Epilogue(wide[:, :N], steps, **opd, **more_d), n0=n0, n1=n1, k_splits=1, **kw)
        out = host_bits(wide)
        assert np.array_equal(out[:, n0:n1], po.pp(got[:, n0:n1].copy(), steps, odt, **{k: v[n0:n1].copy() for k, v in (*opo.items(), *more_o.items())})), odt
        assert np.all(out[:, :n0] == out[0, -1]) and np.all(out[:, n1:] == out[0, -1])


@pytest.mark.parametrize("M,K,N,slices", [(40, 8192, 200, 4), (70, 5120, 1000, 2), (250, 8200, 500, 2), (60, 3080, 700, 4)])
@pytest.mark.parametrize("kind", ["bf16", "w8", "i8"])
def test_slices(po, kind, M, K, N, slices):
    """K cut over workgroups: the same bits on every run, counters back at zero, within the bar of the unsplit call."""
    if kind == "i8":
        K *= 2
    A, packed, ref, kw, rng = _operands(po, kind, M, K, N)
    ws = torch.zeros(WORKSPACE_BYTES, dtype=torch.uint8, device="cuda")
    outs = []
    for rep in range(3):
        acc = torch.zeros((M, N), dtype=torch.int32 if kind == "i8" else torch.float32, device="cuda")
        mx.gemm(A, packed, N, mx.Epilogue(acc), ws=ws, **kw)
        assert "wave_ring" in mx.last_kernel(), mx.last_kernel()
        if kind == "bf16":
            assert mx.last_kernel().endswith(f"_ksplit{slices}"), mx.last_kernel()
        outs.append(host_bits(acc))
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
    assert not ws[:16 << 10].any().item()
    if kind == "i8":
        assert np.array_equal(outs[0], ref)
    else:
        check_float_parity(outs[0], ref, mx.last_kernel())
    y = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
    bias = (rng.standard_normal(N) * 0.1).astype(np.float32)
    deq = np.float32(2.0 ** -8)
    mx.gemm(A, packed, N, mx.Epilogue(y, 7, bias=dev(bias), deq_scale=float(deq)), ws=ws, **kw)
    assert np.array_equal(host_bits(y), po.pp(outs[0], 7, po.BF16, bias=bias, deq=deq))
    # a workspace of the size that the query names holds the same slices
    need = mx.gemm_workspace_bytes(*{"bf16": (mx.BF16, mx.BF16), "w8": (mx.BF16, mx.I8), "i8": (mx.I8, mx.I8)}[kind], M, K, N)
    split = mx.last_kernel().partition("_ksplit")[1:]
    assert (need > 0) == (split[0] != ""), (need, split)
    if need:
        acc = torch.zeros_like(acc)
        mx.gemm(A, packed, N, mx.Epilogue(acc), ws=ws[:need], **kw)
        assert mx.last_kernel().partition("_ksplit")[1:] == split, (mx.last_kernel(), split)
        assert np.array_equal(host_bits(acc), outs[0])
    # without the slices' memory the call is not split
    mx.gemm(A, packed, N, mx.Epilogue(acc), ws=ws[:(16 << 10) + 256], **kw)
    assert "ksplit" not in mx.last_kernel(), mx.last_kernel()


def test_four_wavefronts_over_int8_weights(po):
    M, K, N = 700, 3080, 1537
    A, packed, ref, kw, rng = _operands(po, "w8", M, K, N)
    C = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    mx.gemm(A, packed, N, mx.Epilogue(C), k_splits=1, **kw)
    assert "64x64_wave_ring4w" in mx.last_kernel(), mx.last_kernel()
    check_float_parity(host_bits(C), ref, mx.last_kernel())


def test_slices_replay_from_a_hip_graph(po):
    M, K, N = 50, 8192, 320
    A, packed, ref, kw, rng = _operands(po, "bf16", M, K, N)
    A = A.clone()
    ws = torch.zeros(WORKSPACE_BYTES, dtype=torch.uint8, device="cuda")
    y = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    g, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        mx.gemm(A, packed, N, mx.Epilogue(y), ws=ws)
        side.synchronize()
        with torch.cuda.graph(g, stream=side):
            mx.gemm(A, packed, N, mx.Epilogue(y), ws=ws)
    assert "wave_ring" in mx.last_kernel() and "ksplit" in mx.last_kernel(), mx.last_kernel()
    torch.cuda.synchronize()
    for rep in range(4):
        A.copy_(torch.randn((M, K), device="cuda").to(torch.bfloat16))
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        got = host_bits(y).copy()
        y2 = torch.zeros_like(y)
        mx.gemm(A, packed, N, mx.Epilogue(y2), ws=ws)
        assert np.array_equal(got, host_bits(y2)), rep


@pytest.mark.parametrize("M,K,N,tile", [(40, 200, 96, "32x64"), (130, 1024, 2048, "64x64"), (250, 1032, 2048, "64x64"), (300, 1544, 2112, "64x64")])
@pytest.mark.parametrize("kind", ["bf16", "w8"])
def test_gate_up(po, kind, M, K, N, tile):
    rng = np.random.default_rng(K)
    x = po.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
    w = rng.integers(-7, 8, (2, N, K)).astype(np.float32)  # whole numbers: exact in both weight types
    g, u = (po.gemm_bf16(x, np.ascontiguousarray(po.f32_to_bf16(v).T)).astype(np.float64) * 2.0 ** -6 for v in w)
    both = np.concatenate([v[n:n + 32] for n in range(0, N, 32) for v in w])  # gate and up in turn, 32 columns each
    packed = mx.repack_b(dev_bf16(po.f32_to_bf16(both)), transpose=True) if kind == "bf16" else mx.repack_b(dev(both.astype(np.int8)), transpose=True)
    want = g / (1.0 + np.exp(-g)) * u
    for deq in (dict(deq_scale=2.0 ** -6), dict(deq_scale_per_oc=torch.full((2 * N,), 2.0 ** -6, device="cuda"))):
        h = torch.zeros((M, N), dtype=torch.float32, device="cuda")
        mx.gemm(_in_nan(dev_bf16(x), 8), packed, 2 * N, mx.Epilogue(h, mx.PP_SILU_GATE | mx.PP_DEQUANT, **deq), **({} if kind == "bf16" else {"b_dtype": mx.I8}))
        assert "wave_ring" in mx.last_kernel() and (kind == "w8" or tile in mx.last_kernel()), mx.last_kernel()
        got = host_bits(h).astype(np.float64)
        # silu is a 2^-14 approximation of g / (1 + exp(-g)); twice that for the roundings around it
        assert np.linalg.norm(got - want) <= 2.0 ** -13 * np.linalg.norm(want), mx.last_kernel()


def test_what_stays_with_the_tile_kernels(po):
    """Rows of A that are not whole aligned 16-byte pieces, a forced tile, a count of K slices, and products that fill the chip."""
    A, packed, ref, kw, rng = _operands(po, "bf16", 64, 1024, 256)
    C = torch.zeros((64, 256), dtype=torch.float32, device="cuda")
    mx.gemm(A, packed, 256, mx.Epilogue(C))
    assert "wave_ring" in mx.last_kernel()
    mx.gemm(_in_nan(A, 3), packed, 256, mx.Epilogue(C))
    assert "masked" in mx.last_kernel(), mx.last_kernel()
    mx.gemm(A, packed, 256, mx.Epilogue(C), k_splits=2)
    assert "wave_ring" not in mx.last_kernel() and mx.last_kernel().endswith("ksplit2"), mx.last_kernel()
    try:
        mx.set_tile("128x64")
        mx.gemm(A, packed, 256, mx.Epilogue(C))
        assert "128x64_ring" in mx.last_kernel(), mx.last_kernel()
    finally:
        mx.set_tile("")
    x = torch.randn((1024, 4096), device="cuda").to(torch.bfloat16)
    big = mx.repack_b((torch.randn((4096, 11008), device="cuda") * 0.02).to(torch.bfloat16))
    mx.gemm(x, big, 11008, mx.Epilogue(torch.zeros((1024, 11008), dtype=torch.bfloat16, device="cuda")))
    assert "wave_ring" not in mx.last_kernel(), mx.last_kernel()


@pytest.mark.parametrize("kind,M,K,N", [("w8", 895, 9760, 1792), ("w8", 678, 7680, 2016), ("bf16", 517, 4280, 1120), ("bf16", 889, 4928, 640)])
def test_deep_products_whose_tiles_split_k_stay_with_the_tile_kernels(kind, M, K, N):
    """The margin that a K split has to win by among the tile kernels is no part of their time: with it these went to the small
    tiles, 9 to 23 % slower."""
    packed = mx.repack_b(torch.zeros((K, N), dtype=torch.int8 if kind == "w8" else torch.bfloat16, device="cuda"))
    A, C = torch.zeros((M, K), dtype=torch.bfloat16, device="cuda"), torch.empty((M, N), device="cuda")
    mx.workspace()
    mx.gemm(A, packed, N, mx.Epilogue(C), **({"b_dtype": mx.I8} if kind == "w8" else {}))
    assert "wave_ring" not in mx.last_kernel() and "ksplit" in mx.last_kernel(), mx.last_kernel()
