"""The decode kernels (M <= 32) at a K that ends inside the last fragments of the packed weights, and with rows of x of any
length and alignment, against the oracle: every form that stages x (streaming, half panels, chunks with and without a K
split, two panels at a time, gate/up pairs), remainders of 1 element to one less than a fragment; and that the general
kernel is what ran for short rows that are aligned, and there alone."""
import numpy as np
import pytest
import torch

import mm_amx_amd as mx
from gpu_util import check_float_parity, dev, dev_bf16, host_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    mx.init(0)


def _in_nan(t, pad):
    """t inside a wider matrix of NaN (bf16) or 77 (int8): what lies behind a row must not enter the result."""
    wide = torch.full((t.shape[0], t.shape[1] + pad), float("nan") if t.dtype == torch.bfloat16 else 77, dtype=t.dtype, device="cuda")
    wide[:, :t.shape[1]] = t
    return wide[:, :t.shape[1]]


def _operands(po, kind, M, K, N, seed):
    """x, the packed weights and the exact product's oracle (int4: of the quantised values, before the scales)."""
    rng = np.random.default_rng(seed)
    x = rng.integers(-127, 128, (M, K)).astype(np.int8) if kind == "i8" else po.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
    if kind in ("w8", "i8"):
        W = rng.integers(-127, 128, (K, N)).astype(np.int8)
        return x, mx.repack_b(dev(W)), (po.gemm_i8(x, W) if kind == "i8" else po.gemm_bf16(x, po.f32_to_bf16(W.astype(np.float32))))
    W = po.f32_to_bf16((rng.standard_normal((K, N)) * 0.05).astype(np.float32))
    if kind == "bf16":
        return x, mx.repack_b(dev_bf16(W)), po.gemm_bf16(x, W)
    q, deq = po.quantize_int4(W)
    return x, mx.quantize_pack_int4(dev_bf16(W))[0], po.gemv_w8(x, q, deq, want_acc=True)[1]


KW = {"bf16": {}, "w8": {"b_dtype": mx.I8}, "w4": {"b_dtype": mx.I4}, "i8": {}}


def _short_tail(kind, M, K, stride):
    """Aligned rows of x with a K so short that the general kernel is the faster one (up to 256 panels, no gate/up pairs)."""
    k, group, few, many = {"bf16": (16, 64, 24, 20), "w8": (32, 128, 32 if M <= 8 else 24, 16), "w4": (64, 256, 10, 8)}[kind]
    return (2 * (K if M == 1 else stride)) % 16 == 0 and K % group != 0 and -(-K // k) <= (few if M <= 16 else many)


@pytest.mark.parametrize("M", [1, 4, 7, 32])
@pytest.mark.parametrize("K", [8, 9, 15, 17, 63, 65, 96, 190, 1000, 1088, 1337])
@pytest.mark.parametrize("kind", ["bf16", "w8", "w4", "i8"])
def test_x_in_lds(po, kind, K, M):
    """Short x: the streaming kernel, with every alignment of the rows, and the general one where it is the faster one."""
    if kind == "i8":
        K = (K + 15) // 16 * 16   # (rows that are not whole 16-byte pieces go to the tile kernels)
    N = 100
    x, packed, ref = _operands(po, kind, M, K, N, K + M)
    es = 1 if kind == "i8" else 2
    for pad in ((-K * es % 16) // es + 16 // es, 0, 3):
        C = torch.zeros((M, N), dtype=torch.int32 if kind == "i8" else torch.float32, device="cuda")
        mx.gemm(_in_nan((dev if kind == "i8" else dev_bf16)(x), pad), packed, N, mx.Epilogue(C), **KW[kind])
        if kind != "i8" and _short_tail(kind, M, K, K + pad):
            assert mx.last_kernel() == f"skinny_{kind}", mx.last_kernel()
        elif kind != "i8" or pad != 3 or M == 1:
            if (M + 1) * K * es <= 40000:
                assert mx.last_kernel().startswith(f"skinny_stream_{kind}"), mx.last_kernel()
            assert mx.last_kernel() not in ("skinny_bf16", "skinny_w8", "skinny_w4")
        if kind == "i8":
            assert np.array_equal(host_bits(C), ref), mx.last_kernel()
        else:
            check_float_parity(host_bits(C), ref, f"{kind} {M}x{K} pad={pad} {mx.last_kernel()}")


@pytest.mark.parametrize("kind,M,K,N,splits,want", [
    ("bf16", 3, 2600, 1000, 0, "skinny_half_bf16"),       # half panels: an odd number of fragments (163)
    ("w8", 1, 10450, 1000, 1, "skinny_half_w8"),          # (327)
    ("bf16", 12, 3680, 160, 1, "skinny_chunk_bf16"),      # chunks, two fragments per wavefront
    ("bf16", 30, 3681, 160, 1, "skinny_chunk_bf16"),
    ("bf16", 20, 7476, 1007, 0, "skinny_chunk_bf16_ksplit"),
    ("bf16", 21, 2500, 8300, 0, "skinny_chunk_bf16_2p"),
    ("w8", 16, 4160, 8300, 0, "skinny_chunk_w8"),
    ("w8", 32, 4190, 700, 0, "skinny_chunk_w8_ksplit"),
    ("w8", 24, 2611, 8300, 0, "skinny_chunk_w8_2p"),
    ("w4", 11, 5313, 300, 0, "skinny_chunk_w4_ksplit"),
    ("w4", 29, 1800, 300, 1, "skinny_chunk_w4"),
    ("w4", 9, 6850, 8300, 1, "skinny_chunk_w4"),
])
def test_x_through_lds_in_chunks_and_half_panels(po, kind, M, K, N, splits, want):
    x, packed, ref = _operands(po, kind, M, K, N, K)
    for pad in ((-K % 8) + 8, 1):
        C = torch.zeros((M, N), dtype=torch.float32, device="cuda")
        mx.gemm(_in_nan(dev_bf16(x), pad), packed, N, mx.Epilogue(C), k_splits=splits, **KW[kind])
        assert mx.last_kernel().startswith(want), mx.last_kernel()
        check_float_parity(host_bits(C), ref, f"{kind} {M}x{K}x{N} pad={pad} {mx.last_kernel()}")


# The largest x that each rule takes, the next larger one, few and many panels, K that fills its fragments and not.  stream: whether the
# streaming kernel is the faster one, WHOLE: over rows that are whole aligned 16-byte pieces only (over others, chunked and streaming, us:
# bf16 31 x 2301 x 4032 9.1 / 12.4, int8 weights 14 x 4861 x 3680 9.7 / 12.9).
WHOLE = "whole rows"


@pytest.mark.parametrize("kind,M,K,N,stream", [
    ("bf16", 32, 2400, 4800, WHOLE), ("bf16", 32, 2424, 4800, False), ("bf16", 24, 1990, 2900, False), ("bf16", 24, 2624, 2900, False),
    ("bf16", 16, 4544, 8192, WHOLE), ("w8", 16, 4544, 4807, WHOLE), ("w8", 31, 2450, 2900, False), ("w8", 31, 2496, 2900, False), ("w8", 8, 7360, 1280, False),
    ("w4", 13, 5632, 4800, WHOLE), ("w4", 8, 5100, 4800, True), ("w4", 8, 5056, 4800, False), ("w4", 4, 6913, 2900, True), ("w4", 5, 6913, 2900, False),
    ("w4", 4, 8192, 8300, True), ("w4", 3, 6000, 8300, False),
    # (int4 shares of 9 to 21 fragments: every batch of the rolling window, with repeats and without)
    ("w4", 2, 4417, 100, True), ("w4", 1, 5120, 100, True), ("w4", 1, 5700, 100, True), ("w4", 1, 6300, 100, True), ("w4", 1, 7168, 100, True),
    ("w4", 1, 7681, 100, True), ("w4", 1, 8705, 100, True), ("w4", 1, 9984, 100, True), ("w4", 1, 10689, 100, True),
    ("i8", 32, 4096, 4800, True), ("i8", 32, 4864, 4800, False), ("i8", 16, 4608, 1280, False), ("i8", 24, 2048, 8300, False),
    # (rows that are not whole pieces: up to 10, panels for up to 3/4 of the CUs)
    ("bf16", 10, 5005, 6100, True), ("bf16", 11, 5005, 6100, False), ("bf16", 10, 5005, 6150, False), ("w8", 9, 5853, 6100, True), ("w4", 11, 5101, 6300, False),
    # (slices for up to half of the CUs)
    ("bf16", 25, 2112, 2900, WHOLE), ("bf16", 27, 2432, 2900, False), ("bf16", 30, 1536, 2900, False), ("w8", 12, 4480, 2900, WHOLE), ("w8", 12, 4528, 2900, False),
    ("w8", 13, 3840, 2900, False), ("w8", 4, 10944, 2900, False), ("i8", 22, 4352, 2900, True), ("i8", 26, 4864, 2900, False), ("i8", 6, 10240, 2900, True),
    ("i8", 13, 10496, 2900, False),
    # (and for more; panels for nearly all CUs)
    ("w8", 4, 9728, 4128, WHOLE), ("w8", 3, 10496, 4128, False), ("bf16", 6, 8064, 8000, False), ("w8", 15, 4352, 8064, False), ("w8", 15, 4608, 8064, WHOLE)])
def test_long_x_in_lds(po, kind, M, K, N, stream):
    x, packed, ref = _operands(po, kind, M, K, N, K + M)
    es = 1 if kind == "i8" else 2
    for pad in ((8, 1) if kind != "i8" else (16, 0)):
        C = torch.zeros((M, N), dtype=torch.int32 if kind == "i8" else torch.float32, device="cuda")
        pad += -K % 8 if pad == 8 else 0
        mx.gemm(_in_nan((dev if kind == "i8" else dev_bf16)(x), pad), packed, N, mx.Epilogue(C), **KW[kind])
        streams = (K * es % 16 == 0 and pad != 1) if stream is WHOLE else stream
        assert mx.last_kernel().startswith((f"skinny_stream_{kind}",) if streams else (f"skinny_chunk_{kind}", f"skinny_direct_{kind}")), mx.last_kernel()
        if kind == "i8":
            assert np.array_equal(host_bits(C), ref), mx.last_kernel()
        else:
            check_float_parity(host_bits(C), ref, f"{kind} {M}x{K}x{N} pad={pad} {mx.last_kernel()}")


@pytest.mark.parametrize("M,K", [(3, 200), (2, 2104), (16, 2104), (32, 1001)])
@pytest.mark.parametrize("kind", ["bf16", "w8", "w4"])
def test_gate_up(po, kind, M, K):
    N = 96
    rng = np.random.default_rng(K)
    x = po.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
    w = rng.integers(-7, 8, (2, N, K)).astype(np.float32)  # whole numbers: exact in all three weight types, int4's scale is 1
    w[:, :, 0] = 7.0
    g, u = (po.gemm_bf16(x, np.ascontiguousarray(po.f32_to_bf16(v).T)).astype(np.float64) * 2.0 ** -6 for v in w)
    both = np.concatenate([v[n:n + 32] for n in range(0, N, 32) for v in w])  # gate and up in turn, 32 columns each
    packed = {"bf16": lambda: mx.repack_b(dev_bf16(po.f32_to_bf16(both)), transpose=True), "w8": lambda: mx.repack_b(dev(both.astype(np.int8)), transpose=True),
              "w4": lambda: mx.quantize_pack_int4(dev_bf16(po.f32_to_bf16(both)), transpose=True)[0]}[kind]()
    h = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    mx.gemm(_in_nan(dev_bf16(x), 5), packed, 2 * N, mx.Epilogue(h, mx.PP_SILU_GATE | mx.PP_DEQUANT, deq_scale=2.0 ** -6), **KW[kind])
    assert "gateup" in mx.last_kernel(), mx.last_kernel()
    # silu is a 2^-14 approximation of g / (1 + exp(-g)); twice that for the roundings around it
    want, got = g / (1.0 + np.exp(-g)) * u, host_bits(h).astype(np.float64)
    assert np.linalg.norm(got - want) <= 2.0 ** -13 * np.linalg.norm(want), mx.last_kernel()


# The largest x with one workgroup on a CU and the next one; x that LDS holds twice; K that fills the batches, its fragments, and neither;
# more panels than CUs, where panels 128 KiB apart (K 1985 to 2048) are the chunked kernel's (16 x 2048 x 2 7328 13.1 / 15.2 us)
@pytest.mark.parametrize("M,K,N,stream", [(28, 1344, 96, True), (17, 1001, 96, True), (32, 2400, 96, True), (32, 2424, 96, False), (16, 4096, 4096, True),
                                          (16, 4096, 4160, False), (4, 7000, 96, True), (9, 2049, 8192, True), (12, 2049, 8192, False), (9, 2688, 8224, False), (18, 2304, 8192, WHOLE),
                                          (16, 2304, 6816, WHOLE), (16, 2304, 6848, False), (20, 2048, 4608, False), (20, 1990, 4608, False),
                                          (20, 1984, 4608, WHOLE), (20, 2048, 4096, True)])
def test_gate_up_over_a_long_x(M, K, N, stream):
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn((M, K), device="cuda", generator=g).to(torch.bfloat16)
    w = (torch.randn((2, N, K), device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    packed = mx.repack_gate_up(w[0], w[1])
    a, b = (x.double() @ v.double().t() for v in w)
    for pad in (-K % 8 + 8, 5):
        h = torch.zeros((M, N), dtype=torch.float32, device="cuda")
        mx.gemm(_in_nan(x, pad), packed, 2 * N, mx.Epilogue(h, mx.PP_SILU_GATE))
        streams = (K % 8 == 0 and pad != 5) if stream is WHOLE else stream
        assert mx.last_kernel() == f"skinny_{'stream' if streams else 'chunk'}_bf16_gateup", mx.last_kernel()
        want = a / (1.0 + torch.exp(-a)) * b  # silu within 2^-14, and twice that for the roundings around it
        assert (h.double() - want).norm() <= 2.0 ** -13 * want.norm(), mx.last_kernel()


@pytest.mark.parametrize("kind,M,K,N,splits,want", [
    ("bf16", 12, 2600, 64, 0, "skinny_stream_bf16"),
    ("w8", 12, 2600, 64, 0, "skinny_stream_w8"),
    ("w4", 7, 2600, 64, 0, "skinny_stream_w4"),
    ("bf16", 24, 2600, 64, 1, "skinny_chunk_bf16"),      # rows that end between two pieces of 16 bytes
    ("w8", 20, 2612, 64, 1, "skinny_chunk_w8"),
    ("w4", 12, 2600, 64, 1, "skinny_chunk_w4"),
    ("bf16", 24, 2624, 64, 1, "skinny_chunk_bf16"),      # rows that end between two fragments of a chunk
    ("bf16", 12, 3712, 64, 1, "skinny_chunk_bf16"),      # (two fragments of a panel per wavefront)
    ("bf16", 32, 4160, 1000, 0, "skinny_chunk_bf16_ksplit"),
    ("bf16", 24, 2624, 8300, 0, "skinny_chunk_bf16_2p"),
    ("w8", 32, 4224, 1000, 1, "skinny_chunk_w8"),
    ("w8", 12, 4224, 1000, 0, "skinny_chunk_w8_ksplit"),
    ("w8", 32, 4224, 8300, 0, "skinny_chunk_w8_2p"),
    ("w4", 16, 2304, 64, 1, "skinny_chunk_w4"),
    ("w4", 32, 2304, 64, 1, "skinny_chunk_w4"),
    ("bf16", 6, 11072, 8300, 0, "skinny_direct_bf16"),
])
def test_infinite_x_at_the_end_of_k(kind, M, K, N, splits, want):
    """The end of a row that a load repeats behind it is not multiplied again: an infinite last element gives infinities, no NaN."""
    x = torch.ones((M, K), dtype=torch.bfloat16, device="cuda")
    x[:, K - 1] = float("inf")
    W = torch.ones((K, N), dtype=torch.bfloat16, device="cuda")
    packed = {"bf16": lambda: mx.repack_b(W), "w8": lambda: mx.repack_b(W.to(torch.int8)), "w4": lambda: mx.quantize_pack_int4(W)[0]}[kind]()
    C = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    mx.gemm(x, packed, N, mx.Epilogue(C), k_splits=splits, **KW[kind])
    assert mx.last_kernel().startswith(want), mx.last_kernel()
    assert torch.isinf(C).all(), mx.last_kernel()


@pytest.mark.parametrize("M,K,N,splits,want", [
    (12, 2600, 64, 0, "skinny_stream_bf16"),        # fragments that a wavefront's batch repeats behind the end of K
    (12, 2624, 64, 0, "skinny_stream_bf16"),        # (whole 128-byte groups of K)
    (2, 1000, 64, 1, "skinny_stream_bf16"),
    (3, 2600, 1000, 0, "skinny_half_bf16"),
    (3, 2624, 1000, 0, "skinny_half_bf16"),
    (30, 3681, 160, 1, "skinny_chunk_bf16"),
    (24, 2624, 160, 0, "skinny_chunk_bf16_ksplit"),
    (6, 11072, 8300, 0, "skinny_direct_bf16"),
])
def test_infinite_weights_at_the_end_of_k(M, K, N, splits, want):
    """What a load repeats behind the end of K is not multiplied: infinite weights in the last row of B give infinities, no NaN."""
    W = torch.ones((K, N), dtype=torch.bfloat16, device="cuda")
    W[K - 1] = float("inf")
    C = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    mx.gemm(torch.ones((M, K), dtype=torch.bfloat16, device="cuda"), mx.repack_b(W), N, mx.Epilogue(C), k_splits=splits)
    assert mx.last_kernel().startswith(want), mx.last_kernel()
    assert torch.isinf(C).all(), mx.last_kernel()


def test_int8_with_a_count_of_slices_is_refused_as_ever(po):
    """A forced K split belongs to the tile kernels, which refuse it at such a K; the call without one takes the decode kernels."""
    M, K, N = 8, 2112, 256
    x, packed, ref = _operands(po, "i8", M, K, N, 1)
    C = torch.zeros((M, N), dtype=torch.int32, device="cuda")
    with pytest.raises(mx.MmxError, match="K a multiple of 128 bytes"):
        mx.gemm(dev(x), packed, N, mx.Epilogue(C), k_splits=2)
    mx.gemm(dev(x), packed, N, mx.Epilogue(C))
    assert mx.last_kernel() == "skinny_stream_i8", mx.last_kernel()
    assert np.array_equal(host_bits(C), ref)


@pytest.mark.parametrize("M,K,want", [(6, 1000, "skinny_stream_bf16_gateup"), (6, 1408, "skinny_stream_bf16_gateup"), (3, 3200, "skinny_half_bf16_gateup")])
def test_infinite_weights_at_the_end_of_k_of_gate_up_pairs(M, K, want):
    """As above for pairs: infinite weights of `up` in the last column, behind a finite gate."""
    N = 64
    gate, up = (torch.ones((N, K), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    up[:, K - 1] = float("inf")
    C = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    x = torch.full((M, K), 2.0 ** -12, dtype=torch.bfloat16, device="cuda")
    mx.gemm(x, mx.repack_gate_up(gate, up), 2 * N, mx.Epilogue(C, mx.PP_SILU_GATE))
    assert mx.last_kernel().startswith(want), mx.last_kernel()
    assert torch.isinf(C).all(), mx.last_kernel()
