"""Weight preparation kernels against the oracle at the edges of their units: 32 rows x 128 bytes (rows of B^T), 8 squares
of 8 x 8 bf16 or 16 x 16 bytes (rows of B)."""
import numpy as np
import pytest
import torch

import mm_amx_amd as mx
from gpu_util import call_us, dev, dev_bf16, host_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    mx.init(0)


@pytest.mark.parametrize("dt", ["bf16", "int8", "uint8"])
@pytest.mark.parametrize("K", [1, 2, 3, 7, 9, 15, 16, 63, 64, 65, 128, 511, 1025])
@pytest.mark.parametrize("N", [1, 2, 3, 5, 7, 8, 9, 15, 17, 31, 64, 129, 257])
def test_repack_unit_edges(po, dt, K, N):
    rng = np.random.default_rng(K * 1000 + N)
    if dt == "bf16":
        B, up = rng.integers(1, 65536, (K, N)).astype(np.uint16), dev_bf16
        want = po.repack(B, layout="mfma")
    else:
        B, up = rng.integers(-128, 128, (K, N)).astype(np.int8), dev
        want = po.repack(B, layout="mfma")
        if dt == "uint8":  # stored as u - 128
            B = (B.astype(np.int16) + 128).astype(np.uint8)
    assert np.array_equal(host_bits(mx.repack_b(up(B))).view(np.uint8), want.view(np.uint8))
    # rows that start at any multiple of the element, inside a wider matrix
    wide = torch.zeros((N, K + 3), dtype=up(B).dtype, device="cuda")
    wide[:, 1:K + 1] = up(np.ascontiguousarray(B.T))
    assert np.array_equal(host_bits(mx.repack_b(wide[:, 1:K + 1], transpose=True)).view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (5, 64), (33, 1029), (2, 70001), (700, 8), (4100, 9), (1025, 130),
                                       (70, 8193), (5, 32767), (5, 32768), (9, 2048)])
@pytest.mark.parametrize("gap", [0, 5])
def test_quantisers_row_ends_and_gaps(po, rows, cols, gap):
    """Rows that end in the middle of a 16-byte load, with and without a gap behind them; the largest weight last."""
    rng = np.random.default_rng(rows * 7 + cols)
    W = po.f32_to_bf16((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    W[-1, -1] = po.f32_to_bf16(np.array([-3.0], np.float32))[0]
    wide = torch.full((rows, cols + gap), float("nan"), dtype=torch.bfloat16, device="cuda")  # (a gap takes no part)
    wide[:, :cols] = dev_bf16(W)
    got, scales = mx.quantize_weights(wide[:, :cols])
    want, dq, q = po.quantize_weights(W)
    assert np.array_equal(host_bits(got), want)
    assert host_bits(scales).tolist() == [np.float32(q), np.float32(dq)]
    assert np.array_equal(host_bits(mx.quantize_weights_scaled(wide[:, :cols], 1234.5)), po.quantize_scale_trunc(W, 1234.5))


@pytest.mark.parametrize("K", [1, 15, 16, 127, 128, 129, 300])
@pytest.mark.parametrize("N", [1, 7, 8, 9, 31, 33, 64, 65, 130])
def test_scaled_pack_is_quantised_then_packed(po, K, N):
    """One pass over W against the two it stands for, at the edges of its units (64 columns x 128 of k), rows of any alignment."""
    rng = np.random.default_rng(K * 1000 + N)
    W = rng.integers(0, 65536, (K, N)).astype(np.uint16)  # any weight: infinite, NaN and denormal ones among them
    wide = torch.full((K, N + 3), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[:, 1:N + 1] = dev_bf16(W)
    for scale in (30.0, 0.0, float("inf")):
        want = po.repack(po.quantize_scale_trunc(W, scale), layout="mfma")
        for B in (dev_bf16(W), wide[:, 1:N + 1]):
            assert np.array_equal(host_bits(mx._lib.quantize_pack_scaled(B, scale)).view(np.uint8), want.view(np.uint8))


def test_scaled_pack_of_every_bf16(po):
    W = np.arange(65536).astype(np.uint16).reshape(512, 128)
    for scale in (1.0, 127.0, 1e-3, 1e30, -2.5):
        want = po.repack(po.quantize_scale_trunc(W, scale), layout="mfma")
        assert np.array_equal(host_bits(mx.repackB_1xL(dev_bf16(W), torch.int8, 2, scale)).view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("rows,cols", [(1, 1), (300, 100), (4096, 1024), (70, 8193)])
def test_quantisers_scratch_of_one_word(po, rows, cols):
    """mmx_quantize_weights with the one word that its signature promises, filled with ones before the call."""
    L, C = mx._lib, mx._lib.C
    W = po.f32_to_bf16((np.random.default_rng(rows).standard_normal((rows, cols)) * 0.02).astype(np.float32))
    Wd, got = dev_bf16(W), torch.empty((rows, cols), dtype=torch.int8, device="cuda")
    scales, word = torch.empty(2, device="cuda"), torch.full((3,), -1, dtype=torch.int32, device="cuda")
    assert L.lib().mmx_quantize_weights(Wd.data_ptr(), cols * 2, rows, cols, got.data_ptr(), cols, scales.data_ptr(), word.data_ptr() + 4, L._stream()) == 0
    want, dq, q = po.quantize_weights(W)
    assert np.array_equal(host_bits(got), want) and host_bits(scales).tolist() == [np.float32(q), np.float32(dq)]
    assert host_bits(word)[[0, 2]].tolist() == [-1, -1]


@pytest.mark.parametrize("rows,cols", [(1000000, 8), (131072, 128), (16384, 1024)])
def test_gaps_between_short_rows_cost_little(rows, cols):
    """With a gap as long as the row up to twice the lines are read.  A workgroup to a row took 25 times as long as without
    gaps at 131072 x 128 and 250 times at 1000000 x 8; with the rows shared out it is less than twice."""
    W = torch.randn((rows, 2 * cols), device="cuda").to(torch.bfloat16)
    for f in (mx.quantize_weights, lambda w: mx.quantize_weights_scaled(w, 30.0)):
        whole, gaps = W[:, :cols].contiguous(), W[:, :cols]
        assert call_us(lambda: f(gaps)) <= 6 * call_us(lambda: f(whole))


@pytest.mark.parametrize("K", [1, 64, 65, 129, 255, 256, 257, 513, 2056])
@pytest.mark.parametrize("N", [1, 33, 96])
def test_int4_pack_unit_edges(po, K, N):
    rng = np.random.default_rng(K * 31 + N)
    W = po.f32_to_bf16((rng.standard_normal((K, N)) * 0.02).astype(np.float32))
    W[:, N // 2] = 0  # (a column without a scale)
    W[K - 1, N - 1] = po.f32_to_bf16(np.array([0.5], np.float32))[0]  # (a largest weight in the last row and column)
    q, deq = po.quantize_int4(W)
    want = po.pack_int4(q)
    for W_, trans in ((W, False), (np.ascontiguousarray(W.T), True)):
        wide = torch.full((W_.shape[0], W_.shape[1] + 3), float("nan"), dtype=torch.bfloat16, device="cuda")
        wide[:, 1:1 + W_.shape[1]] = dev_bf16(W_)
        packed, d = mx.quantize_pack_int4(wide[:, 1:1 + W_.shape[1]], transpose=trans)
        assert np.array_equal(host_bits(packed), np.ascontiguousarray(want).view(np.uint8).reshape(-1))
        assert np.array_equal(host_bits(d), deq)


@pytest.mark.parametrize("K", [32, 128])
def test_int4_pack_of_a_short_k_costs_no_more_than_its_bytes(K):
    """K = 32 and 128 move 0.15 and 0.3 of the bytes of K = 512 (the packed form pads K to 256).  With sixteen wavefronts to
    every panel they took 0.53 to 0.77 of its time, with the panel held in registers 0.15 to 0.27."""
    N = 1 << 17
    long, short = (torch.randn((N, k), device="cuda").to(torch.bfloat16) for k in (512, K))
    for trans in (True, False):
        a, b = (long, short) if trans else (long.t().contiguous(), short.t().contiguous())
        assert call_us(lambda: mx.quantize_pack_int4(b, transpose=trans)) <= 0.45 * call_us(lambda: mx.quantize_pack_int4(a, transpose=trans))


def test_rows_that_end_inside_16_bytes_are_one_trip_to_memory():
    """Bytes from [K, N], a square of 16 x 16 per lane: fetched element by element at the end of a row they took 3 times as
    long at N = 3001 as at N = 3008."""
    took = {}
    for N in (3001, 3008):
        B = torch.randint(-128, 128, (512, N), device="cuda", dtype=torch.int8)
        out = torch.empty(mx.packed_b_bytes(mx.I8, 512, N), dtype=torch.uint8, device="cuda")
        call = (mx.I8, B.data_ptr(), N, 512, N, 0, out.data_ptr(), torch.cuda.current_stream().cuda_stream)
        took[N] = call_us(lambda: mx.lib().mmx_repack_b(*call), n=50)
    assert took[3001] <= 1.7 * took[3008], took


@pytest.mark.parametrize("K", [257, 2048, 2049, 4096, 4100, 8192, 8191, 8200, 12288, 12289])
@pytest.mark.parametrize("N", [1, 8, 41])
def test_int4_weights_read_once(po, K, N):
    """[N, K] held in registers, 2, 4, 8 or 12 fragments a wavefront, and the first K that is not: rows at any address, columns that
    do not fill a group, infinities, NaN and a column of zeros."""
    rng = np.random.default_rng(K + N)
    W = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    W[K - 1, N - 1] = 3.0  # (the largest of its column in the last place)
    if N > 8:
        W[:, 2], W[5, 3], W[K - 2, 4] = 0.0, np.inf, np.nan
    W = po.f32_to_bf16(W)
    q, deq = po.quantize_int4(W)
    wide = torch.full((N + 1, K + 3), float("nan"), dtype=torch.bfloat16, device="cuda")
    Wt = wide[1:, 1:K + 1]
    Wt.copy_(dev_bf16(np.ascontiguousarray(W.T)))
    packed, deq_gpu = mx.quantize_pack_int4(Wt, transpose=True)
    assert np.array_equal(host_bits(deq_gpu).view(np.uint32), deq.view(np.uint32))
    assert np.array_equal(host_bits(packed), po.pack_int4(q))


@pytest.mark.parametrize("K", [12290, 12295, 12296, 12297, 14336, 14337, 14343, 14344, 16383])
@pytest.mark.parametrize("N", [1, 33])
def test_int4_weights_of_a_deep_k(po, K, N):
    """[N, K] that is read twice (K > 12288): rows that end anywhere in a lane's 16 bytes and in a lane's four loads, a largest weight at
    their end, infinities around them that take no part."""
    rng = np.random.default_rng(K + N)
    W = (rng.standard_normal((K, N)) * 0.05).astype(np.float32)
    W[K - 1 - np.arange(N) % 9, np.arange(N)] = 2.0 + np.arange(N)
    W = po.f32_to_bf16(W)
    q, deq = po.quantize_int4(W)
    wide = torch.full((N + 2, K + 3), float("inf"), dtype=torch.bfloat16, device="cuda")
    Wt = wide[1:N + 1, 1:K + 1]
    Wt.copy_(dev_bf16(np.ascontiguousarray(W.T)))
    packed, deq_gpu = mx.quantize_pack_int4(Wt, transpose=True)
    assert np.array_equal(host_bits(deq_gpu).view(np.uint32), deq.view(np.uint32))
    assert np.array_equal(host_bits(packed), po.pack_int4(q))


@pytest.mark.parametrize("gap", [0, 5])
@pytest.mark.parametrize("rows,cols", [(1, 1), (300, 100), (4096, 1024), (70, 8193), (5, 40000), (3000, 2500)])
def test_quantisers_scratch_of_4_kib(po, rows, cols, gap):
    """A word for every workgroup of the maxima, filled with ones before the call (a NaN, the largest pattern of all, were it read), and
    the words on both sides of it."""
    L, n = mx._lib, mx._lib.QUANTIZE_SCRATCH_BYTES // 4
    W = po.f32_to_bf16((np.random.default_rng(rows).standard_normal((rows, cols)) * 0.02).astype(np.float32))
    wide = torch.full((rows, cols + gap), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[:, :cols] = dev_bf16(W)
    got = torch.empty((rows, cols), dtype=torch.int8, device="cuda")
    scales, words = torch.empty(2, device="cuda"), torch.full((n + 2,), -1, dtype=torch.int32, device="cuda")
    assert L.lib().mmx_quantize_weights_scratch(wide.data_ptr(), (cols + gap) * 2, rows, cols, got.data_ptr(), cols, scales.data_ptr(),
                                                words.data_ptr() + 4, 4 * n, L._stream()) == 0
    want, dq, q = po.quantize_weights(W)
    assert np.array_equal(host_bits(got), want) and host_bits(scales).tolist() == [np.float32(q), np.float32(dq)]
    assert host_bits(words)[[0, n + 1]].tolist() == [-1, -1]
