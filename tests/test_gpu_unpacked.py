"""Matmul with a second operand that is used once (constB = False): read where it lies, without packing.  Operands are small
integers, so that every order of fp32 summation gives the same sums and results have to equal the packed form's, and the
64-bit product, exactly."""
import ctypes

import pytest
import torch

import mm_amx_amd as mx
from gpu_util import call_us
from mm_amx_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    mx.init(0)


def _ints(shape, seed, pad=0):
    """Integers of [-8, 8] as bf16, inside a wider matrix of NaN when pad > 0 (rows of any alignment)."""
    t = torch.randint(-8, 9, shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).cuda()
    if not pad:
        return t
    wide = torch.full((shape[0] + 1, shape[1] + pad), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[:-1, pad // 2:pad // 2 + shape[1]] = t
    return wide[:-1, pad // 2:pad // 2 + shape[1]]


def _run(const, trans, A, B, C, **kw):
    pp = mx.BiasGeluStore(C, kw.get("steps", mx.Steps.NONE), kw.get("bias"))
    if "q" in kw:
        pp.set_q_scale(kw["q"])
    mx.Matmul(const, trans)(A, B, ppkernel=pp)
    return C


def _entry(trans, A, B, C):
    """The C entry itself, which also takes the shapes for which packing first is the faster way."""
    (M, K), N = A.shape, C.shape[1]
    s, ws = L.Epilogue(C).struct(), L.workspace()
    L._check(L.lib().mmx_gemm_unpacked(L.BF16, A.data_ptr(), L._row_stride_bytes(A), B.data_ptr(), L._row_stride_bytes(B), int(trans), M, K, N,
                                       ctypes.byref(s), ws.data_ptr(), ws.numel(), L._stream()))


# one step of k for one wavefront, shares with and without a remainder, a K split and none; rows on both sides of a block
# of 16, 32 and 64; a strip of 128 columns with 8 of them live, full, and one more
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("M,K,N", [(1, 32, 8), (15, 288, 128), (16, 4096, 136), (17, 1056, 264), (32, 8192, 256), (33, 96, 640),
                                   (64, 2080, 384), (65, 4096, 128), (130, 640, 1000), (256, 1024, 1024), (300, 4128, 200)])
@pytest.mark.parametrize("pad", [0, 5])
def test_exact_sums(M, K, N, trans, pad):
    A, B = _ints((M, K), 1, pad), _ints((N, K) if trans else (K, N), 2, pad)
    wide = torch.full((M + 1, N + 3), -7.0, device="cuda")
    _entry(trans, A, B, wide[:M, :N])
    assert mx.last_kernel().startswith("unpacked_" + ("nk" if trans else "kn")), mx.last_kernel()
    if K >= 4096 and M <= 32:  # (few strips and a long K)
        assert not mx.last_kernel().endswith("ksplit1"), mx.last_kernel()
    ref = A.double() @ (B.double().t() if trans else B.double())
    assert torch.equal(wide[:M, :N].double(), ref)
    assert (wide[M] == -7.0).all() and (wide[:, N:] == -7.0).all()  # nothing beyond the result is written
    again = torch.empty((M, N), device="cuda")
    for _ in range(3):  # (the arrival counters are back at zero)
        _entry(trans, A, B, again)
    assert torch.equal(again.double(), ref)
    assert torch.equal(_run(False, trans, A, B, again.zero_()).double(), ref)  # whichever way the rule takes


@pytest.mark.parametrize("trans", [False, True])
def test_a_smaller_workspace_means_fewer_slices(trans):
    """All of the workspace it asks for, half of it, and none; another call's workspace is left as it is behind the limit."""
    M, K, N = 16, 8192, 520
    A, B = _ints((M, K), 30), _ints((N, K) if trans else (K, N), 31)
    ref = A.double() @ (B.double().t() if trans else B.double())
    need = L.lib().mmx_gemm_unpacked_workspace_bytes(L.BF16, M, K, N, K * 2, B.shape[1] * 2, int(trans))
    ws, slices = torch.zeros(need, dtype=torch.uint8, device="cuda"), []
    for limit in (need, need // 2, 1 << 14, 0):
        C = torch.empty((M, N), device="cuda")
        s = L.Epilogue(C).struct()
        ws[limit:] = 0xA5
        L._check(L.lib().mmx_gemm_unpacked(L.BF16, A.data_ptr(), K * 2, B.data_ptr(), B.shape[1] * 2, int(trans), M, K, N, ctypes.byref(s),
                                           ws.data_ptr() if limit else None, limit, L._stream()))
        assert torch.equal(C.double(), ref) and (ws[limit:] == 0xA5).all()
        slices.append(int(mx.last_kernel().split("ksplit")[1]))
    assert slices[0] > slices[1] > 1 and slices[2:] == [1, 1], slices


@pytest.mark.parametrize("trans", [False, True])
def test_b_at_an_odd_address(trans):
    """A caller of the C entry may hand over a B that is not aligned to its element, as it may to mmx_repack_b."""
    M, K, N = 20, 160, 136
    A, B = _ints((M, K), 28), _ints((N, K) if trans else (K, N), 29)
    room = torch.zeros(B.numel() * 2 + 1, dtype=torch.uint8, device="cuda")
    room[1:] = B.contiguous().view(torch.uint8).view(-1)
    C = torch.empty((M, N), device="cuda")
    s = L.Epilogue(C).struct()
    L._check(L.lib().mmx_gemm_unpacked(L.BF16, A.data_ptr(), K * 2, room.data_ptr() + 1, B.shape[1] * 2, int(trans), M, K, N, ctypes.byref(s),
                                       None, 0, L._stream()))
    assert torch.equal(C.double(), A.double() @ (B.double().t() if trans else B.double()))


# 16, 32 and 64 rows to a workgroup, with K slices and without, the last workgroup with a few rows; one step of k and a
# column of C's last four that stands alone
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("M,K,N,rows", [(50, 512, 520, 16), (100, 512, 520, 32), (129, 2080, 2056, 32), (250, 1024, 4104, 64),
                                        (64, 4096, 8200, 64), (49, 32, 72, 16)])
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16, torch.int8])
def test_every_row_block_and_store(out, M, K, N, rows, trans):
    A, B = _ints((M, K), 32), _ints((N, K) if trans else (K, N), 33)
    N -= 3 if trans else 0  # (from [N, K] any column count)
    B = B[:N] if trans else B
    wide = torch.full((M + 1, N + 5), -7, dtype=out, device="cuda")
    _entry(trans, A, B, wide[:M, 1:N + 1])  # rows of C at any multiple of an element
    assert f"_rows{rows}_" in mx.last_kernel(), mx.last_kernel()
    ref = A.double() @ (B.double().t() if trans else B.double())
    assert torch.equal(wide[:M, 1:N + 1], ref.clamp(-128, 127).to(out) if out == torch.int8 else ref.to(out))
    assert (wide[M] == -7).all() and (wide[:, N + 1:] == -7).all() and (wide[:, 0] == -7).all()


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("M,K,N", [(96, 64, 65536), (128, 128, 32768), (96, 256, 65536), (64, 512, 512), (64, 1024, 256), (128, 512, 1024),
                                   (96, 1024, 2048), (1, 8192, 640)])
def test_the_faster_way_is_taken(M, K, N, trans):
    """Device time of the way the query names against packing first.  In workgroups of 64 rows throughout, with two-byte
    stores, these took up to 2.1 times as long as packing first; now 0.5 to 1.0 times."""
    lib, C = L.lib(), torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    A, B = (torch.randn(shape, device="cuda").to(torch.bfloat16) for shape in ((M, K), (N, K) if trans else (K, N)))
    s, ws, ldb = L.Epilogue(C).struct(), L.workspace(), B.shape[1] * 2
    packed = torch.empty(mx.packed_b_bytes(mx.BF16, K, N), dtype=torch.uint8, device="cuda")
    if lib.mmx_gemm_unpacked_workspace_bytes(L.BF16, M, K, N, K * 2, ldb, int(trans)) < 0:
        return  # packed first

    def unpacked():
        L._check(lib.mmx_gemm_unpacked(L.BF16, A.data_ptr(), K * 2, B.data_ptr(), ldb, int(trans), M, K, N, ctypes.byref(s), ws.data_ptr(),
                                       ws.numel(), L._stream()))

    def pack_first():
        L._check(lib.mmx_repack_b(L.BF16, B.data_ptr(), ldb, K, N, int(trans), packed.data_ptr(), L._stream()))
        L._check(lib.mmx_gemm_splitk(L.BF16, L.BF16, A.data_ptr(), K * 2, packed.data_ptr(), M, K, N, 0, N, ctypes.byref(s), 0, ws.data_ptr(),
                                     ws.numel(), L._stream()))
    took = [call_us(f, n=30) for f in (unpacked, pack_first)]
    assert took[0] <= 1.25 * took[1], took


@pytest.mark.parametrize("N", [8, 131, 250])
def test_any_column_count_from_rows_of_k(N):
    A, B = _ints((24, 96), 3), _ints((N, 96), 4)
    C = _run(False, True, A, B, torch.empty((24, N), device="cuda"))
    assert mx.last_kernel().startswith("unpacked_nk")
    assert torch.equal(C.double(), A.double() @ B.double().t())


@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16, torch.int8])
@pytest.mark.parametrize("steps", [mx.Steps.NONE, mx.Steps.BIAS, mx.Steps.BIAS_GELU, mx.Steps.DEQUANT_BIAS_GELU_QUANT])
def test_post_ops_equal_the_packed_form(out, steps):
    M, K, N = 19, 2048, 264
    A, B = _ints((M, K), 5), _ints((K, N), 6)
    kw = {"steps": steps, "bias": torch.linspace(-3, 3, N, device="cuda") if steps & mx.Steps.BIAS else None}
    if steps & mx.Steps.QUANT:
        kw["q"] = torch.linspace(0.01, 0.1, N, device="cuda")
    got = _run(False, False, A, B, torch.empty((M, N), dtype=out, device="cuda"), **kw)
    assert mx.last_kernel().startswith("unpacked_kn")
    want = _run(True, False, A, B, torch.empty((M, N), dtype=out, device="cuda"), **kw)
    assert torch.equal(got, want)


@pytest.mark.parametrize("trans", [False, True])
def test_infinities_stay_in_their_column_and_row(trans):
    M, K, N = 20, 320, 200
    A, B = _ints((M, K), 7), _ints((N, K) if trans else (K, N), 8)
    A[3, 1] = float("nan")
    (B if trans else B.t())[5, 0], (B if trans else B.t())[199, 319] = float("inf"), float("-inf")
    got = _run(False, trans, A, B, torch.empty((M, N), device="cuda"))
    assert mx.last_kernel().startswith("unpacked"), mx.last_kernel()
    want = _run(True, trans, A, B, torch.empty((M, N), device="cuda"))
    assert not torch.isfinite(want[:, [5, 199]]).any() and torch.isfinite(want[0, :5]).all()
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    ok = torch.isfinite(want)
    assert torch.equal(got[ok], want[ok])


def test_what_it_does_not_take_is_packed():
    for (M, K, N), trans in [((4, 40, 64), False), ((4, 64, 63), False), ((2000, 256, 256), False), ((4, 33, 64), True)]:
        A, B = _ints((M, K), 9), _ints((N, K) if trans else (K, N), 10)
        C = _run(False, trans, A, B, torch.empty((M, N), device="cuda"))
        assert not mx.last_kernel().startswith("unpacked")
        assert torch.equal(C.double(), A.double() @ (B.double().t() if trans else B.double()))


def test_column_ranges_are_packed():
    A, B = _ints((4, 64), 11), _ints((64, 96), 12)
    C = torch.zeros((4, 96), device="cuda")
    mx.Matmul(False, False)(A, B, 32, 64, mx.BiasGeluStore(C))
    assert torch.equal(C[:, 32:64].double(), (A.double() @ B.double())[:, 32:64]) and not C[:, :32].any() and not C[:, 64:].any()


@pytest.mark.parametrize("trans", [False, True])
def test_a_result_over_b_is_packed(trans):
    M, K, N = 24, 512, 512
    A, B = _ints((M, K), 16), _ints((K, N), 17)
    ref = A.double() @ (B.double().t() if trans else B.double())
    for rows in (slice(0, M), slice(K - M, K)):
        over = B.clone()
        C = over[rows]  # the first and the last rows of B itself
        _run(False, trans, A, over, C)
        assert not mx.last_kernel().startswith("unpacked")
        assert torch.equal(C, ref.to(torch.bfloat16))
    both = torch.cat([B, B[:M]])  # right behind B: no overlap
    _run(False, trans, A, both[:K], both[K:])
    assert mx.last_kernel().startswith("unpacked") and torch.equal(both[K:], ref.to(torch.bfloat16))


def test_replays_from_a_hip_graph():
    M, K, N = 24, 8192, 256
    A, B, C = _ints((M, K), 13), _ints((K, N), 14), torch.empty((M, N), device="cuda")
    op, pp = mx.Matmul(False, False), mx.BiasGeluStore(C)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        op(A, B, ppkernel=pp)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            op(A, B, ppkernel=pp)
        assert mx.last_kernel().startswith("unpacked") and not mx.last_kernel().endswith("ksplit1"), mx.last_kernel()
    for seed in range(15, 19):
        A.copy_(_ints((M, K), seed))
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C.double(), A.double() @ B.double())


@pytest.mark.parametrize("trans", [False, True])
def test_a_first_call_under_capture_packs(trans):
    """A stream that is being captured gets no workspace; unsplit, a shape that wants slices is several times slower than
    packed (1 x 65536 x 512 from [N, K] 462 against 129 us)."""
    M, K, N = 4, 8192, 256
    A, B, C = _ints((M, K), 21), _ints((N, K) if trans else (K, N), 22), torch.empty((M, N), device="cuda")
    op, pp = mx.Matmul(False, trans), mx.BiasGeluStore(C)
    side = torch.cuda.Stream()
    mx.release_workspaces()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        op(A, B, ppkernel=pp)
    assert not mx.last_kernel().startswith("unpacked"), mx.last_kernel()
    for seed in range(23, 26):
        B.copy_(_ints(tuple(B.shape), seed))
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C.double(), A.double() @ (B.double().t() if trans else B.double()))


def test_gate_and_up_in_turn_are_packed():
    """A post-op of the caller's own may ask for SILU_GATE over a B whose panels alternate already."""
    M, K, N = 8, 256, 128
    A, B = _ints((M, K), 26), _ints((K, 2 * N), 27)

    class GateStore:
        def __init__(self, C):
            self.C = C

        def descriptor(self):
            return L.Epilogue(self.C, L.PP_SILU_GATE)

    got, want = (torch.empty((M, N), device="cuda") for _ in range(2))
    mx.Matmul(False, False)(A, B, ppkernel=GateStore(got))
    mx.Matmul(True, False)(A, B, ppkernel=GateStore(want))
    assert torch.equal(got, want)


def test_errors_of_the_c_entry():
    A, B, C = _ints((4, 64), 1), _ints((64, 64), 2), torch.empty((4, 64), device="cuda")
    s = L.Epilogue(C).struct()
    call = lambda dt, lda, ldb, st: L.lib().mmx_gemm_unpacked(dt, A.data_ptr(), lda, B.data_ptr(), ldb, 0, 4, 64, 64, ctypes.byref(st), None, 0, L._stream())
    assert call(L.BF16, 128, 128, s) == 0
    assert call(L.I8, 128, 128, s) != 0 and call(L.BF16, 126, 128, s) != 0 and call(L.BF16, 128, 126, s) != 0 and call(L.BF16, 129, 128, s) != 0
    s.steps = L.PP_SILU_GATE
    assert call(L.BF16, 128, 128, s) != 0
