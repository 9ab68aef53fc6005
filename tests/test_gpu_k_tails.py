"""The tile kernels at a K that does not fill its last 128 bytes (aligned rows: the ring pipeline's last step; rows of any
alignment: the masked pipeline), against the oracle: remainders of 2 to 126 bytes, one whole k-iteration in front or many,
every tile that takes a tail, the K split, the gate/up store; and that the kernel named is the one that ran."""
import numpy as np
import pytest
import torch

import mm_amx_amd as mx
from gpu_util import call_us, check_float_parity, dev, dev_bf16, host_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    mx.init(0)
    yield
    mx.set_tile("")


def _in_nan(t, pad):
    """t inside a wider matrix of NaN (bf16) or 77 (int8): what lies behind a row must not enter the result."""
    wide = torch.full((t.shape[0], t.shape[1] + pad), float("nan") if t.dtype == torch.bfloat16 else 77, dtype=t.dtype, device="cuda")
    wide[:, :t.shape[1]] = t
    return wide[:, :t.shape[1]]


@pytest.mark.parametrize("tile", ["", "256x192", "128x128", "128x64", "64x128"])
@pytest.mark.parametrize("K", [3, 7, 8, 9, 63, 65, 72, 127, 200, 1089])
@pytest.mark.parametrize("kind", ["bf16", "w8", "i8"])
def test_k_tail(po, kind, K, tile):
    M, N = (300, 200) if tile == "" else (131, 97)
    if kind == "i8":
        K *= 2
    rng = np.random.default_rng(K)
    W = rng.integers(-127, 128, (K, N)).astype(np.int8)
    if kind == "i8":
        A = rng.integers(-127, 128, (M, K)).astype(np.int8)
        up, ref, kw, odt = dev, po.gemm_i8(A, W), {}, torch.int32
    else:
        A = po.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
        if kind == "bf16":
            W = po.f32_to_bf16((rng.standard_normal((K, N)) * 0.05).astype(np.float32))
        ref = po.gemm_bf16(A, W if kind == "bf16" else po.f32_to_bf16(W.astype(np.float32)))
        up, kw, odt = dev_bf16, ({} if kind == "bf16" else {"b_dtype": mx.I8}), torch.float32
    packed = mx.repack_b((dev_bf16 if kind == "bf16" else dev)(W))
    es = 1 if kind == "i8" else 2
    mx.set_tile(tile)
    for pad in ((-K * es % 16) // es + 16 // es, 3):   # rows 16-byte aligned, and not
        C = torch.zeros((M, N), dtype=odt, device="cuda")
        mx.gemm(_in_nan(up(A), pad), packed, N, mx.Epilogue(C), **kw)
        if pad != 3 and K * es > 128:  # (no 128x64 tile over int8 weights)
            assert (("128x128" if kind == "w8" and tile == "128x64" else tile) + "_ring") in mx.last_kernel(), mx.last_kernel()
        else:
            assert "128x128_masked" in mx.last_kernel(), mx.last_kernel()
        if kind == "i8":
            assert np.array_equal(host_bits(C), ref), mx.last_kernel()
        else:
            check_float_parity(host_bits(C), ref, f"{kind} K={K} pad={pad} {mx.last_kernel()}")
    mx.set_tile("")


@pytest.fixture
def tile(request):
    """The tile of the case, forced (the small tiles, which have tests of their own, would take these shapes)."""
    mx.set_tile(request.param)
    yield request.param
    mx.set_tile("")


@pytest.mark.parametrize("tile", ["128x128", "64x128"], indirect=True)
@pytest.mark.parametrize("K", [4104, 4400])
@pytest.mark.parametrize("kind", ["bf16", "w8", "i8"])
def test_k_tail_behind_a_k_split(po, kind, K, tile):
    """Few tiles and a long K: the last slice, and it alone, takes the tail (16 and 96 bytes of A)."""
    M, N = 64, 256
    rng = np.random.default_rng(K)
    if kind == "i8":
        K *= 2
        A, B = (rng.integers(-127, 128, shape).astype(np.int8) for shape in ((M, K), (K, N)))
        C, up, ref = torch.zeros((M, N), dtype=torch.int32, device="cuda"), dev, po.gemm_i8(A, B)
    else:
        A = po.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
        B = po.f32_to_bf16((rng.standard_normal((K, N)) * 0.05).astype(np.float32)) if kind == "bf16" else \
            rng.integers(-127, 128, (K, N)).astype(np.int8)
        C, up = torch.zeros((M, N), dtype=torch.float32, device="cuda"), dev_bf16
        ref = po.gemm_bf16(A, B if kind == "bf16" else po.f32_to_bf16(B.astype(np.float32)))
    mx.gemm(up(A), mx.repack_b((dev_bf16 if kind == "bf16" else dev)(B)), N, mx.Epilogue(C), **({"b_dtype": mx.I8} if kind == "w8" else {}))
    assert f"_{tile}_ring_" in mx.last_kernel() and "ksplit" in mx.last_kernel(), mx.last_kernel()
    if kind == "i8":
        assert np.array_equal(host_bits(C), ref), mx.last_kernel()
    else:
        check_float_parity(host_bits(C), ref, mx.last_kernel())


@pytest.mark.parametrize("tile", ["256x256", "128x256", "128x192"], indirect=True)
@pytest.mark.parametrize("K", [65, 72, 191, 200, 1096])
@pytest.mark.parametrize("kind", ["bf16", "w8", "i8"])
def test_k_tail_wide_tiles(po, kind, K, tile):
    """One k-iteration before the tail and many, tails of whole 16-byte pieces and not, more than one tile each way; and gate/up pairs."""
    M, N = 270, 576
    rng = np.random.default_rng(K)
    if kind == "i8":
        K *= 2
    W = rng.integers(-127, 128, (K, N)).astype(np.int8)
    if kind == "i8":
        A = rng.integers(-127, 128, (M, K)).astype(np.int8)
        up, ref, kw, odt = dev, po.gemm_i8(A, W), {}, torch.int32
    else:
        A = po.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
        if kind == "bf16":
            W = po.f32_to_bf16((rng.standard_normal((K, N)) * 0.05).astype(np.float32))
        ref = po.gemm_bf16(A, W if kind == "bf16" else po.f32_to_bf16(W.astype(np.float32)))
        up, kw, odt = dev_bf16, ({} if kind == "bf16" else {"b_dtype": mx.I8}), torch.float32
    es = 1 if kind == "i8" else 2
    x = _in_nan(up(A), (-K * es % 16) // es + 16 // es)  # (rows 16-byte aligned, NaN or 77 behind them)
    packed = mx.repack_b((dev_bf16 if kind == "bf16" else dev)(W))
    C = torch.zeros((M, N), dtype=odt, device="cuda")
    mx.gemm(x, packed, N, mx.Epilogue(C), **kw)
    assert f"_{tile}_ring" in mx.last_kernel(), mx.last_kernel()
    if kind == "i8":
        assert np.array_equal(host_bits(C), ref), mx.last_kernel()
        return
    check_float_parity(host_bits(C), ref, f"{kind} K={K} {mx.last_kernel()}")
    if tile != "128x192":  # gate and up panels in turn; silu within 2^-14 as below
        scale = 1.0 if kind == "bf16" else 2.0 ** -10
        h = torch.zeros((M, N // 2), dtype=torch.float32, device="cuda")
        mx.gemm(x, packed, N, mx.Epilogue(h, mx.PP_SILU_GATE | (mx.PP_DEQUANT if kind == "w8" else 0), deq_scale=scale), **kw)
        assert f"_{tile}_ring" in mx.last_kernel(), mx.last_kernel()
        g, u = (np.concatenate([ref[:, n:n + 32] for n in range(32 * i, N, 64)], axis=1).astype(np.float64) * scale for i in (0, 1))
        want = g / (1.0 + np.exp(-g)) * u
        assert np.linalg.norm(host_bits(h).astype(np.float64) - want) <= 2.0 ** -13 * np.linalg.norm(want), mx.last_kernel()


@pytest.mark.parametrize("kind,M,K,pad", [("bf16", 64, 4100, 4), ("bf16", 64, 4100, 0), ("w8", 64, 4100, 4), ("i8", 64, 8201, 7),
                                          ("i8", 16, 8256, 0), ("i8", 16, 8320, 0), ("bf16", 16, 8200, 0)])
def test_the_plan_does_not_depend_on_earlier_calls(kind, M, K, pad):
    """The first call of a stream and a call that finds the stream's workspace: the same kernel, the same bits."""
    N = 256
    g = torch.Generator(device="cuda").manual_seed(K)
    A = torch.randn((M, K + pad), device="cuda", generator=g)[:, :K] if kind != "i8" else \
        torch.randint(-127, 128, (M, K + pad), device="cuda", generator=g, dtype=torch.int8)[:, :K]
    A = A if kind == "i8" else _in_nan(A.to(torch.bfloat16), pad)
    W = torch.randint(-127, 128, (K, N), device="cuda", generator=g, dtype=torch.int8)
    packed = mx.repack_b(W.to(torch.bfloat16) if kind == "bf16" else W)
    kw = {"b_dtype": mx.I8} if kind == "w8" else {}
    out = torch.zeros((2, M, N), dtype=torch.float32, device="cuda")
    mx.release_workspaces()
    mx.gemm(A, packed, N, mx.Epilogue(out[0]), **kw)
    first = mx.last_kernel()
    mx.workspace()
    mx.gemm(A, packed, N, mx.Epilogue(out[1]), **kw)
    assert mx.last_kernel() == first
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("tile", ["128x128"], indirect=True)  # (the only one with pairs and a tail)
@pytest.mark.parametrize("kind", ["bf16", "w8"])
def test_k_tail_gate_up(po, kind, tile):
    M, K, N = 70, 200, 96
    rng = np.random.default_rng(5)
    x = po.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
    h = torch.zeros((M, N), dtype=torch.float32, device="cuda")
    if kind == "bf16":
        wg, wu = (po.f32_to_bf16((rng.standard_normal((N, K)) * 0.05).astype(np.float32)) for _ in range(2))
        mx.gemm(dev_bf16(x), mx.repack_gate_up(dev_bf16(wg), dev_bf16(wu)), 2 * N, mx.Epilogue(h, mx.PP_SILU_GATE))
    else:  # (gate and up in turn, 32 columns each; the scale keeps silu where it bends)
        wg, wu = (rng.integers(-127, 128, (N, K)).astype(np.int8) for _ in range(2))
        both = np.concatenate([w[n:n + 32] for n in range(0, N, 32) for w in (wg, wu)])
        mx.gemm(dev_bf16(x), mx.repack_b(dev(both), transpose=True), 2 * N,
                mx.Epilogue(h, mx.PP_SILU_GATE | mx.PP_DEQUANT, deq_scale=2.0 ** -10), b_dtype=mx.I8)
    assert f"_{tile}_ring_" in mx.last_kernel(), mx.last_kernel()
    g, u = (po.gemm_bf16(x, np.ascontiguousarray((w if kind == "bf16" else po.f32_to_bf16(w.astype(np.float32))).T)) for w in (wg, wu))
    if kind == "w8":
        g, u = g * 2.0 ** -10, u * 2.0 ** -10
    # silu is a 2^-14 approximation of g / (1 + exp(-g)); twice that for the roundings around it
    want = g / (1.0 + np.exp(-g.astype(np.float64))) * u
    got = host_bits(h).astype(np.float64)
    assert np.linalg.norm(got - want) <= 2.0 ** -13 * np.linalg.norm(want), mx.last_kernel()


def test_a_tail_is_one_trip_to_memory():
    """The masked pipeline at a K with one k-iteration: fetched in a chain its loads took 1.31 times as long as those of a K
    that fills the iteration, all in flight 1.06 times."""
    M, N = 1500, 65536
    ep = mx.Epilogue(torch.empty((M, N), dtype=torch.bfloat16, device="cuda"))
    took = {}
    for K in (40, 64):
        A = torch.randn((M, K + 3), device="cuda").to(torch.bfloat16)[:, :K]
        packed = mx.repack_b(torch.randn((K, N), device="cuda").to(torch.bfloat16))
        took[K] = call_us(lambda: mx.gemm(A, packed, N, ep))
        assert "masked" in mx.last_kernel()
    assert took[40] <= 1.2 * took[64], took


@pytest.mark.parametrize("M,K,N", [(33, 513, 64), (40, 1001, 257), (130, 1999, 96), (300, 2234, 700), (64, 5003, 40)])
@pytest.mark.parametrize("kind", ["bf16", "w8", "i8"])
def test_dense_rows_that_are_not_whole_pieces(po, kind, M, K, N):
    """Copied to the workspace first: an infinity (127s) in one row stays in that row, the workspace ends with the copy and its counters
    are zero afterwards; a smaller one, or none, leaves the call to the masked pipeline."""
    rng = np.random.default_rng(K)
    W = rng.integers(-127, 128, (K, N)).astype(np.int8)
    if kind == "i8":
        A = rng.integers(-127, 128, (M, K)).astype(np.int8)
        A[3] = 127
        ref, up, kw, odt, es = po.gemm_i8(A, W), dev, {}, torch.int32, 1
    else:
        A = po.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
        if kind == "bf16":
            W = po.f32_to_bf16((rng.standard_normal((K, N)) * 0.05).astype(np.float32))
        ref, up, kw, odt, es = po.gemm_bf16(A, W if kind == "bf16" else po.f32_to_bf16(W.astype(np.float32))), dev_bf16, \
            ({} if kind == "bf16" else {"b_dtype": mx.I8}), torch.float32, 2
    packed, x = mx.repack_b((dev_bf16 if kind == "bf16" else dev)(W)), up(A)
    if kind != "i8":
        x[3, 0] = float("inf")
    others = np.arange(M) != 3
    room = (16 << 10) + (M + 1) * ((K * es + 127) // 128 * 128) + (8 << 20)
    ws = torch.zeros(room + 64, dtype=torch.uint8, device="cuda")
    ws[room:] = 0xA5
    for how in ("stream", "given", "small", "none"):
        C = torch.full((M + 1, N + 3), -7, dtype=odt, device="cuda")
        extra = {"stream": {}, "given": {"ws": ws[:room]}, "small": {"ws": ws[:16 << 10]}, "none": {"k_splits": 1}}[how]
        mx.gemm(x, packed, N, mx.Epilogue(C[:M, :N]), **kw, **extra)
        assert mx.last_kernel().endswith("_rows_copied") == (how in ("stream", "given")), (how, mx.last_kernel())
        got = host_bits(C)
        assert (got[M] == -7).all() and (got[:, N:] == -7).all()
        if kind == "i8":
            assert np.array_equal(got[:M, :N], ref), (how, mx.last_kernel())
        else:
            assert not np.isfinite(got[3, :N]).any()
            check_float_parity(got[:M, :N][others], ref[others], f"{how} {mx.last_kernel()}")
    assert not ws[:16 << 10].any().item() and (ws[room:] == 0xA5).all().item()


# either side of the line: one nearly full round of masked tiles, more than one, half of one, fewer rows, longer ones
@pytest.mark.parametrize("kind,M,K,N,copied", [("i8", 1867, 1109, 2103, False), ("w8", 1909, 519, 1118, False), ("bf16", 1898, 555, 1887, False), ("bf16", 1898, 555, 2200, True),
                                               ("i8", 1801, 1185, 1000, True), ("i8", 994, 1297, 2276, True), ("w8", 1795, 901, 1800, True)])
def test_dense_rows_are_copied_where_that_is_faster(kind, M, K, N, copied):
    """us, masked / copied: 15.5 / 18.8 for the first, 16.1 / 14.5 for int8 994 x 1297 x 2276."""
    g = torch.Generator(device="cuda").manual_seed(K)
    x, W = (torch.randint(-127, 128, s, device="cuda", generator=g, dtype=torch.int8) for s in ((M, K), (K, N)))
    want = x.double() @ W.double()
    C = torch.zeros((M, N), dtype=torch.int32 if kind == "i8" else torch.float32, device="cuda")
    mx.gemm(x if kind == "i8" else x.to(torch.bfloat16), mx.repack_b(W.to(torch.bfloat16) if kind == "bf16" else W), N, mx.Epilogue(C),
            b_dtype=mx.BF16 if kind == "bf16" else mx.I8)
    assert mx.last_kernel().endswith("_rows_copied") == copied and ("masked" in mx.last_kernel()) != copied, mx.last_kernel()
    assert torch.equal(C.double(), want)  # (whole numbers below 2^24: exact in any order)


# few rows and many, slices of every kind of kernel that the copy goes on to and none, a column range; int8 down to one row (the decode kernels)
@pytest.mark.parametrize("kind,M,K,N,n0,n1", [("bf16", 40, 1001, 1024, 0, 1024), ("bf16", 100, 5001, 1000, 0, 1000), ("bf16", 300, 2234, 700, 64, 601), ("bf16", 64, 9001, 512, 0, 512),
                                              ("bf16", 500, 9001, 1100, 0, 1100), ("bf16", 700, 700, 900, 0, 900), ("w8", 64, 4099, 256, 0, 256), ("w8", 300, 8001, 2000, 0, 2000),
                                              ("i8", 64, 8199, 256, 0, 256), ("i8", 400, 3333, 1000, 0, 1000), ("i8", 1, 4001, 300, 0, 300), ("i8", 17, 9990, 640, 0, 640),
                                              ("i8", 32, 515, 1000, 32, 1000), ("i8", 32, 7999, 640, 0, 640)])
def test_the_workspace_query_is_enough(po, kind, M, K, N, n0, n1):
    """Dense rows of an odd K with a workspace of just the size that the query names: the kernel and the bits are those of the standard
    workspace, and what lies behind it stays; with 256 bytes less the copy or a slice does not fit, and the result is right all the same."""
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randint(-127, 128, (M, K), device="cuda", generator=g, dtype=torch.int8)
    W = torch.randint(-127, 128, (K, N), device="cuda", generator=g, dtype=torch.int8)
    if kind != "i8":
        x = x.to(torch.bfloat16)
    packed = mx.repack_b(W if kind != "bf16" else W.to(torch.bfloat16))
    # (products of whole numbers below 2^24 in every partial sum of int8; of bf16 the sums are compared to the precision of 32 bits)
    want = (x.double() @ W.double())[:, n0:n1]
    types, es = (mx.I8 if kind == "i8" else mx.BF16, mx.BF16 if kind == "bf16" else mx.I8), 1 if kind == "i8" else 2
    need = mx.gemm_workspace_bytes(*types, M, K, N, n0=n0, n1=n1)
    pitch = (K * es + 127) // 128 * 128
    beside = max(16 << 10, mx.gemm_workspace_bytes(*types, M, pitch // es, N, n0=n0, n1=n1))
    tight = M > 32 and need < beside + M * pitch + 512  # (not where aligned rows of this K take more, for slices)
    assert (16 << 10) < need <= mx._lib.WORKSPACE_BYTES
    answers = []
    for size in (mx._lib.WORKSPACE_BYTES, need, need - 256):
        ws = torch.zeros(mx._lib.WORKSPACE_BYTES + 4096, dtype=torch.uint8, device="cuda")
        ws[size:] = 0xA5
        C = torch.zeros((M, N), dtype=torch.int32 if kind == "i8" else torch.float32, device="cuda")
        mx.gemm(x, packed, N, mx.Epilogue(C), b_dtype=types[1], n0=n0, n1=n1, ws=ws[:size])
        answers.append((mx.last_kernel(), C))
        assert (ws[size:] == 0xA5).all().item() and not ws[:16 << 10].any().item(), (size, mx.last_kernel())
        if kind == "i8":
            assert torch.equal(C[:, n0:n1].double(), want), (size, mx.last_kernel())
        else:  # 32-bit sums of K products, in any order
            assert ((C[:, n0:n1].double() - want).abs() <= K * 2.0 ** -24 * (x.double().abs() @ W.double().abs())[:, n0:n1]).all(), (size, mx.last_kernel())
        assert not C[:, :n0].any().item() and not C[:, n1:].any().item()
    assert answers[0][0].endswith("_rows_copied") and answers[1][0] == answers[0][0], [a[0] for a in answers]
    assert not tight or answers[2][0] != answers[0][0], [a[0] for a in answers]
    assert torch.equal(answers[0][1], answers[1][1])
    if kind == "i8" and M <= 32:  # (the decode kernels take the copy where x fits in LDS or its rows are whole chunks)
        assert answers[0][0].startswith("skinny_") == (M * pitch <= 45 << 10 or pitch % 256 == 0), answers[0][0]


def test_dense_rows_replay_from_a_graph():
    """Copy and product in a captured graph, new rows before each replay."""
    M, K, N = 200, 1335, 384
    x = torch.zeros((M, K), dtype=torch.bfloat16, device="cuda")
    packed, C = mx.repack_b(torch.randn((K, N), device="cuda").to(torch.bfloat16)), torch.zeros((M, N), device="cuda")
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        mx.gemm(x, packed, N, mx.Epilogue(C))
        assert mx.last_kernel().endswith("_rows_copied")
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            mx.gemm(x, packed, N, mx.Epilogue(C))
    for seed in range(3):
        x.copy_(torch.randn((M, K), device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed)).to(torch.bfloat16))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        eager = torch.zeros((M, N), device="cuda")
        mx.gemm(x, packed, N, mx.Epilogue(eager))
        assert torch.equal(C, eager), seed
