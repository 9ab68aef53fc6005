"""The native host side of a call (csrc/host_call.cpp) against the Python form: the same kernel, the same bits, the same errors.

Every call is made twice, through native code and with it switched off.  `taken` says whether native code is to take it:
what is not regular in every respect is the Python form's, which accepts it or says what is wrong."""
import numpy as np
import pytest
import torch

import mm_amx_amd as mx
from gpu_util import host_bits
from mm_amx_amd import _host_call
from mm_amx_amd import _lib as L

pytestmark = pytest.mark.gpu


class _Watch:
    """The native module, noting what it answered."""

    def __init__(self, module):
        self.module, self.answers = module, []

    def __getattr__(self, name):
        def call(*a):
            self.answers.append(getattr(self.module, name)(*a))
            return self.answers[-1]
        return call


def _both(monkeypatch, call):
    """[(result or error text, kernel)] of the call through native code and through Python, and native code's answers."""
    mx.lib()
    watch, out = _Watch(L._native), []
    for native in (watch, None):
        monkeypatch.setattr(L, "_native", native)
        try:
            r = call()
            out.append((host_bits(r).copy(), mx.last_kernel()))
        except L.MmxError as e:
            out.append((str(e), None))
    return out, watch.answers


def _bf(*shape):
    return torch.randn(shape, device="cuda").to(torch.bfloat16)


def _gemm_calls():
    torch.manual_seed(3)
    M, K, N = 48, 192, 160
    x, xi = _bf(M, K), torch.randint(-127, 128, (M, K), device="cuda", dtype=torch.int8)
    W = _bf(N, K)
    pb = mx.repack_b(W, transpose=True)
    p8 = mx.repack_b(torch.randint(-127, 128, (N, K), device="cuda", dtype=torch.int8), transpose=True)
    p4, d4 = mx.quantize_pack_int4(W, transpose=True)
    bias, scale = torch.randn(N, device="cuda"), torch.rand(N, device="cuda")
    ws = torch.zeros(L.WORKSPACE_BYTES, dtype=torch.uint8, device="cuda")

    def call(A, B, n=N, dt=torch.float32, rows=M, cols=N, steps=0, wide=0, C=None, edit=None, ep=None, **kw):
        def go():
            out = torch.zeros((rows, cols + wide), dtype=dt, device="cuda") if C is None else C()
            e = mx.Epilogue(out[:, :cols] if C is None else out, steps, **(ep or {}))
            if edit:
                edit(e)
            mx.gemm(A, B, n, e, **kw)
            return out
        return go

    short = dict(bias=bias[:N - 1].contiguous())
    return {
        "bf16": (True, call(x, pb)),
        "post-op": (True, call(x, pb, dt=torch.bfloat16, steps=7, wide=3, ep=dict(bias=bias, deq_scale=0.5))),
        "scales of columns": (True, call(xi, p8, dt=torch.int8, steps=13, ep=dict(deq_scale_per_oc=scale, q_scale_per_oc=scale, bias=bias))),
        "int32": (True, call(xi, p8, dt=torch.int32)),
        "int8 weights": (True, call(x, p8, steps=1, b_dtype=L.I8)),
        "int4 weights": (True, call(x[:3], p4, steps=1, dt=torch.bfloat16, ep=dict(deq_scale_per_oc=d4), b_dtype=L.I4)),
        "some columns": (True, call(x, pb, n0=32, n1=96)),
        "a row": (True, call(x[5:6], pb)),
        "a row of any stride": (True, call(x.as_strided((1, K), (7, 1)), pb)),
        "rows with gaps": (True, call(_bf(M, K + 9)[:, 4:K + 4], pb)),
        "a workspace": (True, call(x, pb, ws=ws, k_splits=0)),
        "two slices": (True, call(x, pb, ws=ws, k_splits=2)),
        "unsplit": (True, call(x, pb, k_splits=1)),
        "an error of the library": (True, call(x, pb, n0=16)),
        "a parameter": (True, call(torch.nn.Parameter(x, requires_grad=False), pb)),
        "a count of slices without a workspace": (False, call(x, pb, k_splits=2)),
        "a numpy N": (False, call(x, pb, n=np.int64(N))),
        "columns of A": (False, call(_bf(K, M).t(), pb)),
        "fp32 A": (False, call(x.float(), pb)),
        "too few packed bytes": (False, call(x, pb[:-1])),
        "packed of another type": (False, call(x, pb.view(torch.int8))),
        "a small C": (False, call(x, pb, rows=M - 1)),
        "a narrow C": (False, call(x, pb, cols=N - 1)),
        "a C of doubles": (False, call(x, pb, dt=torch.float64)),
        "a short bias": (False, call(x, pb, steps=2, ep=short)),
        "columns behind the end": (False, call(x, pb, n0=32, n1=N + 32)),
        "no columns": (False, call(x, pb, n0=64, n1=64)),
        "a bias of another type": (False, call(x, pb, steps=0, edit=lambda e: setattr(e, "bias", bias.double()))),
        "A on the CPU": (False, call(x.cpu(), pb)),
        "a vector": (False, call(x[0], pb)),
        "a workspace of floats": (False, call(x, pb, ws=ws.view(torch.float32))),
    }


NAMES = ["bf16", "post-op", "scales of columns", "int32", "int8 weights", "int4 weights", "some columns", "a row", "a row of any stride",
         "rows with gaps", "a workspace", "two slices", "unsplit", "an error of the library", "a parameter",
         "a count of slices without a workspace", "a numpy N", "columns of A", "fp32 A", "too few packed bytes", "packed of another type",
         "a small C", "a narrow C", "a C of doubles", "a short bias", "columns behind the end", "no columns", "a bias of another type",
         "A on the CPU", "a vector", "a workspace of floats"]


@pytest.mark.parametrize("name", NAMES)
def test_gemm(monkeypatch, name):
    taken, call = _gemm_calls()[name]
    (native, python), answers = _both(monkeypatch, call)
    assert native[1] == python[1] and np.array_equal(native[0], python[0]), (native, python)
    assert all((a is not None) == taken for a in answers) and (answers or not taken), answers


def test_first_call_that_wants_a_workspace(monkeypatch):
    """Without the stream's workspace a call that splits K is left to the Python form, which makes it; the next one is taken."""
    x, W = _bf(40, 8192), _bf(224, 8192)
    packed, C = mx.repack_b(W, transpose=True), torch.zeros((40, 224), device="cuda")
    L.release_workspaces()
    watch = _Watch(L._native)
    monkeypatch.setattr(L, "_native", watch)
    outs = []
    for _ in range(2):
        mx.gemm(x, packed, 224, mx.Epilogue(C))
        assert "ksplit" in mx.last_kernel()
        outs.append(host_bits(C).copy())
    assert watch.answers == [None, 0] and np.array_equal(*outs)


@pytest.mark.parametrize("M,K,N,trans,taken", [(1, 256, 96, False, True), (4, 512, 512, True, True), (32, 8192, 512, False, True),
                                               (7, 300, 70, False, False), (900, 512, 512, False, False)])
def test_unpacked(monkeypatch, M, K, N, trans, taken):
    x, B = _bf(M, K), _bf(N, K) if trans else _bf(K, N)
    mx.workspace()
    bias = torch.randn(N, device="cuda")

    def call():
        y = torch.zeros((M, N + 3), device="cuda")
        pp = mx.BiasGeluStore(y[:, :N], mx.Steps.BIAS, bias)
        mx.Matmul(False, trans)(x, B, ppkernel=pp)
        return y
    (native, python), answers = _both(monkeypatch, call)
    assert native[1] == python[1] and np.array_equal(native[0], python[0])
    assert (answers[0] is not None) == taken, answers
    # a result that lies over B, and operands that do not fit together
    if taken:
        wide = torch.zeros((max(M, K, N), max(K, N) * 4), dtype=torch.bfloat16, device="cuda")
        over = wide[:B.shape[0], :B.shape[1]]
        watch = _Watch(_host_call)
        monkeypatch.setattr(L, "_native", watch)
        over.copy_(B)
        assert not L.gemm_unpacked(x, over, trans, mx.Epilogue(wide[:M, :N])) and watch.answers == [None]
        with pytest.raises(L.MmxError, match="differ"):
            L.gemm_unpacked(x[:, :-1], B, trans, mx.Epilogue(torch.zeros((M, N), device="cuda")))


@pytest.mark.parametrize("M,K,N,trans", [(300, 288, 1440, True), (700, 96, 201, True), (300, 200, 70, False), (300, 8192, 64, True)])
def test_packed_and_used_once(monkeypatch, M, K, N, trans):
    """Where the library would have B packed first both launches are one native call, on any rows and columns; what it cannot say is left
    to the Python form: a workspace that the stream does not have yet, operands that do not fit together."""
    x, B, bias = _bf(M, K + 3)[:, :K], _bf(N, K) if trans else _bf(K, N), torch.randn(N, device="cuda")
    op = mx.Matmul(False, trans)

    def call():
        y = torch.zeros((M, N + 3), device="cuda")
        op(x, B, ppkernel=mx.BiasGeluStore(y[:, :N], mx.Steps.BIAS, bias))
        return y
    mx.workspace()
    (native, python), answers = _both(monkeypatch, call)
    assert native[1] == python[1] and np.array_equal(native[0], python[0])
    assert answers[0] is None and isinstance(answers[1], torch.Tensor) and len(answers) == 2, answers
    assert torch.equal(op.internalB, mx.repack_b(B, transpose=trans))
    needs = mx.gemm_workspace_bytes(mx.BF16, mx.BF16, M, K, N) > 0
    L.release_workspaces()
    watch = _Watch(_host_call)
    monkeypatch.setattr(L, "_native", watch)
    assert np.array_equal(host_bits(call()), native[0]) and isinstance(watch.answers[1], torch.Tensor) == (not needs), watch.answers
    with pytest.raises(L.MmxError, match="differ"):
        L.gemm_once(x[:, :-1], B, trans, mx.Epilogue(torch.zeros((M, N), device="cuda")))


@pytest.mark.parametrize("kind", ["bf16", "i8"])
def test_matvec(monkeypatch, kind):
    M, K = 100, 96
    new = _bf if kind == "bf16" else lambda *s: torch.randint(-127, 128, s, device="cuda", dtype=torch.int8)
    A, b, dt = new(M, K + 5), new(K), torch.float32 if kind == "bf16" else torch.int32
    for taken, rows, vec, size, out_dt in ((True, A[:, :K], b, M, dt), (True, A[:1, :K], b, M, dt), (False, A[:, :K], b[:-1], M, dt),
                                           (False, A[:, :K], b, M - 1, dt), (False, A[:, :K], b, M, torch.float64), (False, A[:, :K].t(), b, M, dt)):
        with monkeypatch.context() as m:
            (native, python), answers = _both(m, lambda: mx.MatmulVector()(rows, vec, torch.zeros(size, dtype=out_dt, device="cuda")))
        assert native[1] == python[1] and np.array_equal(native[0], python[0])
        assert [a is not None for a in answers] == [taken], answers


def test_matvec_initialises_its_device(monkeypatch):
    """The first call on a GPU asks the library whether it has code for it, before anything is launched there."""
    A, b, out = _bf(64, 96), _bf(96), torch.zeros(64, device="cuda")
    mx.lib()
    watch = _Watch(L._native)
    monkeypatch.setattr(L, "_native", watch)
    monkeypatch.setattr(L, "_initialised", set())
    mx.matvec(A, b, out)
    assert L._initialised == {torch.cuda.current_device()} and not watch.answers
    mx.matvec(A, b, out)
    assert watch.answers == [0]


@pytest.mark.parametrize("K,N", [(1, 1), (96, 33), (257, 130)])
def test_packing(monkeypatch, K, N):
    """repack_b and the quantisers: the same bytes, types and shapes either way, and the same refusals."""
    mx.init(0)
    mx.lib()
    whole, i8 = _bf(N + 1, K + 4), torch.randint(-127, 128, (N, K), device="cuda", dtype=torch.int8)
    W = whole[1:, 3:K + 3]  # rows with gaps, at an odd address
    calls = [(True, lambda: mx.repack_b(W, transpose=True)), (True, lambda: mx.repack_b(W)), (True, lambda: mx.repack_b(i8, transpose=True)),
             (True, lambda: mx.repack_b(i8.view(torch.uint8))), (True, lambda: mx.quantize_weights(W)), (True, lambda: mx.quantize_weights(W.contiguous())),
             (True, lambda: L.quantize_weights_scaled(W, 100.0)), (True, lambda: mx.quantize_pack_int4(W, transpose=True)), (True, lambda: mx.quantize_pack_int4(W)),
             (False, lambda: mx.repack_b(W, transpose=1)), (False, lambda: mx.repack_b(W.float())), (False, lambda: mx.quantize_weights(W.float())),
             (False, lambda: mx.quantize_weights(W.cpu())), (False, lambda: L.quantize_weights_scaled(W[0], 100.0)), (False, lambda: mx.quantize_pack_int4(i8)),
             (False, lambda: mx.quantize_weights(whole[:, :0]))]
    for n, (taken, call) in enumerate(calls):
        watch, got = _Watch(_host_call), []
        for native in (watch, None):
            monkeypatch.setattr(L, "_native", native)
            try:
                r = call()
                got.append([(t.dtype, tuple(t.shape), t.stride(), host_bits(t).tobytes()) for t in (r if isinstance(r, tuple) else (r,))])
            except L.MmxError as e:
                got.append(str(e))
        assert got[0] == got[1], (n, got[0][:200], got[1][:200])
        assert [a is not None for a in watch.answers] == [taken], n
