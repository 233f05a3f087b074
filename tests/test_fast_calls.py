"""The native call path of the Python wrappers (kami_amd/host/fast_calls.cpp) takes plain calls
only and leaves every other to the wrapper's own checks.  On the CPU: whatever is not a
plain GPU call is answered with None, so the wrappers' errors are the same with it as
without.  On the GPU: a call through it equals, bit for bit, the same call with its stream
named (which takes the wrapper's own path)."""
import ctypes

import numpy as np
import pytest

import kami_amd as K

torch = pytest.importorskip("torch")


class Sub(torch.Tensor):
    pass


def block_args(A, B, C=None, prec=-1, lay=K.B_NK, iters=1, tiled=0):
    return (A, B, C, prec, 0, 0, lay, iters, 1.0, 0.0, 0, 0, tiled)


def test_everything_but_a_plain_gpu_call_is_left_to_the_wrapper():
    f = K._fast()
    a = torch.zeros(2, 64, 64, dtype=torch.float64)
    for args in [(), (a,), block_args(a, a), block_args(1, 2), block_args(None, a), block_args(a, a, a),
                 block_args(a.as_subclass(Sub), a), block_args(a, a, prec="x"), block_args(a, a, lay=None),
                 block_args(a.to_sparse(), a), block_args(a, a, iters=1 << 40)]:
        assert f.block_gemm(*args) is None
    i = torch.zeros(3, dtype=torch.int32)
    bsr = (2, 2, 16, i, i[:1], torch.zeros(1, 16, 16, dtype=torch.float64))
    assert f.bsr_spmm(*bsr, a[0], None, 0, -1, 1.0, 0.0) is None
    assert f.bsr_spmm(*bsr[:3]) is None
    assert f.bsr_spgemm(*bsr, *bsr, -1, 1.0) is None
    assert f.bsr_spgemm("a", *bsr[1:], *bsr, -1, 1.0) is None
    assert f.batched_execute("x") is None and f.batched_execute(0) is None
    with pytest.raises(TypeError):
        f.bind(1, 2)


def vmapped(x):
    return torch.func.vmap(lambda a: K.block_gemm(a, a))(x)


def test_a_tensor_without_an_address_raises_as_before():
    with pytest.raises((RuntimeError, ValueError)):
        vmapped(torch.zeros(3, 64, 64, dtype=torch.float64))


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["f64", "f16", "bf16"])
def test_same_results_as_the_wrappers_own_path(prec, dev):
    print(f"\n[case] {prec}", flush=True)
    dt = {"f64": torch.float64, "f16": torch.float16, "bf16": torch.bfloat16}[prec]
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    rand = lambda *s: torch.randn(s, generator=g, device=dev, dtype=torch.float64).to(dt)  # noqa: E731
    here = torch.cuda.current_stream()
    A, B = rand(5, 64, 64), rand(5, 64, 64)
    for kw in ({}, {"b_layout": "kn"}, {"alpha": 2.0}, {"partition": "2d", "ranks": 2}, {"iters": 3}):
        assert torch.equal(K.block_gemm(A, B, **kw), K.block_gemm(A, B, stream=here, **kw))
        assert torch.equal(K.block_gemm(A[0], B[0], **kw), K.block_gemm(A[0], B[0], stream=here, **kw))
    C = K.block_gemm(A, B)
    D = C.clone()
    assert K.block_gemm(A, B, C, beta=1.0) is C
    K.block_gemm(A, B, D, beta=1.0, stream=here)
    assert torch.equal(C, D)
    if prec == "f64":
        X, Y = rand(2, 64, 96), rand(2, 128, 96)
        assert torch.equal(K.split_gemm(X, Y), K.split_gemm(X, Y, stream=here))
    # the call runs on the stream that is current
    other = torch.cuda.Stream()
    other.wait_stream(here)
    with torch.cuda.stream(other):
        E = K.block_gemm(A, B)
    here.wait_stream(other)
    assert torch.equal(E, K.block_gemm(A, B))
    probs = [(A[0], B[0], torch.empty(64, 64, dtype=C.dtype, device=dev))]
    with K.BatchedPlan(probs) as plan:
        plan.execute()
        first = probs[0][2].clone()
        plan.execute(here)
        assert torch.equal(first, probs[0][2])
    with pytest.raises(K.KamiError):
        plan.execute()
    rp = torch.tensor([0, 2, 2, 3], dtype=torch.int32, device=dev)
    ci = torch.tensor([0, 2, 1], dtype=torch.int32, device=dev)
    S = K.BsrMatrix(3, 3, 16, rp, ci, rand(3, 16, 16))
    W = rand(32, 48)
    assert torch.equal(K.bsr_spmm(S, W), K.bsr_spmm(S, W, stream=here))
    P, Q = K.bsr_spgemm(S, S), K.bsr_spgemm(S, S, stream=here)
    for x, y in ((P.rowptr, Q.rowptr), (P.colidx, Q.colidx), (P.vals, Q.vals)):
        assert torch.equal(x, y) and x.shape == y.shape
    # no output blocks; and operands that the checks refuse
    N = K.BsrMatrix(3, 3, 16, torch.tensor([0, 1, 1, 1], dtype=torch.int32, device=dev),
                    torch.tensor([2], dtype=torch.int32, device=dev), rand(1, 16, 16))
    Z = K.bsr_spgemm(N, N)
    assert Z.nnzb == 0 and tuple(Z.vals.shape) == (0, 16, 16)
    with pytest.raises(ValueError):
        K.block_gemm(A, B.transpose(1, 2))
    with pytest.raises(ValueError):
        K.bsr_spmm(S, W[:, :40])
    with pytest.raises(K.KamiError):
        K.block_gemm(rand(1, 48, 48), rand(1, 48, 48))
    P1 = torch.nn.Parameter(A, requires_grad=False)
    assert torch.equal(K.block_gemm(P1, B), K.block_gemm(A, B))
