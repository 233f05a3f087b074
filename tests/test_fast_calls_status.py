"""What the native call path does with a library call's status: an error of the HIP runtime is
raised after one call (work may be enqueued by then, and a second call would add to C twice);
a call that the library refuses before it launches anything is left to the wrapper.  Entry points
are replaced by functions that count their calls."""
import ctypes

import pytest

import kami_amd as K
from kami_amd import _abi

torch = pytest.importorskip("torch")

NAMES = ["block_gemm", "split_gemm", "batched_execute", "symbolic", "fill", "numeric", "spmm", "structure"]


@pytest.fixture
def stub():
    f, real, keep = K._fast(), K._fast_entry_points(), []

    def bind(**by_name):
        at = list(real)
        for name, fn in by_name.items():
            keep.append(fn)
            at[NAMES.index(name)] = ctypes.cast(fn, ctypes.c_void_p).value
        f.bind(K.check, *at)
    yield bind
    f.bind(K.check, *real)


def counting(n_args, status, calls):
    def fn(*args):
        calls.append(status)
        return status
    return ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_void_p] * n_args)(fn)


def test_bind_wants_a_check_and_eight_addresses():
    f = K._fast()
    for args in [(), tuple(range(1, 9)), (1, *range(1, 9)), (K.check, 0, *range(1, 8))]:
        with pytest.raises((TypeError, ValueError)):
            f.bind(*args)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["block_gemm", "split_gemm", "batched_execute", "spmm", "structure"])
def test_a_hip_error_is_raised_after_one_call(name, stub, dev):
    print(f"\n[case] {name}", flush=True)
    A = torch.ones(1, 64, 64, dtype=torch.float64, device=dev)
    C = torch.ones(1, 64, 64, dtype=torch.float64, device=dev)
    S = K.BsrMatrix(1, 1, 16, torch.tensor([0, 1], dtype=torch.int32, device=dev),
                    torch.zeros(1, dtype=torch.int32, device=dev),
                    torch.ones(1, 16, 16, dtype=torch.float64, device=dev))
    W = torch.ones(16, 16, dtype=torch.float64, device=dev)
    plan = K.BatchedPlan([(A[0], A[0], C[0])])
    run = {"block_gemm": lambda: K.block_gemm(A, A, C, beta=1.0), "split_gemm": lambda: K.split_gemm(A, A, C, beta=1.0),
           "batched_execute": plan.execute, "spmm": lambda: K.bsr_spmm(S, W, W.clone(), beta=1.0),
           "structure": lambda: K.bsr_spgemm(S, S)}[name]
    n_args = {"block_gemm": 9, "split_gemm": 9, "batched_execute": 2, "spmm": 11, "structure": 9}[name]
    calls = []
    stub(**{name: counting(n_args, _abi.EHIP, calls)})
    with pytest.raises(K.KamiError) as e:
        run()
    assert e.value.status == _abi.EHIP and calls == [_abi.EHIP]
    assert torch.equal(C, torch.ones_like(C))  # no call of the wrapper's own either
    # refused before any launch: the wrapper makes the call, and it succeeds
    calls.clear()
    stub(**{name: counting(n_args, _abi.ENOTSUP, calls)})
    run()
    assert calls == [_abi.ENOTSUP]
    plan.close()
