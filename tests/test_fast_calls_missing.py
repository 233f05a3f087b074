"""Without the native call path's extension every call is the wrapper's own, after one warning."""
import sys
import warnings

import pytest

import kami_amd as K

torch = pytest.importorskip("torch")


@pytest.fixture
def without_extension(monkeypatch):
    monkeypatch.setitem(sys.modules, "kami_amd._fast_calls", None)  # importing it raises ImportError
    monkeypatch.delattr(K, "_fast_calls", raising=False)
    monkeypatch.setattr(K, "_FAST", None)
    with pytest.warns(RuntimeWarning, match="native call path"):
        yield K._fast()


def test_one_warning_and_the_wrappers_checks(without_extension):
    a = torch.zeros(2, 64, 64, dtype=torch.float64)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        with pytest.raises(ValueError, match="GPU tensor"):
            K.block_gemm(a, a)


@pytest.mark.gpu
def test_calls_run_without_it(without_extension, dev):
    A = torch.randn(2, 64, 64, dtype=torch.float64, device=dev)
    here = torch.cuda.current_stream()
    assert torch.equal(K.block_gemm(A, A), K.block_gemm(A, A, stream=here))
    assert torch.equal(K.split_gemm(A, A), K.split_gemm(A, A, stream=here))
    C = torch.empty(64, 64, dtype=torch.float64, device=dev)
    with K.BatchedPlan([(A[0], A[0], C)]) as plan:
        plan.execute()
        assert torch.isfinite(C).all()
    S = K.BsrMatrix(1, 1, 16, torch.tensor([0, 1], dtype=torch.int32, device=dev),
                    torch.zeros(1, dtype=torch.int32, device=dev),
                    torch.ones(1, 16, 16, dtype=torch.float64, device=dev))
    assert torch.equal(K.bsr_spgemm(S, S).vals[0], K.bsr_spmm(S, S.vals[0]))
