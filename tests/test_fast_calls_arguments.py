"""Arguments that the wrappers refuse are refused by the native call path too."""
import pytest

import kami_amd as K

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [-1, -2, 6, 1 << 40, "f64", 0.5])
def test_an_unknown_precision_is_refused(prec, dev):
    print(f"\n[case] {prec!r}", flush=True)
    A = torch.zeros(2, 64, 64, dtype=torch.float64, device=dev)
    S = K.BsrMatrix(1, 1, 16, torch.tensor([0, 1], dtype=torch.int32, device=dev),
                    torch.zeros(1, dtype=torch.int32, device=dev),
                    torch.zeros(1, 16, 16, dtype=torch.float64, device=dev))
    here = torch.cuda.current_stream()
    for call in (lambda **kw: K.block_gemm(A, A, precision=prec, **kw),
                 lambda **kw: K.split_gemm(A, A, precision=prec, **kw),
                 lambda **kw: K.bsr_spmm(S, A[0, :, :16].contiguous(), precision=prec, **kw),
                 lambda **kw: K.bsr_spgemm(S, S, precision=prec, **kw)):
        with pytest.raises(Exception) as with_stream:
            call(stream=here)
        with pytest.raises(type(with_stream.value)) as plain:
            call()
        assert str(plain.value) == str(with_stream.value)


@pytest.mark.gpu
def test_split_gemm_needs_a_precision(dev):
    A = torch.zeros(64, 64, dtype=torch.float64, device=dev)
    for stream in (None, torch.cuda.current_stream()):
        with pytest.raises(Exception):
            K.split_gemm(A, A, precision=None, stream=stream)
