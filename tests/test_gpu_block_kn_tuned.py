"""kami_block_gemm_autotune with B stored K x N: the persistent FP64 form is among what it times,
and the choice it reports is the form of the next AUTO call (whose bits no form changes)."""
import ctypes

import pytest

import kami_amd as K
from kami_amd import _abi

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("edge,count", [(32, 64), (64, 300), (128, 600)])
def test_tuned_choice(edge, count, dev):
    print(f"\n[case] {edge} x {count}", flush=True)
    g = torch.Generator().manual_seed(edge)
    A, B = (torch.rand((count, edge, edge), generator=g, dtype=torch.float64).to(dev) for _ in range(2))
    C = torch.empty_like(A)
    ref = K.block_gemm(A, B.transpose(1, 2).contiguous())
    d = K.make_desc(edge, edge, edge, K.PREC_F64, b_layout="kn")
    chosen = _abi.GemmConfig()
    try:
        st = K.lib().kami_block_gemm_autotune(ctypes.byref(d), A.data_ptr(), B.data_ptr(), C.data_ptr(),
                                              count, torch.cuda.current_stream().cuda_stream,
                                              ctypes.byref(chosen))
        assert st == _abi.OK
        assert chosen.as_dict() == K.query(edge, edge, edge, K.PREC_F64, b_layout="kn")
        assert torch.equal(K.block_gemm(A, B, b_layout="kn"), ref)
    finally:
        K.lib().kami_tune_clear()
