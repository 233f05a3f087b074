"""NaN and infinity in the FP16 / BF16 split path: every element of C whose row of A or row of
B holds one is NaN, as in the form with a workgroup per problem (pipeline 1), and every other
element has the bits it has without them.  One case for each tile form of the default path."""
import numpy as np
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SPLITS = [(K.PREC_F64_SPLIT_F16, 6), (K.PREC_F64_SPLIT_F16, 7), (K.PREC_F64_SPLIT_BF16, 7)]
# 32-wide, 64-wide (128 units or more) and 128-wide tiles; the last two are block shapes too
FORMS = [(1, 64, 192, 64), (130, 64, 64, 64), (256, 128, 128, 128)]


@pytest.mark.parametrize("prec,slices", SPLITS, ids=["f16-s6", "f16-s7", "bf16-s7"])
@pytest.mark.parametrize("shape", FORMS, ids=lambda s: "x".join(map(str, s)))
def test_nonfinite_rows_reach_c(shape, prec, slices, dev):
    print(f"\n[case] {shape} {prec} {slices}", flush=True)
    count, m, n, k = shape
    rng = np.random.default_rng(k)
    A = torch.from_numpy(rng.uniform(-1, 1, (count, m, k))).to(dev)
    B = torch.from_numpy(rng.uniform(-1, 1, (count, n, k))).to(dev)
    clean = K.split_gemm(A, B, precision=prec, slices=slices)
    B[0, 9, 2] = 0.0
    A[0, 3, 5], A[0, 17, k - 1], A[count - 1, 40, 31] = float("nan"), float("inf"), -float("inf")
    B[0, 7, 33], B[count - 1, 63, 0] = float("inf"), float("nan")
    bad = ~torch.isfinite(A).all(2)[:, :, None] | ~torch.isfinite(B).all(2)[:, None, :]
    C = K.split_gemm(A, B, precision=prec, slices=slices)
    assert torch.equal(torch.isnan(C), bad)
    same = ~bad
    same[0, :, 9] = False
    assert torch.equal(C[same], clean[same])
    if m == n == k:
        assert torch.equal(torch.isnan(K.block_gemm(A, B, precision=prec, slices=slices)), bad)
        assert torch.equal(torch.isnan(K.block_gemm(A, B, precision=prec, slices=slices, pipeline=1)), bad)
