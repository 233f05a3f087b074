"""Split-precision FP64 in each tile form of the persistent kernels: 32 x 32 tiles (few
units), 64 x 64 (from 128 units on) and 128 x 128 (where its rounds over the chip are fewer),
with one and with several K chunks.  Integer inputs are exact in every form; the 32- and
64-wide forms take the same chunks, digits and order, so a problem's result is the same
bits however many others run beside it; and every form stays within 1e-13 of the Dot2
product, also for rows whose scaling reaches the ends of the exponent range."""
import numpy as np
import pytest

import kami_amd as K
import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SPLITS = [(K.PREC_F64_SPLIT_F16, 6), (K.PREC_F64_SPLIT_F16, 7), (K.PREC_F64_SPLIT_BF16, 7)]
SIDS = ["f16-s6", "f16-s7", "bf16-s7"]


def product(A, B, prec, slices, dev):
    return K.split_gemm(torch.from_numpy(A).to(dev), torch.from_numpy(B).to(dev), precision=prec,
                        slices=slices).cpu().numpy()


# (count, m, n, k): 32-wide, 64-wide (128 units, ragged tile grid), 128-wide (1024 units)
FORMS = [(1, 64, 192, 32), (1, 64, 64, 352), (2, 576, 512, 32), (130, 64, 64, 96), (256, 128, 128, 64)]


@pytest.mark.parametrize("prec,slices", SPLITS, ids=SIDS)
@pytest.mark.parametrize("shape", FORMS, ids=lambda s: "x".join(map(str, s)))
def test_forms_integer_exact(shape, prec, slices, dev):
    print(f"\n[case] {shape} {prec} {slices}", flush=True)
    count, m, n, k = shape
    rng = np.random.default_rng(k)
    A = rng.integers(-1000, 1001, (count, m, k)).astype(np.float64)
    B = rng.integers(-1000, 1001, (count, n, k)).astype(np.float64)
    np.testing.assert_array_equal(product(A, B, prec, slices, dev), oracle.gemm_f64(A, B))


@pytest.mark.parametrize("prec,slices", SPLITS, ids=SIDS)
def test_forms_agree_and_meet_the_bound(prec, slices, dev):
    rng = np.random.default_rng(3)
    count, s, k = 256, 128, 96
    A = np.where(rng.random((count, s, k)) < 0.5, -1.0, 1.0) * 10.0 ** rng.uniform(-4, 4, (count, s, k))
    B = np.where(rng.random((count, s, k)) < 0.5, -1.0, 1.0) * 10.0 ** rng.uniform(-4, 4, (count, s, k))
    A[0, 3] *= 2.0 ** -1000  # tiny, subnormal, huge and zero rows
    A[0, 4] = rng.integers(-50, 51, k) * 2.0 ** -1074
    A[0, 5] *= 1e280
    B[0, 6] = 0.0
    A[1, 7, :] = np.nextafter(1.0, 0.0)  # rounds up to the next power of two
    wide = product(A, B, prec, slices, dev)                 # 128-wide
    some = product(A[:40], B[:40], prec, slices, dev)       # 64-wide
    few = product(A[:4], B[:4], prec, slices, dev)          # 32-wide
    np.testing.assert_array_equal(few, some[:4])
    exact, mag = oracle.gemm_dot2(A[:4], B[:4])
    top = np.max(np.abs(A[:4]), axis=2)[:, :, None] * np.max(np.abs(B[:4]), axis=2)[:, None, :]
    for C in (few, wide[:4]):
        # digits leave at most 2^-(BETA S) of the row maxima per term, with six digits or
        # BF16's seven (54 and 56 bits) as with seven; the sums' own rounding is beside it
        bits = {6: 54, 7: 63}[slices] if prec == K.PREC_F64_SPLIT_F16 else 56
        tol = 4 * k * 2.0 ** -bits * top + 8 * k * 2.0 ** -53 * mag + 2.0 ** -1070
        assert np.all(np.abs(C - exact) <= tol)
