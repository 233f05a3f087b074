"""Int8 split GEMM with rows on both sides of the exponents from which rows are scaled before
they are cut: scaling a row by a power of two scales its results exactly, so the bits are those
of the unscaled product.  And the precision of the cut itself: entries down to 2^-62 of the
row's largest count, rounded to nearest."""
import numpy as np
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def run(A, B, dev):
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)  # noqa: E731
    return K.block_gemm(t(A), t(B), precision=K.PREC_F64_SPLIT_I8).cpu().numpy()


@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("s", [64, 128])
def test_scaled_rows_keep_their_bits(s, swap, dev):
    print(f"\n[case] {s} {swap}", flush=True)
    rng = np.random.default_rng(s)
    A, B = rng.uniform(0.5, 1, (3, s, s)), rng.uniform(-1, 1, (3, s, s))
    big = rng.choice([950, 959, 960, 961, 970, 1015, 0], (3, s, 1))
    small = rng.choice([-950, -959, -960, -961, -965, -15, -16], (3, s, 1))
    ref = np.ldexp(run(A, B, dev), big + small.transpose(0, 2, 1))
    X, Y = np.ldexp(A, big), np.ldexp(B, small)
    C = run(Y, X, dev).transpose(0, 2, 1) if swap else run(X, Y, dev)
    if swap:
        ref = np.ldexp(run(B, A, dev).transpose(0, 2, 1), big + small.transpose(0, 2, 1))
    np.testing.assert_array_equal(C, ref)


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("s", [64, 128])
def test_units_of_a_row(s, sign, dev):
    A = np.zeros((1, s, s))
    A[0, :, 0] = 0.75  # |x| < 2^0: units of 2^-62
    A[0, :, 1] = sign * 2.0 ** -62 * np.resize([0.25, 0.75, 1.0, 1.25, 129.0, 2.0 ** 31, 2.0 ** 32 - 1], s)
    B = np.zeros((1, s, s))
    B[0, 3, 1] = 1.0  # picks the small entries alone
    want = np.rint(A[0, :, 1] * 2.0 ** 62) * 2.0 ** -62
    np.testing.assert_array_equal(run(A, B, dev)[0, :, 3], want)
