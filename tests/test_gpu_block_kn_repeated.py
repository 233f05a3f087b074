"""Repeated products with B stored K x N: from eight repetitions on, and in the resident forms, the
K rows are turned when they are written to LDS.  Exact on small integers, and the bits of the
N x K layout on random values, for every compiled form."""
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [(e, e, e) for e in (16, 32, 64, 128, 192, 208, 224, 256)] + \
         [(e, e, k) for e in (32, 64, 128, 192, 256) for k in (16, 32)] + [(128, 128, 512)]
TYPES = {"f64": (K.PREC_F64, torch.float64), "f16": (K.PREC_F16_F32, torch.float16),
         "bf16": (K.PREC_BF16_F32, torch.bfloat16)}


def forms(prec, m, n, k, iters):
    yield {}
    for part in ("1d", "2d", "3d"):
        for ranks in (1, 2, 4, 8, 12, 13, 14, 16):
            try:
                K.query(m, n, k, prec, partition=part, ranks=ranks, iters=iters, b_layout="kn")
            except K.KamiError:
                continue
            yield dict(partition=part, ranks=ranks)


@pytest.mark.parametrize("name", list(TYPES))
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_repeated_kn(shape, name, dev):
    m, n, k = shape
    prec, dt = TYPES[name]
    try:
        K.query(m, n, k, prec)
    except K.KamiError:
        return
    print(f"\n[case] {name} {shape}", flush=True)
    g = torch.Generator().manual_seed(m + k)
    A = torch.randint(-2, 3, (3, m, k), generator=g).double()
    B = torch.randint(-2, 3, (3, k, n), generator=g).double()
    ref = (A @ B).to(dev)
    A, B = A.to(dt).to(dev), B.to(dt).to(dev)
    R, S = torch.randn((3, m, k), generator=g).to(dt).to(dev), torch.randn((3, k, n), generator=g).to(dt).to(dev)
    St = S.transpose(1, 2).contiguous()
    for iters in (2, 7, 8, 9):
        for kw in forms(prec, m, n, k, iters):
            out = K.block_gemm(A, B, b_layout="kn", iters=iters, **kw)
            assert torch.equal(out.double(), iters * ref), (iters, kw)
            assert torch.equal(K.block_gemm(R, S, b_layout="kn", iters=iters, **kw),
                               K.block_gemm(R, St, iters=iters, **kw)), (iters, kw)
