"""Block GEMM with B stored K x N, every compiled partition of every shape, streaming and
repeated: exact on small integers against an FP64 product, and on random values the bits of the
N x K layout through the same instance (the same products in the same order)."""
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

LOW = [(e, e, k) for e in (16, 32, 64, 128, 192, 208, 224, 256) for k in {16, 32, e, 512}]
SHAPES = {"f64": [(e, e, e) for e in (16, 32, 64, 128)] + [(64, 64, 512), (128, 128, 512)], "f16": LOW, "bf16": LOW}
PREC = {"f64": (K.PREC_F64, torch.float64), "f16": (K.PREC_F16_F32, torch.float16),
        "bf16": (K.PREC_BF16_F32, torch.bfloat16)}


def forms(prec, m, n, k):
    for part in ("1d", "2d", "3d"):
        for ranks in (1, 2, 4, 8, 12, 13, 14, 16):
            try:
                K.query(m, n, k, prec, partition=part, ranks=ranks)
            except K.KamiError:
                continue
            yield part, ranks


@pytest.mark.parametrize("name,shape", [(p, s) for p in SHAPES for s in SHAPES[p] if list(forms(PREC[p][0], *s))],
                         ids=str)
def test_kn_exact_and_as_nk(name, shape, dev):
    print(f"\n[case] {name} {shape}", flush=True)
    prec, dt = PREC[name]
    m, n, k = shape
    g = torch.Generator().manual_seed(m + k)
    A = torch.randint(-3, 4, (3, m, k), generator=g).double()
    B = torch.randint(-3, 4, (3, k, n), generator=g).double()
    ref = (A @ B).to(dev)
    R, S = torch.randn((3, m, k), generator=g).to(dt).to(dev), torch.randn((3, k, n), generator=g).to(dt).to(dev)
    St = S.transpose(1, 2).contiguous()
    A, B = A.to(dt).to(dev), B.to(dt).to(dev)
    for part, ranks in forms(prec, m, n, k):
        for iters in (1, 3):
            kw = dict(partition=part, ranks=ranks, iters=iters)
            out = K.block_gemm(A, B, b_layout="kn", **kw)
            assert torch.equal(out.double(), iters * ref), kw
            nk = K.block_gemm(R, St, pipeline=1, **kw)
            for pipe in (0, 1):
                assert torch.equal(K.block_gemm(R, S, b_layout="kn", pipeline=pipe, **kw), nk), (kw, pipe)
    if name == "f64":  # more problems than the persistent form has workgroups; alpha, beta
        if m * k <= 64 * 64:
            A, B = A[:1].repeat(5000, 1, 1), B[:1].repeat(5000, 1, 1)
            A[1::2] *= 2
            out = K.block_gemm(A, B, torch.ones((5000, m, n), dtype=dt, device=dev), b_layout="kn", alpha=3.0, beta=-1.0)
            assert torch.equal(out[::2], (3 * ref[0] - 1).expand(2500, m, n))
            assert torch.equal(out[1::2], (6 * ref[0] - 1).expand(2500, m, n))
