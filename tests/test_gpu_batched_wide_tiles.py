"""Batched GEMM through the largest wave tiles (64 x 64 for 2-byte inputs, 64 x 32 for FP64): queues
long enough for them with K around 128, problems whose last strips leave one to three atoms, both
layouts, and a
queue too short for them.  Small integers make every sum exact (|sums| <= 4 K < 2^24), so each
problem equals the FP64 product."""
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [(64, 64, 128), (128, 192, 144), (80, 112, 160), (144, 208, 128), (96, 176, 272), (16, 256, 400),
          (256, 48, 192), (240, 224, 208)]


@pytest.mark.parametrize("count", [250, 1400], ids=["short", "long"])
@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float16, torch.bfloat16], ids=["f64", "f16", "bf16"])
def test_wide_tiles_exact(dtype, layout, count, dev):
    print(f"\n[case] {dtype} {layout} x{count}", flush=True)
    g = torch.Generator(device=dev).manual_seed(count)
    ints = lambda r, c: torch.randint(-2, 3, (r, c), generator=g, device=dev)  # noqa: E731
    probs, refs = [], []
    for i in range(count):
        m, n, k = SHAPES[i % len(SHAPES)]
        A = ints(m, k).to(dtype)
        B = (ints(n, k) if layout == "nk" else ints(k, n)).to(dtype)
        C = ints(m, n).to(torch.float64 if dtype == torch.float64 else torch.float32)
        refs.append(2.0 * (A.double() @ (B.double().t() if layout == "nk" else B.double())) - C.double())
        probs.append((A, B, C))
    with K.BatchedPlan(probs, b_layout=layout, alpha=2.0, beta=-1.0) as plan:
        plan.execute()
    for (_, _, C), ref in zip(probs, refs):
        assert torch.equal(C.double(), ref)
