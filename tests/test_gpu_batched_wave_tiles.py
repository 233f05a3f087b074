"""Batched GEMM at the edges of its wave tiles: every count of 16 x 16 atoms a wave tile can
hold, K at and beside the ends of its 128-byte stages (16 FP64 or 64 FP16 / BF16 values),
both layouts of B, C at any element offset, and queues on both sides of the length below
which wave tiles are made smaller (4096 of them).  Integer inputs make every sum exact, so
each problem equals the oracle's triple loop bit for bit (|sums| <= 4 K < 2^24)."""
import numpy as np
import pytest

import kami_amd as K
import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

EDGES = [(m, n, k) for m, n in [(16, 16), (16, 48), (32, 16), (48, 32), (80, 112), (144, 16), (16, 144),
                                (208, 144)] for k in (16, 32, 48, 64, 80, 144)]


@pytest.mark.parametrize("repeat", [1, 40], ids=["short", "long"])
@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float16, torch.bfloat16], ids=["f64", "f16", "bf16"])
def test_wave_tile_edges_exact(dtype, layout, repeat, dev):
    print(f"\n[case] {dtype} {layout} x{repeat}", flush=True)
    rng = np.random.default_rng(5)
    out = torch.float64 if dtype == torch.float64 else torch.float32
    probs, refs = [], []
    for m, n, k in EDGES:
        A = rng.integers(-2, 3, (m, k)).astype(np.float64)
        B = rng.integers(-2, 3, (n, k)).astype(np.float64)
        C0 = rng.integers(-4, 5, (m, n)).astype(np.float64)
        At = torch.from_numpy(A).to(dev).to(dtype)
        Bt = torch.from_numpy(B if layout == "nk" else np.ascontiguousarray(B.T)).to(dev).to(dtype)
        for r in range(repeat):
            pool = torch.full((m * n + 8,), 7.0, dtype=out, device=dev)
            off = (len(probs) + r) % 4  # C needs only its element's alignment
            C = pool[off:off + m * n].view(m, n)
            C.copy_(torch.from_numpy(C0))
            probs.append((At, Bt, C, pool, off))
            refs.append(2.0 * oracle.gemm_f64(A[None], B[None])[0] - C0 if r == 0 else refs[-1])
    with K.BatchedPlan([p[:3] for p in probs], b_layout=layout, alpha=2.0, beta=-1.0) as plan:
        plan.execute()
        torch.cuda.synchronize()
    for (_, _, C, pool, off), ref in zip(probs, refs):
        np.testing.assert_array_equal(C.double().cpu().numpy(), ref)
        rest = torch.cat([pool[:off], pool[off + C.numel():]])
        assert bool((rest == 7.0).all()), "written outside C"
