"""FP64 queues of wide problems in the K x N layout take the larger wave tiles whatever K is: on
either side of the rule's width and length, with problems whose last strips are one to three
atoms, exact on integers."""
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("count", [430, 700])
@pytest.mark.parametrize("shapes", [[(256, 256, 16), (240, 272, 32), (208, 304, 48)], [(256, 160, 16), (224, 176, 32)],
                                    [(16, 1024, 16), (1024, 272, 16)]], ids=["wide", "narrow", "long"])
def test_exact(shapes, count, dev):
    print(f"\n[case] {shapes} x{count}", flush=True)
    g = torch.Generator(device=dev).manual_seed(count)
    probs, refs = [], []
    for i in range(count):
        m, n, k = shapes[i % len(shapes)]
        A, B, C = (torch.randint(-2, 3, s, generator=g, device=dev).double() for s in ((m, k), (k, n), (m, n)))
        refs.append(2.0 * (A @ B) - C)
        probs.append((A, B, C))
    with K.BatchedPlan(probs, b_layout="kn", alpha=2.0, beta=-1.0) as plan:
        plan.execute()
    for (_, _, C), ref in zip(probs, refs):
        assert torch.equal(C, ref)
