"""Calls captured into a HIP graph: every replay, with eager work and new inputs between them, gives
the bits of the eager call, with the result given or allocated in the capture."""
import pytest

import kami_amd as K

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def block(prec, dt, dev, g, layout):
    A, B = torch.randn((64, 64, 64), generator=g).to(dt).to(dev), torch.randn((64, 64, 64), generator=g).to(dt).to(dev)
    C = torch.empty((64, 64, 64), dtype=torch.float64 if dt == torch.float64 else torch.float32, device=dev)
    return A, C, lambda: K.block_gemm(A, B, C, b_layout=layout), lambda: K.block_gemm(A, B, b_layout=layout)


def split(dev, g):
    A, B = (torch.randn((192, 160), generator=g, dtype=torch.float64).to(dev) for _ in range(2))
    C = torch.empty((192, 192), dtype=torch.float64, device=dev)
    return A, C, lambda: K.split_gemm(A, B, C), lambda: K.split_gemm(A, B)


def spmm(dt, dev, g):
    rp = torch.tensor([0, 2, 2, 5], dtype=torch.int32, device=dev)
    ci = torch.tensor([0, 3, 1, 2, 3], dtype=torch.int32, device=dev)
    V = torch.randn((5, 32, 32), generator=g).to(dt).to(dev)
    S = K.BsrMatrix(3, 4, 32, rp, ci, V)
    B = torch.randn((48, 128), generator=g).to(dt).to(dev)
    C = torch.empty((96, 48), dtype=torch.float64 if dt == torch.float64 else torch.float32, device=dev)
    return V, C, lambda: K.bsr_spmm(S, B, C), lambda: K.bsr_spmm(S, B)


def batched(dt, dev, g, layout):
    probs = []
    for m, n, k in [(16, 48, 80), (256, 128, 64), (112, 32, 16), (64, 64, 256)]:
        probs.append((torch.randn((m, k), generator=g).to(dt).to(dev),
                      torch.randn((n, k) if layout == "nk" else (k, n), generator=g).to(dt).to(dev),
                      torch.empty((m, n), dtype=torch.float64 if dt == torch.float64 else torch.float32, device=dev)))
    plan = K.BatchedPlan(probs, b_layout=layout, use_graph=layout == "nk")
    return probs[1][0], probs[1][2], plan.execute, None


CASES = {"block-f64": lambda d, g: block(K.PREC_F64, torch.float64, d, g, "nk"),
         "block-f16-kn": lambda d, g: block(K.PREC_F16_F32, torch.float16, d, g, "kn"),
         "split": split,
         "spmm-f16": lambda d, g: spmm(torch.float16, d, g), "spmm-f64": lambda d, g: spmm(torch.float64, d, g),
         "batched-f64": lambda d, g: batched(torch.float64, d, g, "nk"),
         "batched-bf16-kn": lambda d, g: batched(torch.bfloat16, d, g, "kn")}


@pytest.mark.parametrize("name", list(CASES))
def test_replays_are_the_eager_call(name, dev):
    print(f"\n[case] {name}", flush=True)
    x, C, given, allocating = CASES[name](dev, torch.Generator().manual_seed(1))
    given()  # warm, before the capture
    if allocating:
        allocating()
    torch.cuda.synchronize()
    graph, own = torch.cuda.CUDAGraph(), None
    with torch.cuda.graph(graph):
        given()
        if allocating:
            own = allocating()
    for _ in range(4):
        C.fill_(float("nan"))
        x.mul_(-0.5)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got, got_own = C.clone(), own.clone() if own is not None else None
        C.fill_(float("nan"))
        given()
        torch.cuda.synchronize()
        assert torch.equal(got, C) and not torch.isnan(got).any()
        assert got_own is None or torch.equal(got_own, C)
