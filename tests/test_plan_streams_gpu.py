"""Plans on streams: a plan built on one stream runs on another with no event between them (its
length arrays bound every address it reads, so they are in place when the constructor
returns), and a captured run() or call replays to the eager result."""
import pytest
import torch

from dsa_triton_ascend_amd import PrefillPlan, lightning_indexer
from dsa_triton_ascend_amd.dense_loss import DenseLossPlan, dense_lightning_indexer_softmax_lse
from dsa_triton_ascend_amd.lightning_indexer import IndexerPlan
from dsa_triton_ascend_amd.sli_grad_kl_loss import KLLossPlan
from dsa_triton_ascend_amd.sparse_flash_attention import AttentionPlan, sparse_flash_attention
from dsa_triton_ascend_amd.sparse_flash_attention_grad import GradPlan

pytestmark = pytest.mark.gpu
B, S, N1, D, K = 2, 96, 16, 512, 64
LENS = [96, 70]


@pytest.fixture(scope="module")
def tensors():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    g = torch.Generator().manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    t = dict(q=r(B, S, N1, D), k=r(B, S, 1, D), qr=r(B, S, N1, 64), kr=r(B, S, 1, 64), do=r(B, S, N1, D),
             qi=r(B, S, 32, 128), ki=r(B, S, 1, 128), w=r(B, S, 32))
    t["si"] = lightning_indexer(t["qi"], t["ki"], t["w"], LENS, LENS, sparse_count=K)[0]
    t["out"], t["max"], t["sum"] = sparse_flash_attention(
        t["q"], t["k"], t["k"], t["si"], 0.04, actual_seq_lengths_query=LENS, actual_seq_lengths_kv=LENS,
        query_rope=t["qr"], key_rope=t["kr"], sparse_mode=3, return_softmax_lse=True)
    t["mi"], t["smi"] = dense_lightning_indexer_softmax_lse(t["qi"], t["ki"], t["w"], LENS, LENS)
    torch.cuda.synchronize()
    return t


def _plan(kind, t):
    if kind == "indexer":
        return IndexerPlan(t["qi"], t["ki"], t["w"], LENS, LENS, sparse_count=K, return_value=True)
    if kind == "attention":
        return AttentionPlan(t["q"], t["k"], t["k"], t["si"], 0.04, None, LENS, LENS, t["qr"], t["kr"], sparse_mode=3,
                             return_softmax_lse=True)
    if kind == "grad":
        return GradPlan(t["q"], t["k"], t["k"], t["si"], t["do"], t["out"], t["max"], t["sum"], 0.04, t["qr"], t["kr"],
                        LENS, LENS)
    if kind == "kl":
        return KLLossPlan(t["q"], t["k"], t["qi"], t["ki"], t["w"], t["si"].clamp_min(0), t["max"], t["sum"], t["qr"],
                          t["kr"], LENS, LENS, 0.04)
    if kind == "dense":
        return DenseLossPlan(t["q"], t["k"], t["qi"], t["ki"], t["w"], t["max"], t["sum"], t["mi"], t["smi"], 0.04,
                             t["qr"], t["kr"], LENS, LENS)
    flat = lambda n: t[n].reshape(B * S, *t[n].shape[2:])
    return PrefillPlan(flat("qi"), flat("ki"), flat("w"), flat("q"), flat("k"), flat("qr"), flat("kr"), [96, 192], K, 0.04,
                       return_softmax_lse=True)


@pytest.mark.parametrize("kind", ["indexer", "attention", "grad", "kl", "dense", "prefill"])
def test_plan_runs_on_another_stream(tensors, kind):
    want = [o.clone() for o in _plan(kind, tensors).run()]
    torch.cuda.synchronize()
    build, use = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(build):
        torch.cuda._sleep(40_000_000)   # the constructor's work is queued behind this
        plan = _plan(kind, tensors)
    with torch.cuda.stream(use):
        got = plan.run()
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        if kind in ("kl", "dense"):   # fp32 atomics: the order of a sum, then one rounding to 16 bits
            assert (a.float() - b.float()).norm() <= 4e-3 * b.float().norm()
        else:
            assert torch.equal(a, b)


@pytest.mark.parametrize("kind", ["indexer", "attention", "prefill"])
def test_captured_run_replays(tensors, kind):
    plan = _plan(kind, tensors)
    want = [o.clone() for o in plan.run()]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = plan.run()
    for _ in range(3):
        for o in got:
            o.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)
        _plan(kind, tensors).run()   # eager work of its own between the replays
        torch.cuda.synchronize()


def test_captured_call_replays(tensors):
    """The whole call under capture: its length arrays are written by a node of the graph."""
    call = lambda: lightning_indexer(tensors["qi"], tensors["ki"], tensors["w"], LENS, LENS, sparse_count=K,
                                     return_value=True)
    want = [o.clone() for o in call()]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = call()
    for _ in range(3):
        for o in got:
            o.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)
        call()
        torch.cuda.synchronize()
