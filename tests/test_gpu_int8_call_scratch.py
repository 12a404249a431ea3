"""GPU: the quantised rows of an int8 call are the call's own -- not in the scratch that the calls of a stream share, which all
graphs captured on that stream would write."""

import pytest
import torch

from keras_amd import ops as kops
from keras_amd.layers import Dense, EinsumDense

pytestmark = pytest.mark.gpu


def make(kind, policy):
    if kind == "dense":
        layer = Dense(768, dtype=policy, device="cuda:0")
    else:
        layer = EinsumDense("btd,dnh->btnh", (None, 6, 128), dtype=policy, device="cuda:0")
    layer.build((None, 512) if kind == "dense" else (None, None, 512))
    layer.quantize("int8")
    return layer


@pytest.mark.parametrize("kind", ["dense", "einsum"])
@pytest.mark.parametrize("policy,rows", [("float32", 16), ("mixed_bfloat16", 100), ("float32", 2000)])
def test_graphs_of_one_stream_side_by_side(dev, monkeypatch, kind, policy, rows):
    layer = make(kind, policy)
    shape = (rows, 512) if kind == "dense" else (1, rows, 512)
    xs = [torch.randn(shape, generator=torch.Generator().manual_seed(i)).to(dev) for i in range(2)]
    want = [layer(x) for x in xs]
    shared = []
    real = kops._workspace
    monkeypatch.setattr(kops, "_workspace", lambda *a: (shared.append(a), real(*a))[1])
    capture, graphs, outs = torch.cuda.Stream(), [], []
    capture.wait_stream(torch.cuda.current_stream())
    for x in xs:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=capture):
            outs.append(layer(x))
        graphs.append(g)
    # (a split of K keeps its partial sums there, which these shapes do not ask for)
    assert not shared
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(20):
        for y in outs:
            y.zero_()
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(y, w) for y, w in zip(outs, want))
