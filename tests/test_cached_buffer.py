"""The cached workspace and counters of a (device, stream): what a captured graph was given stays its own when a later,
larger call on the stream gets another buffer."""

import weakref

import pytest
import torch

from bpt_amd import paged_attention
from bpt_amd.paged_attention import cached_buffer


def test_an_outgrown_buffer_stays_alive_and_the_kept_ones_are_bounded(monkeypatch):
    monkeypatch.setattr(paged_attention, "_BUFFERS", {})
    monkeypatch.setattr(paged_attention, "_OUTGROWN", [])
    cpu = torch.device("cpu", 0)
    sizes, refs = [], []
    for nbytes in (100, 1 << 20, (1 << 20) + 1, (2 << 20) + 1, 5 << 20, 64 << 20, 3 << 20):
        buf = cached_buffer("partials", cpu, 7, nbytes)
        assert buf.numel() >= nbytes and not buf[:4096].any()
        refs.append(weakref.ref(buf))
        sizes.append(buf.numel())
        del buf
    assert all(r() is not None for r in refs)  # a graph may hold the address of any of them
    assert sizes == sorted(sizes)
    assert sum(b.numel() for b in paged_attention._OUTGROWN) < sizes[-1]


@pytest.mark.gpu
def test_a_graph_replays_into_its_own_buffers_after_a_larger_call():
    from test_gpu_decode import make_case

    from bpt_amd import paged_decode_attention

    def call(c, n, out=None):
        return paged_decode_attention(c["q"], c["k"], c["v"], c["table"], c["lens"], c["ks"], c["vs"], scale=0.09, max_context=n, out=out)

    small, large = make_case("fp8", [3000], nq=2, seed=1), make_case("fp8", [4096] * 6, hq=32, nq=256, seed=2)
    side = torch.cuda.Stream()
    want = call(small, 3000)
    out = torch.empty_like(want)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        call(small, 3000, out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(small, 3000, out)
    with torch.cuda.stream(side):
        call(large, 4096)  # outgrows the side stream's buffers
        others = [torch.full((1 << 18,), 7, dtype=torch.int32, device="cuda") for _ in range(8)]
    torch.cuda.synchronize()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert all((t == 7).all().item() for t in others)
        with torch.cuda.stream(side):
            call(large, 4096)
        torch.cuda.synchronize()
