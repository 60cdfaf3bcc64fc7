"""The route check: error counts of the dispatch plan reach the host whichever
kernels build the plan, and waiting for them waits for nothing else."""

import pytest
import torch

import mirai_amd
from mirai_amd import _native as nat
from mirai_amd import workloads as wl

from helpers import build_module

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _nothing_left_behind():
    mirai_amd.check_route_errors()
    yield
    mirai_amd.check_route_errors()


def _layer(E, d=64, f=64):
    w = wl.Workload("route_check", 14, 1, d, f, E, 1, 1, 1.0, "bf16", torch.bfloat16)
    return build_module(w, wl.dense_weights(w), None)


def _call(m, T, k, bad=0, d=64):
    idx = torch.arange(T * k, device="cuda").view(T, k) % m.num_experts
    idx.view(-1)[5:5 + bad] = m.num_experts
    x = torch.ones(T, d, dtype=torch.bfloat16, device="cuda")
    with torch.no_grad():
        return m.run_direct_routed(x, torch.ones(T, k, device="cuda"), idx)


def test_waiting_for_the_count_waits_for_no_other_stream():
    m = _layer(8)
    _call(m, 64, 2)
    mirai_amd.check_route_errors()
    a = torch.ones(8192, 8192, dtype=torch.bfloat16, device="cuda")
    b, c = torch.ones_like(a), torch.empty_like(a)
    busy = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):  # about 1 ms each
        for _ in range(200):
            torch.mm(a, b, out=c)
        done = torch.cuda.Event()
        done.record()
    _call(m, 64, 2, bad=3)
    with pytest.raises(mirai_amd.RouteIndexError, match="^3 route slot"):
        mirai_amd.check_route_errors()
    assert not done.query()
    _call(m, 64, 2)
    mirai_amd.check_route_errors()
    assert not done.query()
    done.synchronize()


@pytest.mark.parametrize("side", [False, True])
def test_a_long_wait_asks_the_stream_of_the_call(side, monkeypatch):
    monkeypatch.setattr(nat, "_ASK_AFTER", 0.01)
    m = _layer(8)
    a = torch.ones(8192, 8192, dtype=torch.bfloat16, device="cuda")
    b, c = torch.ones_like(a), torch.empty_like(a)
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream() if side else torch.cuda.default_stream()):
        for _ in range(200):
            torch.mm(a, b, out=c)
        _call(m, 64, 2, bad=3)
        with pytest.raises(mirai_amd.RouteIndexError, match="^3 route slot"):
            mirai_amd.check_route_errors()
    torch.cuda.synchronize()
