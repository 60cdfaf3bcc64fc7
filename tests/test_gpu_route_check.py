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


def _busy(n=200):
    a = torch.ones(8192, 8192, dtype=torch.bfloat16, device="cuda")
    for _ in range(n):  # about 1 ms each
        torch.mm(a, a)


def test_slots_of_failed_calls_are_not_given_out_under_their_stores(monkeypatch):
    """Calls that fail after their plan was queued leave stores on their way to
    their slots. 256 calls later the slots come round: the stores of the failed
    calls (two bad ids each) must not be read as a valid call's count."""
    m = _layer(8)
    _call(m, 64, 2)
    mirai_amd.check_route_errors()
    call = nat.call

    def failing(name, *args):
        call(name, *args)
        if name == "mx_moe_forward_watched":
            raise RuntimeError("failed after the plan")

    _busy()
    monkeypatch.setattr(nat, "call", failing)
    for _ in range(300):
        with pytest.raises(RuntimeError, match="failed after the plan"):
            _call(m, 64, 2, bad=2)
    monkeypatch.setattr(nat, "call", call)
    _call(m, 64, 2)
    while nat._pending:
        nat.poll_route_errors()
    _call(m, 64, 2, bad=3)
    with pytest.raises(mirai_amd.RouteIndexError, match="^3 route slot"):
        mirai_amd.check_route_errors()


def test_a_count_that_never_lands_is_an_error_of_its_own(monkeypatch):
    monkeypatch.setattr(nat, "_ASK_AFTER", 0.01)
    m = _layer(8)
    call = nat.call
    monkeypatch.setattr(nat, "call", lambda name, *a: None if name == "mx_moe_forward_watched"
                        else call(name, *a))
    _call(m, 64, 2)
    monkeypatch.setattr(nat, "call", call)
    with pytest.raises(RuntimeError, match="without storing"):
        mirai_amd.check_route_errors()
    _call(m, 64, 2)
    mirai_amd.check_route_errors()


def test_the_slots_come_round():
    m = _layer(8)
    _busy(50)  # the host runs ahead of all 256 slots
    for i in range(600):
        _call(m, 64, 2, bad=4 if i == 599 else 0)
    with pytest.raises(mirai_amd.RouteIndexError, match="^4 route slot"):
        mirai_amd.check_route_errors()


# Tokens, top-k and experts of each way to build the plan: one workgroup, the
# fused kernel over several blocks, and the scan of its own above 1024 experts
# and above 65536 block counts.
@pytest.mark.parametrize("T,k,E", [(2048, 2, 8), (2049, 2, 8), (9000, 4, 64), (3000, 2, 1100),
                                   (33000, 2, 256)])
@pytest.mark.parametrize("mode", ["deferred", "sync"])
def test_every_plan_stores_its_count(T, k, E, mode):
    m = _layer(E)
    previous = nat.route_check_mode()
    mirai_amd.set_route_check(mode)
    try:
        _call(m, T, k)
        mirai_amd.check_route_errors()
        with pytest.raises(mirai_amd.RouteIndexError, match="^37 route slot"):
            _call(m, T, k, bad=37)
            mirai_amd.check_route_errors()
    finally:
        mirai_amd.set_route_check(previous)
