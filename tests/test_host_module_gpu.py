"""The host module's manners towards the rest of the program: other Python threads, the caller's device, the stage hook,
inputs that it must not launch with."""
import threading
import time

import pytest
import torch

from conftest import randn_lp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _longest_stall(call):
    """Seconds `call` took and the longest time within it that another Python thread could not run."""
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(1e-3)

    th = threading.Thread(target=tick)
    th.start()
    time.sleep(0.02)
    t0 = time.perf_counter()
    call()
    t1 = time.perf_counter()
    time.sleep(0.02)
    stop.set()
    th.join()
    marks = [t for t in ticks if t0 <= t <= t1]
    return t1 - t0, max(b - a for a, b in zip([t0, *marks], [*marks, t1]))


@pytest.mark.parametrize("which", ["attention", "vmonarch", "vmonarch_train"])
def test_other_threads_run_while_a_call_waits_in_the_driver(which):
    """A call whose allocation does not fit under the process's limit gives cached memory back first, which waits for the
    GPU (here some 0.2 s of queued matrix products): other threads go on meanwhile."""
    from vmonarch_amd import flash_entropy_attention, vmonarch_attention
    torch.cuda.empty_cache()
    x = [torch.zeros(1, 9600, 256, 64, device=DEV, dtype=torch.bfloat16) for _ in range(3)]   # 315 MB each
    if which == "vmonarch_train":
        x = [t.requires_grad_() for t in x]
    run = (lambda: flash_entropy_attention(*x)) if which == "attention" else (lambda: vmonarch_attention(*x, 4, 64, 2))
    a = torch.randn(8192, 8192, device=DEV, dtype=torch.bfloat16)
    c = torch.empty_like(a)
    torch.mm(a, a, out=c)
    run()   # (everything loaded)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    cached = [torch.empty(100 << 20, device=DEV, dtype=torch.uint8) for _ in range(40)]   # each too small for an output
    del cached
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
        for _ in range(300):
            torch.mm(a, a, out=c)
        print(f"waiting call: {which}", flush=True)
        took, stall = _longest_stall(run)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
    print(f"took {took:.3f} s, longest stall {stall:.3f} s", flush=True)
    assert took > 0.05, "the call did not wait: nothing tested"
    assert stall < 0.5 * took


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs a second GPU")
@pytest.mark.parametrize("order", ["with_r0", "start"])
def test_tensors_on_another_gpu_than_the_current_one(monkeypatch, order):
    """The launches, the allocations and the fork's events go to the tensors' GPU whichever is current."""
    import vmonarch_amd.vmonarch as vm
    monkeypatch.setattr(vm, "_RECOMPUTE_OVERLAP", order)
    g = torch.Generator().manual_seed(3)
    x = [randn_lp(g, 1, 2, 256, 64, scale=0.5) for _ in range(3)]
    out = []
    for dev in (0, 1):
        with torch.cuda.device(0):
            leaves = [t.to(f"cuda:{dev}").requires_grad_() for t in x]
            o, e = vm.flash_entropy_attention(*leaves)
            z = vm.vmonarch_attention(*leaves, 4, 64, 2, recompute_tokens=64)
            grads = torch.autograd.grad(o.float().sum() + e.sum() + z.float().sum(), leaves)
            assert torch.cuda.current_device() == 0
            out.append([t.detach().cpu() for t in (o, e, z, *grads)])
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_the_current_gpu_is_left_as_it_was():
    from vmonarch_amd import flash_entropy_attention
    before = torch.cuda.current_device()
    flash_entropy_attention(*(torch.zeros(1, 1, 8, 64, device=DEV, dtype=torch.bfloat16) for _ in range(3)))
    assert torch.cuda.current_device() == before


def test_inputs_off_the_gpu_are_refused_before_a_launch():
    from vmonarch_amd import _lib, flash_entropy_attention, vmonarch_attention
    from vmonarch_amd.kernel import fea_forward
    x, far = torch.zeros(1, 2, 256, 64, device=DEV, dtype=torch.bfloat16), torch.zeros(1, 2, 256, 64, dtype=torch.bfloat16)
    for k, v in ((far, x), (x, far)):
        for call in (lambda: flash_entropy_attention(x, k, v), lambda: vmonarch_attention(x, k, v, 4, 64, 2),
                     lambda: _lib.host().fea_attention(x, k, v, 0.1), lambda: fea_forward(x, k, v, None, 0.1)):
            with pytest.raises(AssertionError, match="GPU|device"):
                call()
    with pytest.raises(ValueError, match="GPU"):
        fea_forward(far, far, far, None, 0.1)
    y = x.clone().requires_grad_()
    with pytest.raises(AssertionError, match="device"):
        vmonarch_attention(y, far, x, 4, 64, 2)


@pytest.mark.parametrize("order", ["auto", "with_r0", "start", "after_r0", "after_r1", "off"])
def test_the_stage_hook_hears_of_every_stage(monkeypatch, order):
    """Every stage begins and ends once, the R- and L-steps in turn on the caller's stream, the recompute on whichever it
    runs; what the hook raises comes out of the call."""
    import vmonarch_amd.vmonarch as vm
    monkeypatch.setattr(vm, "_RECOMPUTE_OVERLAP", order)
    q, k, v = (torch.zeros(1, 2, 256, 64, device=DEV, dtype=torch.bfloat16) for _ in range(3))
    heard = []
    with torch.no_grad():
        vm._vmonarch_fused(q, k, v, 4, 64, 2, 64, 0.01, stage_hook=lambda *a: heard.append(a))
    main, side = torch.cuda.current_stream(), vm._side_stream(q.device)
    calls = [(n, p) for n, p, _ in heard]
    chain = [(f"{s}{i}", p) for i in range(2) for s in ("rstep", "lstep") for p in ("begin", "end")]
    assert [c for c in calls if c[0] != "recompute"] == chain
    assert [p for n, p in calls if n == "recompute"] == ["begin", "end"] and len(calls) == len(chain) + 2
    on = side if order in ("start", "after_r0", "after_r1") else main
    assert all(st == (on if n == "recompute" else main) for n, _, st in heard)
    with pytest.raises(ValueError, match="from the hook"):
        vm._vmonarch_fused(q, k, v, 4, 64, 2, 64, 0.01, stage_hook=lambda n, p, st: _fail() if n == "lstep0" else None)
    torch.cuda.synchronize()


def _fail():
    raise ValueError("from the hook")
