"""ringattn_calls (csrc/ringattn_calls.cpp), which forward() and rank_step_forward() go through where their tensors are what the plan
expects: everything else must fare as on the general way -- what was refused is refused with the same words, what is merely unusual is served --,
and a closed plan is out of its reach."""
import threading

import numpy as np
import pytest
import torch

from ringattention_amd import _lib, api


class Marked(torch.Tensor):
    """A tensor subclass: not for the short way, but a tensor like any other."""


def plan_and_tensors(device, dtype="fp16"):
    plan = api.RingAttention(2, [96, 160], 64, 1, 4, dtype, True, kv_heads=2)
    gen = torch.Generator().manual_seed(3)
    t = api.TORCH_DTYPE[api.DTYPE_CODE[dtype]]
    q, k, v = (torch.randn(1, h, 256, 64, generator=gen).to(device=device, dtype=t) for h in (4, 2, 2))
    return plan, [q, k, v, torch.zeros_like(q), torch.zeros(1, 4, 256, device=device)]


def steps_of(plan, tensors):
    """rank_step_forward(1, 1): the diagonal is step 0, step 1 visits rank 0."""
    q, k, v, o, l = tensors
    return [q[:, :, 96:].contiguous(), k[:, :, :96].contiguous(), v[:, :, :96].contiguous(),
            torch.zeros(1, 4, 160, 64, device=q.device), torch.zeros(1, 4, 160, device=q.device)]


def test_host_tensors_are_refused_in_words():
    plan, t = plan_and_tensors("cpu")
    with pytest.raises(ValueError, match="q must be a device tensor"):
        plan.forward(*t)
    assert plan._forward_call(*t, None) is None
    with pytest.raises(ValueError, match="q must be a device tensor"):
        plan.rank_step_forward(1, 1, *steps_of(plan, t))
    with pytest.raises(ValueError, match="rank and step"):
        plan.rank_step_forward(2, 0, *t)
    with pytest.raises(TypeError):
        plan.rank_step_forward(1.0, 1, *steps_of(plan, t))
    with pytest.raises(ValueError, match="q must be a device tensor"):
        plan.rank_step_forward(np.array(1), True, *steps_of(plan, t))
    plan.close()
    assert plan._forward_call is None


def test_arguments_of_a_call():
    calls = _lib.load_calls()
    spec = ((torch.float16, (1, 2)),) * 5
    for bad in ((0, 1, -1, 0, spec), (1, 1, -1, 0, spec[:4]), (1, 1, -1, 0, ((1, 2),) * 5), (1, 1, -1, 0, ((torch.float16, ("a",)),) * 5)):
        with pytest.raises((ValueError, TypeError)):
            calls.Call(*bad)
    call = calls.Call(1, 1, -1, 0, spec)
    for bad in ((), (None,) * 5, (None,) * 7):
        with pytest.raises(TypeError):
            call(*bad)
    assert call(1, 2, 3, 4, 5, None) is None and call(*(None,) * 6) is None


@pytest.fixture(params=["not built", "not loadable"])
def without_module(request, monkeypatch, tmp_path):
    """A library made by make, which does not build the module, or next to a module made for another torch."""
    path = tmp_path / "ringattn_calls.so"
    if request.param == "not loadable":
        path.write_bytes(b"not a library")
    monkeypatch.setattr(_lib, "CALLS_PATH", str(path))
    monkeypatch.setattr(_lib, "_calls", None)


@pytest.mark.filterwarnings("ignore:.*cannot be loaded")
def test_a_plan_does_without_the_module(without_module):
    plan, t = plan_and_tensors("cpu")
    for call, args in ((plan.forward, t), (lambda *a: plan.rank_step_forward(1, 1, *a), steps_of(plan, t))):
        with pytest.raises(ValueError, match="q must be a device tensor"):
            call(*args)
    plan.close()


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:.*cannot be loaded")
def test_results_without_the_module(without_module):
    plan, t = plan_and_tensors("cuda")
    s = steps_of(plan, t)
    plan.forward(*t)
    plan.rank_step_forward(1, 1, *s)
    assert plan._forward_call is None and not plan._step_calls
    o, l = plan.forward(*t[:3])
    p, m = plan.rank_step_forward(1, 1, *s[:3])
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(t[3:] + s[3:], (o, l, p, m)))
    plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_what_does_not_fit_is_refused_as_ever(dtype):
    plan, t = plan_and_tensors("cuda", dtype)
    other = {"fp16": torch.bfloat16, "bf16": torch.float16}[dtype]
    for call, args in ((plan.forward, t), (lambda *a: plan.rank_step_forward(1, 1, *a), steps_of(plan, t))):
        call(*args)
        for i in range(5):
            wrong = [args[i].cpu(), args[i].to(other if i < 3 else torch.float64), args[i][..., :-1], args[i].transpose(-1, -2).contiguous().transpose(-1, -2),
                     args[i][None]]
            for w in wrong[: 5 if args[i].dim() == 4 else 3]:
                with pytest.raises(ValueError):
                    call(*args[:i], w, *args[i + 1:])
        with pytest.raises((AttributeError, TypeError)):
            call(None, *args[1:])
    buf = torch.zeros(t[3].numel() + 8, dtype=t[3].dtype, device="cuda")
    with pytest.raises(_lib.RingattnError, match="aligned"):   # codes of the library come through
        plan.forward(*t[:3], buf[1:1 + t[3].numel()].view_as(t[3]), t[4])
    plan.close()
    with pytest.raises(_lib.RingattnError):
        plan.forward(*t)
    with pytest.raises(_lib.RingattnError):
        plan.rank_step_forward(1, 1, *steps_of(plan, t))


@pytest.mark.gpu
def test_both_ways_give_the_same():
    plan, t = plan_and_tensors("cuda")
    s = steps_of(plan, t)
    plan.forward(*t)
    plan.rank_step_forward(1, 1, *s)
    want = [x.clone() for x in t[3:] + s[3:]]

    def check(call, outs, expected):
        for x in outs:
            x.zero_()
        call()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(outs, expected))

    marked = [x.as_subclass(Marked) for x in t]
    assert plan._forward_call(*marked, None) is None
    check(lambda: plan.forward(*marked), t[3:], want[:2])
    check(lambda: plan.rank_step_forward(1, 1, *[x.as_subclass(Marked) for x in s]), s[3:], want[2:])
    q = t[0].clone().requires_grad_()   # as ever: served, without a graph
    check(lambda: plan.forward(q, *t[1:]), t[3:], want[:2])
    o, l = plan.forward(*t[:3])         # outputs of its own
    assert torch.equal(o, want[0]) and torch.equal(l, want[1])
    with torch.inference_mode():
        check(lambda: plan.forward(*t), t[3:], want[:2])
    # the current stream, one that is handed over, and another thread's
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for how in ("current", "given", "thread"):
        graph = torch.cuda.CUDAGraph()
        for x in t[3:]:
            x.zero_()
        torch.cuda.synchronize()
        if how == "thread":
            def work():
                with torch.cuda.stream(side):
                    plan.forward(*t)
            th = threading.Thread(target=work)
            th.start()
            th.join()
        else:   # a launch that went to any other stream would not be in the capture
            with torch.cuda.graph(graph, stream=side):
                plan.forward(*t, stream=side if how == "given" else None)
            assert not bool(t[3].any())
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(t[3], want[0]) and torch.equal(t[4], want[1])
    plan.close()


@pytest.mark.gpu
def test_batched_tensors_have_no_address():
    plan, t = plan_and_tensors("cuda")
    plan.forward(*t)
    stacked = torch.stack([t[0], t[0]])

    def one(q):
        assert plan._forward_call(q, *t[1:], None) is None
        return plan.forward(q, *t[1:])[0]

    with pytest.raises((RuntimeError, ValueError)):
        torch.vmap(one)(stacked)
    plan.close()
