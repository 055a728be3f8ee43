"""The optimizer's job table (optim.AdamW._plan, host_module.cpp Updates), kept from step to step: looked at on the CPU, where
no kernel is launched."""
import ctypes

import pytest
import torch

from crystalframer_amd import optim


def _optimizer(*sizes):
    ps = [torch.nn.Parameter(torch.randn(n)) for n in sizes]
    opt = optim.AdamW(ps)
    group = opt.param_groups[0]
    total = sum(-(-n // 4) * 4 for n in sizes)
    offs = [sum(-(-n // 4) * 4 for n in sizes[:i]) for i in range(len(sizes))]
    st = dict(exp_avg=torch.zeros(total), exp_avg_sq=torch.zeros(total), step=torch.zeros(1, dtype=torch.int64),
              offset={id(p): o for p, o in zip(ps, offs)}, numel={id(p): p.numel() for p in ps})
    opt._flat[id(group)] = st
    for p in ps:
        p.grad = torch.ones_like(p)
    return opt, group, st


def test_an_exchanged_parameter_makes_the_job_table_anew():
    opt, group, st = _optimizer(5, 7, 9)
    plan = opt._plan(group, st)
    assert opt._plan(group, st) is plan
    old = group["params"][1]
    new = torch.nn.Parameter(torch.zeros(7))
    new.grad = torch.ones(7)
    group["params"][1] = new
    again = opt._plan(group, st)
    assert again is not plan and again["params"][1] is new
    with pytest.raises(RuntimeError, match="at the first step"):       # it has no moments: refused, not skipped
        opt._fill(again, 0, 0)
    opt.zero_grad()
    assert new.grad is None and old.grad is not None
    group["params"] = (group["params"][0], old, group["params"][2])    # (any sequence)
    assert opt._plan(group, st)["params"][1] is old
    group["params"] = [group["params"][i] for i in (2, 1, 0)]
    assert [id(p) for p in opt._plan(group, st)["params"]] == [id(p) for p in group["params"]]


def test_sizes_that_do_not_fit_the_moments_are_refused():
    """The kernel goes over as many words of parameter, gradient and moments as the table says."""
    opt, group, st = _optimizer(5, 7)
    plan = opt._plan(group, st)
    fill = lambda: plan["native"].fill(ctypes.addressof(plan["jobs"]), 4096, 8192)  # noqa: E731
    assert fill() == 2 and [j.n for j in plan["jobs"]] == [5, 7] and plan["jobs"][1].exp_avg == 4096 + 4 * 8
    p = group["params"][1]
    old = p.data
    for other in (torch.zeros(70), torch.zeros(3), old.double()):
        p.data = other
        assert opt._plan(group, st) is plan and fill() == -1
        with pytest.raises(RuntimeError, match="size or device|float32"):
            opt._fill(plan, 0, 0)
    p.grad = None
    p.data = torch.zeros(70)
    p.grad = torch.zeros(70)                         # fits the parameter, not the moments
    assert fill() == -1
    with pytest.raises(RuntimeError, match="size or device"):
        opt._fill(plan, 0, 0)
    p.grad = None
    p.data = old
    assert fill() == 1
