"""Which kernels the clearance cost's autograd function asks for (a stand-in for the library's
object, on the CPU)."""
import pytest
import torch

from gvx import torch_cost


class Calls:
    def __init__(self):
        self.made = []

    def forward(self, q, out):
        self.made.append("forward")
        return out.copy_(q.sum((1, 2)))

    def forward_grad(self, q, out, dq):
        self.made.append("forward_grad")
        dq.fill_(1.0)
        return out.copy_(q.sum((1, 2))), dq


@pytest.fixture(autouse=True)
def no_device(monkeypatch):
    monkeypatch.setattr(torch_cost, "_sync", lambda: None)


def test_gradient_only_where_it_is_taped():
    q = torch.rand(3, 4, 2, requires_grad=True)
    c = Calls()
    with torch.no_grad():  # a line search
        assert not torch_cost.clearance_cost(q, c).requires_grad
    with torch.inference_mode():
        torch_cost.clearance_cost(q, c)
    torch_cost.clearance_cost(q.detach(), c)
    assert c.made == ["forward"] * 3
    with torch.no_grad(), torch.enable_grad():
        torch_cost.clearance_cost(q, c)
    assert c.made[3:] == ["forward_grad"]


@pytest.mark.parametrize("apply", [torch_cost.clearance_cost, lambda q, c: torch_cost.ClearanceCostFn.apply(q, c)])
def test_gradient_is_the_product_with_the_upstream_one(apply):
    q = torch.rand(3, 4, 2, requires_grad=True)
    up = torch.tensor([1.0, -2.0, 0.5])
    (apply(q, Calls()) * up).sum().backward()
    assert torch.equal(q.grad, up[:, None, None].expand(3, 4, 2))
