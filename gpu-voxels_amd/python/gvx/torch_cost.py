"""torch.autograd.Function over the hand-written clearance-cost kernels.

A pass that needs the gradient takes the costs and each trajectory's own gradient from one
walk over the grid (gvx_cost_forward_grad): the pass is bound by the samples it gathers, and
both need the same ones (256 x 32 waypoints of 7 x 64 spheres on 512^3: 92 us for the costs
alone, 95 for both).  The backward pass is the product with the upstream gradient.
"""
import torch

from . import Cost


def _sync():
    torch.cuda.current_stream().synchronize()


class ClearanceCostFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, cost, taped=True):
        q = q.detach().contiguous().float()
        out = torch.empty(q.shape[0], device=q.device, dtype=torch.float32)
        # needs_input_grad does not know of torch.no_grad(): taped does
        if not (taped and ctx.needs_input_grad[0]):
            _sync()
            return cost.forward(q, out)
        dq = torch.empty_like(q)
        _sync()
        cost.forward_grad(q, out, dq)
        ctx.save_for_backward(q, dq)  # q: changed in place before the backward pass, it is refused there
        return out

    @staticmethod
    def backward(ctx, grad_out):
        _, dq = ctx.saved_tensors
        # zero without contact, also where grad_out is infinite (the root of a cost of zero)
        return torch.where(dq == 0, dq, dq * grad_out.detach().float()[:, None, None]), None, None


def clearance_cost(q, cost: Cost):
    """q: (T, W, L) float32 CUDA tensor of joint values -> (T,) cost per trajectory."""
    return ClearanceCostFn.apply(q, cost, torch.is_grad_enabled())
