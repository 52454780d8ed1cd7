"""When what is kept of weights is made again: the decision for a filter grid (learned-dynamics_amd/painn.py, Message.table_rows, with
the error of a grid stubbed) and the stamps that caches compare (ops.stamp).  Host logic, no kernel of the library runs."""
import importlib

import pytest
import torch


def _message():
    painn = importlib.import_module("learned-dynamics_amd.painn")
    msg, decisions = painn.Message(5.0, 16), []
    msg.requires_grad_(False)
    msg.table_error = lambda rows: decisions.append(rows) or 0.0
    return msg, decisions


class _Scaled(torch.nn.Module):
    """A parametrization: the weight is computed at every access."""

    def forward(self, w):
        return 0.5 * w


@pytest.mark.parametrize("changed", ["plain", "parametrized", "replaced"])
def test_changed_weights_are_decided_on_again(changed):
    msg, decisions = _message()
    lin = msg.mlp_dist.layers[2]
    if changed == "parametrized":
        torch.nn.utils.parametrize.register_parametrization(lin, "weight", _Scaled())
    weight = lin.parametrizations.weight.original if changed == "parametrized" else lin.weight
    for _ in range(3):
        assert msg.table_rows() == msg.TABLE_ROWS[0]
    assert len(decisions) == 1
    for k in range(2, 5):
        if changed == "replaced":
            lin.weight = torch.nn.Parameter(torch.randn(16 * 4, 16 * 4), requires_grad=False)
        else:
            weight.mul_(3.0)
        msg.table_rows()
        msg.table_rows()
        assert len(decisions) == k


def test_a_weight_computed_at_every_access_is_never_taken_for_the_one_before(ops):
    """The stamp of what is kept of such a weight: another one after a change of what it is computed from, although the allocator
    hands the address out again; that of a parameter or of a tensor that stays is the same until it is written."""
    lin = torch.nn.Linear(64, 64)
    stays = torch.randn(8, 8)
    kept = ops.stamp((lin.weight, stays))
    assert ops.stamp((lin.weight, stays)) == kept
    stays.add_(1.0)
    assert ops.stamp((lin.weight, stays)) != kept
    torch.nn.utils.parametrize.register_parametrization(lin, "weight", _Scaled())
    with torch.no_grad():
        kept = [ops.stamp((lin.weight, lin.bias))]
        for _ in range(20):
            lin.parametrizations.weight.original.mul_(3.0)
            kept.append(ops.stamp((lin.weight, lin.bias)))
            assert kept[-1] != kept[-2]
            del kept[0]
