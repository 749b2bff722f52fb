"""Block.packed's parameter lookup: every way a member can stand in for the
registered one reaches the packed tensors, as the attribute would."""
import pytest
import torch
from torch import nn
from torch.nn.utils import parametrize

import nsw
from nsw.layer_helpers import parameter, submodule

# field of the packed dict, owner of the parameter, parameter name
MEMBERS = [("wqkv", "attn.v", "weight"), ("bqkv", "attn.biask", "bias"), ("qn_w", "attn.q_norm.norm", "weight"),
           ("kn_w", "attn.k_norm.norm", "weight"), ("wproj", "attn.proj", "weight"), ("bproj", "attn.biasproj", "bias"),
           ("norm1_w", "norm1.norm", "weight"), ("norm2_w", "norm2.norm", "weight"), ("w1", "mlp.fc1", "weight"),
           ("b1", "mlp.bias1", "bias"), ("w2", "mlp.fc2", "weight"), ("b2", "mlp.bias2", "bias")]


class Doubled(nn.Module):
    def forward(self, w):
        return 2 * w


def _block():
    return nsw.Block(32, 2, (18, 36), (9, 18), 1, shift_size=(4, 9)).eval()


@pytest.mark.parametrize("field,owner,name", MEMBERS)
@pytest.mark.parametrize("how", ["in_place", "assigned", "parametrized", "replaced_module"])
def test_packed_follows_the_member(field, owner, name, how):
    blk = _block()
    before = {k: v.clone() for k, v in blk.packed().items()}
    mod = blk.get_submodule(owner)
    with torch.no_grad():
        if how == "in_place":
            getattr(mod, name).mul_(2).add_(1)
            want = getattr(mod, name)
        elif how == "assigned":
            setattr(mod, name, nn.Parameter(2 * getattr(mod, name) + 1))
            want = getattr(mod, name)
        elif how == "parametrized":
            getattr(mod, name).add_(1)
            want = 2 * getattr(mod, name)
            parametrize.register_parametrization(mod, name, Doubled())
        else:
            new = nn.Module()
            new.eps = getattr(mod, "eps", None)
            setattr(new, name, nn.Parameter(2 * getattr(mod, name) + 1))
            parent, _, leaf = owner.rpartition(".")
            setattr(blk.get_submodule(parent), leaf, new)
            want = getattr(new, name)
        after = blk.packed()
    rows = {"attn.q": 0, "attn.k": 1, "attn.biask": 1, "attn.v": 2}
    got = after[field].chunk(3)[rows[owner]] if owner in rows else after[field]
    assert torch.equal(got, want.detach())
    assert not torch.equal(after[field], before[field])


def test_functional_call_and_plain_objects():
    blk = _block()
    w = torch.full_like(blk.mlp.fc1.weight, 0.5)

    class Look(nn.Module):
        def __init__(self, b):
            super().__init__()
            self.b = b

        def forward(self):
            return parameter(submodule(submodule(self.b, "mlp"), "fc1"), "weight")

    assert torch.equal(torch.func.functional_call(Look(blk), {"b.mlp.fc1.weight": w}, ()), w)
    plain = type("Plain", (), {"weight": w, "fc1": blk})()
    assert parameter(plain, "weight") is w and submodule(plain, "fc1") is blk
    with pytest.raises(AttributeError):
        parameter(blk, "nothing")
