"""Which parts are told of a norm that may be made whole on the way: on the CPU, with stand-ins for the kernels."""
from types import SimpleNamespace as Spec

import pytest
import torch

from geneinfer_amd.parts.mlp import SwiGlu
from geneinfer_amd.parts.norm import NormToMake, RmsNorm, norm_to_make

D, INTER = 16, 32


class OfItsOwn(SwiGlu):
    """Built on the gated feed-forward, with a `forward` to which `then` is the norm that reads next, as the contract of parts says."""

    def forward(self, h, residual, ctx, then=None, overwrite=False):
        return then.handed_weight(), then.eps


class SaysSo(SwiGlu):
    hands_whole_norms = True

    def forward(self, h, residual, ctx, then=None, overwrite=False):
        return super().forward(h, residual, ctx, then=then, overwrite=overwrite)


class Inherits(SwiGlu):
    pass


class SaysNo(SwiGlu):
    hands_whole_norms = False


@pytest.mark.parametrize("cls, told", [(SwiGlu, True), (Inherits, True), (SaysSo, True), (OfItsOwn, False), (SaysNo, False)])
def test_only_a_forward_that_is_made_for_it_gets_a_norm_to_make(cls, told):
    tensors = dict(gate=torch.randn(INTER, D).bfloat16(), up=torch.randn(INTER, D).bfloat16(), down=torch.randn(D, INTER).bfloat16(), norm=torch.ones(D))
    part = cls(Spec(gate_proj="gate", up_proj="up", down_proj="down", intermediate_size=INTER, hidden_size=D, activation="silu"), tensors, torch.bfloat16, "cpu")
    norm = RmsNorm(Spec(weight="norm", eps=1e-5, size=D), tensors, torch.bfloat16, "cpu")
    reader = Spec(accepts_deferred_norm=True, in_dtype=torch.bfloat16)
    then = norm_to_make((norm, reader), part)
    assert (isinstance(then, NormToMake) and then.norm is norm) if told else then is None
