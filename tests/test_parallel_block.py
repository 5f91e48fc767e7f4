"""A layer whose two halves' first products are one: what its feed-forward is told, on the CPU with stand-ins for the products."""
from types import SimpleNamespace as Spec

import pytest
import torch

from geneinfer_amd.parts import base, block
from geneinfer_amd.parts.mlp import DenseMlp

D, MIX, INTER = 16, 24, 32


class Norm(base.Part):
    def __init__(self, spec, tensors, dtype, device):
        pass

    def __call__(self, x, out_dtype):
        return x.to(out_dtype)


class Mixer(base.Part):
    in_dtype = torch.bfloat16

    def __init__(self, spec, tensors, dtype, device):
        self.w = tensors["mix"]

    def input_weight(self):
        return self.w

    def use_input_weight(self, view):
        self.w = view

    def forward(self, h, residual, ctx, cache, projected=None):
        self.told = projected


class Recording(DenseMlp):
    def forward(self, h, residual, ctx, then=None, overwrite=False, projected=None, activated=None):
        self.told = dict(projected=projected, activated=activated)


class OfItsOwn(DenseMlp):
    """Built on the feed-forward without a gate, with a `forward` that knows nothing of activated columns."""

    def forward(self, h, residual, ctx, then=None, overwrite=False, projected=None):
        self.told = dict(projected=projected)


@pytest.fixture(scope="module", autouse=True)
def kinds():
    for register, kind, cls in ((base.register_norm, "stand_in", Norm), (base.register_mixer, "stand_in", Mixer), (base.register_feed_forward, "recording", Recording),
                                (base.register_feed_forward, "of_its_own", OfItsOwn)):
        register(kind, cls)


@pytest.mark.parametrize("kind, taken", [("recording", True), ("recording", False), ("of_its_own", True)])
def test_a_feed_forward_gets_its_columns_as_it_takes_them(kind, taken, monkeypatch):
    up = torch.randn(INTER, D).bfloat16()
    tensors = dict(mix=torch.randn(MIX, D).bfloat16(), up=up, down=torch.randn(D, INTER).bfloat16(), act=torch.tensor([0.3, 0.1]))
    ff = Spec(kind=kind, activation="xielu", activation_params="act", up_proj="up", down_proj="down", intermediate_size=INTER, hidden_size=D)
    spec = Spec(feed_forward_norm=None, mixer_post_norm=None, feed_forward_post_norm=None, mixer_norm=Spec(kind="stand_in"), mixer=Spec(kind="stand_in"), feed_forward=ff)
    b = block.ParallelBlock(spec, tensors, torch.bfloat16, "cpu")
    x = torch.randn(3, D)
    ready = torch.randn(3, INTER).bfloat16()

    def both_at_once(a, weight, params, columns, dtype, out):
        if taken:
            out[:, :MIX] = a.float() @ weight[:MIX].float().T
            return ready

    monkeypatch.setattr(block, "linear_xielu", both_at_once)
    monkeypatch.setattr(block, "linear", lambda a, weight, out: out.copy_(a.float() @ weight.float().T))
    b.forward(x, Spec(n_rows=3, dtype=torch.bfloat16, trace=None), None)
    assert torch.equal(b.mixer.told, x.bfloat16().float() @ tensors["mix"].float().T)
    told = b.feed_forward.told
    if kind == "recording" and taken:
        assert told["activated"] is ready and told["projected"] is None
    else:
        assert torch.equal(told["projected"], x.bfloat16().float() @ up.float().T) and told.get("activated") is None


class EndingMixer(Mixer):
    def __init__(self, spec, tensors, dtype, device):
        super().__init__(spec, tensors, dtype, device)
        self.w_o = tensors["o"]

    def output_weight(self):
        return self.w_o

    def use_output_weight(self, view):
        self.w_o = view

    def forward(self, h, residual, ctx, cache, then=None, projected=None, into=None):
        ends = torch.arange(h.shape[0] * MIX).view(-1, MIX).bfloat16()
        if into is None:
            residual += ends.float() @ self.w_o.float().T
        else:
            into.copy_(ends)


@pytest.mark.parametrize("traced", [False, True])
def test_both_halves_end_in_one_product(traced, monkeypatch):
    """The halves write the two parts of one buffer, which meets the matrices side by side; a traced pass makes the rows between the halves besides, and its own results by the same one product.
    Either way the weights count once."""
    base.register_mixer("ending", EndingMixer)
    tensors = dict(mix=torch.randn(MIX, D).bfloat16(), o=torch.randn(D, MIX).bfloat16(), up=torch.randn(INTER, D).bfloat16(), down=torch.randn(D, INTER).bfloat16(), act=torch.tensor([0.3, 0.1]))
    ff = Spec(kind="dense_mlp", activation="xielu", activation_params="act", up_proj="up", down_proj="down", intermediate_size=INTER, hidden_size=D)
    spec = Spec(feed_forward_norm=None, mixer_post_norm=None, feed_forward_post_norm=None, mixer_norm=Spec(kind="stand_in"), mixer=Spec(kind="ending"), feed_forward=ff)
    b = block.ParallelBlock(spec, tensors, torch.bfloat16, "cpu")
    matrices = sum(tensors[n].numel() * 2 for n in ("mix", "o", "up", "down"))
    assert matrices <= base.weight_bytes(b) <= matrices + 2 * (MIX + INTER) * D + 64          # (the first products' common matrix is named beside its second half)
    x, seen, products = torch.randn(3, D), [], []
    mid = torch.randn(3, INTER).bfloat16()

    def activated(a, weight, params, columns, dtype, out, into=None):
        return mid if into is None else into.copy_(mid)

    def onto(a, weight, residual, then=None, ctx=None):
        products.append((a.shape[1], weight.shape[1]))
        residual += a.float() @ weight.float().T

    monkeypatch.setattr(block, "linear_xielu", activated)
    for module in (block, __import__("geneinfer_amd.parts.mlp", fromlist=["mlp"])):
        monkeypatch.setattr(module, "linear_onto", onto)
    between = x + torch.arange(3 * MIX).view(3, MIX).bfloat16().float() @ tensors["o"].float().T
    want = x + torch.arange(3 * MIX).view(3, MIX).bfloat16().float() @ tensors["o"].float().T + mid.float() @ tensors["down"].float().T
    b.forward(x, Spec(n_rows=3, dtype=torch.bfloat16, trace=(lambda name, rows: seen.append((name, rows.clone()))) if traced else None), None)
    assert torch.allclose(x, want, rtol=1e-5, atol=1e-3)
    assert products == [(MIX, MIX)] * traced + [(MIX + INTER, MIX + INTER)] and [name for name, _ in seen] == ["attn_out", "ffn_out"] * traced
    if traced:
        assert torch.allclose(seen[0][1], between, rtol=1e-5, atol=1e-3) and torch.equal(seen[1][1], x)


@pytest.mark.parametrize("mix,inter,joined", [(24, 32, True), (64, 128, True), (24, 40, True), (64, 40, False), (200, 128, False), (200, 72, True), (24, 20, False)])
def test_matrices_lie_side_by_side_where_the_kernels_for_many_rows_take_them(mix, inter, joined):
    """Not where one is whole blocks of 64 along k and both together are not (nor where one is not 16 bytes long)."""
    base.register_mixer("ending", EndingMixer)
    tensors = dict(mix=torch.randn(mix, D).bfloat16(), o=torch.randn(D, mix).bfloat16(), up=torch.randn(inter, D).bfloat16(), down=torch.randn(D, inter).bfloat16(), act=torch.tensor([0.3, 0.1]))
    ff = Spec(kind="dense_mlp", activation="xielu", activation_params="act", up_proj="up", down_proj="down", intermediate_size=inter, hidden_size=D)
    b = block.ParallelBlock(Spec(feed_forward_norm=None, mixer_post_norm=None, feed_forward_post_norm=None, mixer_norm=Spec(kind="stand_in"), mixer=Spec(kind="ending"), feed_forward=ff), tensors, torch.bfloat16, "cpu")
    assert (b._last is not None) == joined
    assert torch.equal(b.mixer.w_o, tensors["o"]) and torch.equal(b.feed_forward.w_down, tensors["down"])
