"""What a parallel block does with its feed-forward for few rows, with stand-ins for the launches: its two products go out beside the mixer's only if they
are what the feed-forward's `forward` launches."""
from types import SimpleNamespace as NS

import pytest
import torch

from ferrox_amd import ops
from ferrox_amd.parts.block import ParallelBlock
from ferrox_amd.parts.linear import Linear
from ferrox_amd.parts.mlp import GatedMLP, SwiGLU


class Doubled(GatedMLP):
    """A feed-forward with a `forward` of its own."""

    def forward(self, x, ctx, residual, row_scale=None, fresh=False):
        residual += 2.0


class OtherGate(GatedMLP):
    def _act(self, x):
        return torch.full((x.shape[0], self.intermediate_size), 3.0, dtype=x.dtype)


class OtherLinear(Linear):
    pass


class Mixer:
    def forward(self, x, ctx, cache, residual):
        residual += 1.0


def filled(ffn, linear=Linear):
    ffn.gate_up = linear(torch.ones(64, 16, dtype=torch.bfloat16))
    ffn.down = linear(torch.ones(16, 32, dtype=torch.bfloat16))
    return ffn


@pytest.fixture
def launched(monkeypatch):
    """The epilogues of the products that are launched, in their order."""
    log = []

    def gemm(a, w, *, epilogue=ops.EPI_STORE, out=None, **kw):
        log.append(epilogue)
        n = w.shape[0] // 2 if epilogue == ops.EPI_GATED else w.shape[0]
        out = torch.zeros(a.shape[0], n, dtype=a.dtype) if out is None else out
        out += 0.5
        return out

    monkeypatch.setattr(ops, "gemm", gemm)
    return log


def run(ffn, rows=3, mixer=None):
    block = ParallelBlock.__new__(ParallelBlock)
    block.norm1, block.mixer, block.ffn = NS(forward=lambda h, ctx: h.to(torch.bfloat16)), mixer or Mixer(), ffn
    ctx, h = NS(waiting=[], owed=None), torch.zeros(rows, 16)
    block.forward(h, ctx, None)
    assert ctx.waiting == [] and ctx.owed is None
    return h


@pytest.mark.parametrize("rows", [1, 16, 17])
def test_a_feed_forward_with_a_forward_of_its_own_is_called(launched, rows):
    assert torch.equal(run(filled(Doubled(16, 32)), rows), torch.full((rows, 16), 3.0)) and launched == []
    ffn, seen = filled(GatedMLP(16, 32)), []
    ffn.forward = lambda x, ctx, residual: seen.append(x.shape[0])         # (put in its place on the instance)
    run(ffn, rows)
    assert seen == [rows] and launched == []


def test_a_gate_of_its_own_and_matrices_of_another_class_are_used(launched):
    run(filled(OtherGate(16, 32)))
    assert launched == [ops.EPI_RESID]
    assert filled(GatedMLP(16, 32), OtherLinear).gate_up_product(torch.ones(3, 16, dtype=torch.bfloat16)) is None


@pytest.mark.parametrize("ffn", [GatedMLP(16, 32), SwiGLU(16, 32)])
def test_without_a_product_beside_it_the_feed_forward_follows_the_mixer(launched, ffn):
    run(filled(ffn))
    assert launched == [ops.EPI_GATED, ops.EPI_RESID]


def test_nothing_waits_on_after_a_mixer_that_fails(launched):
    class Fails:
        def forward(self, x, ctx, cache, residual):
            raise ValueError("no")

    block = ParallelBlock.__new__(ParallelBlock)
    block.norm1, block.mixer, block.ffn = NS(forward=lambda h, ctx: h.to(torch.bfloat16)), Fails(), filled(GatedMLP(16, 32))
    ctx = NS(waiting=[], owed=None)
    with pytest.raises(ValueError):
        block.forward(torch.zeros(3, 16), ctx, None)
    assert ctx.waiting == [] and ctx.owed is None


def test_a_mixer_derived_from_latent_attention_does_not_take_what_is_owed():
    from ferrox_amd.parts.latent import LatentAttention

    class Scaled(LatentAttention):
        def forward(self, x, ctx, cache, residual, **kw):
            rows = torch.zeros_like(residual)
            super().forward(x, ctx, cache, rows, **kw)
            residual += 0.5 * rows

    for cls, adds in ((LatentAttention, True), (Scaled, False)):
        mixer = cls.__new__(cls)
        mixer.o_proj = Linear(torch.ones(16, 64, dtype=torch.bfloat16))
        assert mixer.adds_owed() == adds
