"""When a block, an attention module or a merge may run as one compiled autograd node: only where calling its submodules
would do the same."""
import numpy as np
import pytest
import torch
from torch import nn

from helpers import random_window_indices
from test_gpu_dense import _stage_pieces

pytestmark = pytest.mark.gpu


def _single(y):
    return "BlockNode" in y.grad_fn.name()


@pytest.mark.parametrize("which", ["drop1", "drop2", "proj_drop", "drop_path"])
def test_dropout_in_train_mode_acts_in_an_eval_block(which):
    """Monte Carlo dropout: the model in eval mode, its dropout modules put back in train mode.  A module obeys its own flag."""
    from sparseswin3d_amd.layers import DropPath
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, False, 5)
    layer.eval()
    plain = run(feats)
    assert _single(plain)
    blk = layer.blocks[1]
    if which == "drop_path":
        blk.drop_path = DropPath(0.5).cuda()
    else:
        (blk.attn if which == "proj_drop" else blk.mlp)._modules[which].p = 0.5
    layer.eval()
    assert torch.equal(run(feats), plain)                         # eval: switched off
    (blk.drop_path if which == "drop_path" else blk.attn.proj_drop if which == "proj_drop" else blk.mlp._modules[which]).train()
    torch.manual_seed(1)
    a = run(feats)
    torch.manual_seed(2)
    b = run(feats)
    assert not torch.allclose(a, plain, rtol=1e-3, atol=1e-3) and not torch.allclose(a, b, rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("which", ["drop1", "drop2", "proj_drop", "drop_path"])
def test_dropout_in_eval_mode_is_off_in_a_training_block(which):
    from sparseswin3d_amd.layers import DropPath
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, False, 5)
    layer.train()
    plain = run(feats)
    blk = layer.blocks[1]
    if which == "drop_path":
        blk.drop_path = DropPath(0.5).cuda()
    drop = blk.drop_path if which == "drop_path" else blk.attn.proj_drop if which == "proj_drop" else blk.mlp._modules[which]
    if which != "drop_path":
        drop.p = 0.5
    drop.eval()
    y = run(feats)
    assert _single(y) and torch.equal(y, plain)
    drop.train()
    assert not torch.allclose(run(feats), plain, rtol=1e-3, atol=1e-3)


class _Weighted(nn.Module):
    """A residual branch of another type than DropPath: scales its branch."""

    def forward(self, x):
        return 3.0 * x


def _of(blk, path):
    for name in path.split("."):
        blk = blk._modules[name]
    return blk


INSIDE = ["attn", "mlp", "attn.proj_drop", "mlp.drop1", "mlp.drop2", "drop_path", "norm1", "norm2", "mlp.fn", "attn.qkv", "attn.proj", "mlp.linear1",
          "mlp.linear2"]
# the projections of a 2-D fp32 call are applied by their weights in the composed block too: no hook of theirs runs
CALLED = [p for p in INSIDE if p not in ("attn.qkv", "attn.proj", "mlp.linear1", "mlp.linear2")]


@pytest.mark.parametrize("training", [True, False], ids=["train", "eval"])
@pytest.mark.parametrize("path", ["drop_path", "attn.proj_drop", "mlp.drop1", "mlp.drop2"])
def test_other_types_in_place_of_dropout_run(path, training):
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, False, 5)
    layer.train(training)
    plain = run(feats)
    parent, _, name = path.rpartition(".")
    owner = _of(layer.blocks[0], parent) if parent else layer.blocks[0]
    setattr(owner, name, _Weighted())
    assert not torch.allclose(run(feats), plain, rtol=1e-3, atol=1e-3)
    setattr(owner, name, nn.Identity())
    assert torch.allclose(run(feats), plain, rtol=1e-4, atol=1e-5)
