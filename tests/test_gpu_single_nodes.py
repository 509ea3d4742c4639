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


@pytest.mark.parametrize("path", CALLED)
def test_hooks_inside_a_block_run(path):
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, False, 5)
    plain = run(feats)
    m = _of(layer.blocks[0], path)
    calls = []
    for register in (m.register_forward_hook, m.register_forward_pre_hook):
        calls.clear()
        handle = register(lambda *a: calls.append(1))
        y = run(feats)
        handle.remove()
        assert len(calls) == (2 if path == "drop_path" else 1)    # both branches
        assert torch.allclose(y, plain, rtol=1e-4, atol=1e-5)
    calls.clear()
    handle = m.register_full_backward_hook(lambda *a: calls.append(1))
    if path != "attn":                                            # a view goes in and comes out: no tensors, no backward hook
        run(feats.clone().requires_grad_(True)).sum().backward()
        assert calls
    handle.remove()


@pytest.mark.parametrize("register", [nn.modules.module.register_module_forward_hook, nn.modules.module.register_module_forward_pre_hook,
                                      nn.modules.module.register_module_full_backward_hook], ids=["forward", "forward_pre", "backward"])
def test_global_module_hooks_see_the_modules_of_a_block_and_a_merge(register):
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, True, 5)
    seen = set()
    handle = register(lambda m, *a: seen.add(id(m)) and None)
    try:
        run(feats.clone().requires_grad_(True)).sum().backward()
    finally:
        handle.remove()
    blk = layer.blocks[0]
    for m in [_of(blk, p) for p in CALLED if p != "attn"] + [layer.downsample.norm]:
        assert id(m) in seen, type(m)


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


@pytest.mark.parametrize("what", ["forward_part1", "forward_part2", "window_view"])
@pytest.mark.parametrize("how", ["subclass", "instance"])
def test_overridden_parts_of_a_block_run(what, how):
    from sparseswin3d_amd.layers import SwinTransformerBlock
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, False, 5)
    plain = run(feats)
    calls = []
    original = getattr(SwinTransformerBlock, what)

    def replaced(self, *a):
        calls.append(1)
        return original(self, *a)

    blk = layer.blocks[0]
    if how == "subclass":
        blk.__class__ = type("Other", (SwinTransformerBlock,), {what: replaced})
    else:
        object.__setattr__(blk, what, replaced.__get__(blk))
    y = run(feats)
    assert len(calls) >= (2 if what == "window_view" else 1)      # the stage asks for the view once itself
    assert torch.allclose(y, plain, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("path", CALLED)
def test_forward_replaced_on_an_instance_runs(path):
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, False, 5)
    m = _of(layer.blocks[0], path)
    calls, original = [], m.forward
    m.forward = lambda *a, **k: (calls.append(1), original(*a, **k))[1]
    run(feats)
    assert calls


def test_merge_modules_replaced_on_an_instance_run():
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, True, 5)
    norm, calls = layer.downsample.norm, []
    original = norm.forward
    norm.forward = lambda x: (calls.append(1), original(x))[1]
    run(feats)
    assert calls == [1]


@pytest.mark.parametrize("x,w", [(torch.bfloat16, torch.float32), (torch.float16, torch.float32), (torch.float32, torch.float16), (torch.float64, torch.float32)])
@pytest.mark.parametrize("grad", [True, False], ids=["grad", "no_grad"])
def test_features_and_weights_of_different_types_are_refused(x, w, grad):
    """Outside autocast a dense layer refuses operands of two types, as nn.Linear does, and does not round the weights; inside
    float64 features stay refused."""
    from sparseswin3d_amd.window_attention import SparseVoxelTensor, WindowAttentionSparse
    torch.manual_seed(0)
    attn = WindowAttentionSparse(96, 3, (5, 5, 5), qkv_bias=True).cuda().to(w)
    ind = torch.from_numpy(random_window_indices(np.random.default_rng(0), 40, 125, 700)).cuda()
    feats = torch.randn(700, 96, device="cuda").to(x)
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="dtype"):
        attn(SparseVoxelTensor(feats, ind, (125,), 40), None)
    if x == torch.float64:
        with torch.set_grad_enabled(grad), torch.autocast("cuda", dtype=torch.float16), pytest.raises(RuntimeError, match="dtype"):
            attn(SparseVoxelTensor(feats, ind, (125,), 40), None)
    layer, run, _ = _stage_pieces(96, 3, 5, w, True, 7)
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError):
        run(torch.randn(3000, 96, device="cuda").to(x))


@pytest.mark.parametrize("path", ["attn.qkv.bias", "attn.proj.bias", "mlp.linear1.bias", "mlp.linear2.bias", "norm1.bias", "norm2.bias", "attn.proj.weight"])
def test_parameters_of_another_type_are_refused(path):
    """One parameter of a fp32 block left in bf16: refused by the layer it belongs to, not rounded or widened on the way."""
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, False, 7)
    owner, _, name = path.rpartition(".")
    m = _of(layer.blocks[0], owner)
    m._parameters[name] = nn.Parameter(m._parameters[name].detach().bfloat16())
    with pytest.raises(RuntimeError):
        run(feats)


@pytest.mark.parametrize("single", [True, False], ids=["node", "composed"])
@pytest.mark.parametrize("grad", [True, False], ids=["grad", "no_grad"])
def test_merge_refuses_rows_that_are_not_its_voxels(single, grad, monkeypatch):
    from sparseswin3d_amd import layers
    from sparseswin3d_amd.window_attention import SparseVoxelTensor
    if not single:
        monkeypatch.setattr(layers, "_fused_dtype", lambda *a: None)
    pool = layers.PoolDownsample(32).cuda()
    cells = np.random.default_rng(0).choice(20 ** 3, size=900, replace=False)
    c4 = torch.from_numpy(np.stack([0 * cells, *np.unravel_index(cells, (20, 20, 20))], 1).astype(np.int32)).cuda()
    with torch.set_grad_enabled(grad):
        for n in (899, 901, 1, 0):
            with pytest.raises(RuntimeError, match="900 voxels"):
                pool(SparseVoxelTensor(torch.randn(n, 32, device="cuda"), c4, (20, 20, 20), 1))
        pool(SparseVoxelTensor(torch.randn(900, 32, device="cuda"), c4, (20, 20, 20), 1))


@pytest.mark.parametrize("owner", ["block", "merge"])
@pytest.mark.parametrize("name", ["weight", "bias"])
@pytest.mark.parametrize("size", [48, 192])
def test_norm_parameters_of_another_size_are_refused(owner, name, size):
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, True, 7)
    norm = layer.blocks[0].norm2 if owner == "block" else layer.downsample.norm
    norm._parameters[name] = nn.Parameter(torch.ones(size, device="cuda"))
    with pytest.raises(RuntimeError):
        run(feats)


@pytest.mark.parametrize("path", ["blocks.0.norm1.weight", "blocks.0.attn.qkv.weight", "blocks.0.attn.proj.bias", "blocks.1.norm2.bias", "blocks.1.mlp.linear1.weight",
                                  "downsample.norm.weight", "downsample.reduction.weight"])
@pytest.mark.parametrize("grad", [True, False], ids=["grad", "no_grad"])
def test_parameters_on_another_device_are_refused(path, grad):
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, True, 7)
    owner, _, name = path.rpartition(".")
    m = layer
    for part in owner.split("."):
        m = m._modules[part]
    m._parameters[name] = nn.Parameter(m._parameters[name].detach().cpu())
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="same device"):
        run(feats)


def test_attention_refuses_masks_and_plans_it_cannot_read():
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan, fused_window_attention
    from sparseswin3d_amd.window_attention import SparseVoxelTensor, WindowAttentionSparse, relative_position_index_3d
    attn = WindowAttentionSparse(96, 3, (5, 5, 5), qkv_bias=True).cuda()
    ind = torch.from_numpy(random_window_indices(np.random.default_rng(0), 40, 125, 700)).cuda()
    feats = torch.randn(700, 96, device="cuda")
    with pytest.raises(RuntimeError, match="same device"):
        attn(SparseVoxelTensor(feats, ind, (125,), 40), torch.zeros(40, 125, dtype=torch.int8))
    ti = BiasTableIndex.build(relative_position_index_3d((5, 5, 5)).cuda(), 729)
    qkv, table = torch.randn(700, 3, 3, 32, device="cuda"), torch.randn(729, 3, device="cuda")
    for kw in (dict(tasks=False), dict(tasks=True, order_only=True), dict(tasks=False, order_only=True)):
        with pytest.raises(RuntimeError, match="without what"):
            fused_window_attention(qkv, table, ind, None, 40, 125, 0.2, plan=TokenPlan(ind, 40, 125, 3, **kw), table_index=ti)
    small = BiasTableIndex.build(relative_position_index_3d((4, 4, 4)).cuda(), 343)
    with pytest.raises(RuntimeError, match="position codes"):
        fused_window_attention(qkv, table, ind, None, 40, 125, 0.2, table_index=small)


@pytest.mark.parametrize("dim,heads,window,mode", [(96, 3, 5, "fp32"), (48, 3, 7, "fp32"), (48, 3, 7, "amp"), (192, 6, 5, "bf16")])
def test_nodes_on_other_streams(dim, heads, window, mode):
    """A stage with its merge on a stream of its own, and on two streams at once from two threads: the bits of the default stream
    (sums are added in a fixed order everywhere)."""
    import threading
    layer, run, feats = _stage_pieces(dim, heads, window, torch.bfloat16 if mode == "bf16" else torch.float32, True, 11)
    up = torch.randn(4096, 2 * dim, device="cuda")

    def once(x):
        with torch.autocast("cuda", dtype=torch.float16, enabled=mode == "amp"):
            y = run(x)
        grads = torch.autograd.grad(y, [x, *layer.parameters()], up[:y.shape[0]].to(y.dtype))
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, enabled=mode == "amp"):
            return [y.detach(), run(x), *grads]

    want = once(feats.clone().requires_grad_(True))
    torch.cuda.synchronize()
    results, errors = {}, []

    def work(k, gate=None):
        try:
            stream = torch.cuda.Stream()
            stream.wait_stream(torch.cuda.default_stream())
            with torch.cuda.stream(stream):
                x = feats.clone().requires_grad_(True)
                if gate is not None:
                    gate.wait()
                for r in range(3):
                    results[k, r] = once(x)
            stream.synchronize()
        except Exception as e:                                    # noqa: BLE001  (told to the main thread)
            errors.append(e)

    work(0)
    gate = threading.Barrier(2)
    threads = [threading.Thread(target=work, args=(k, gate)) for k in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert len(results) == 9
    for got in results.values():
        assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_functions_in_place_of_modules_run():
    """An activation given as a function, a norm that is a function: parts of a block that are no modules."""
    from sparseswin3d_amd.layers import MLP
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, False, 5)
    plain = run(feats)
    blk = layer.blocks[0]
    mlp = MLP(96, 384, act=torch.nn.functional.gelu).cuda()
    mlp.load_state_dict(blk.mlp.state_dict())
    blk.mlp = mlp
    assert torch.allclose(run(feats), plain, rtol=1e-4, atol=1e-5)
    norm = blk.norm1
    del blk.norm1
    blk.norm1 = lambda x: torch.nn.functional.layer_norm(x, (96,), norm.weight, norm.bias, norm.eps)
    assert torch.allclose(run(feats), plain, rtol=1e-4, atol=1e-5)
    norm2, blk2 = layer.blocks[1].norm2, layer.blocks[1]
    del blk2.norm2
    blk2.norm2 = lambda x: torch.nn.functional.layer_norm(x, (96,), norm2.weight, norm2.bias, norm2.eps)
    assert torch.allclose(run(feats), plain, rtol=1e-4, atol=1e-5)
