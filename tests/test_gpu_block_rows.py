"""Compiled blocks with as many rows as the launches for many rows take (the feed-forward part as one launch, 16-bit layers that
read their rows once): against the same stage composed of its modules, and on streams and threads of their own."""
import functools

import pytest
import torch

import test_gpu_single_nodes as nodes
from test_gpu_dense import _stage_pieces

pytestmark = pytest.mark.gpu

# ragged behind the last full tile of 32 rows and behind the last full round of workgroups; windows four fifths full
MANY = dict(grid=(32, 32, 24), n=20001)
CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


def _takes_the_launches(dim, compute):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    assert lib.sswin_mlp_preferred(CODE[compute], MANY["n"], dim, 4 * dim)


# 48 channels: only 16 bit is one launch there; the frozen forms are wired alike for both widths
FORMS = [(96, 3, 5, mode, variant) for mode in ("fp32", "bf16", "amp")
         for variant in ("all", "frozen first layer", "frozen second layer", "frozen biases", "no biases")]
FORMS += [(48, 3, 7, mode, variant) for mode in ("bf16", "amp") for variant in ("all", "no biases")]


@pytest.mark.parametrize("dim,heads,window,mode,variant", FORMS)
def test_stage_of_many_rows_equals_its_composition(dim, heads, window, mode, variant, monkeypatch):
    """Tolerances: those of the same comparison on few rows (fp32 2e-5 of a result's norm: chains of fp32 sums; 16 bit: roundings
    to the type, one intermediate fewer in the compiled block)."""
    from sparseswin3d_amd import layers
    dtype = torch.bfloat16 if mode == "bf16" else torch.float32
    _takes_the_launches(dim, {"fp32": torch.float32, "bf16": torch.bfloat16, "amp": torch.float16}[mode])
    layer, run, feats = _stage_pieces(dim, heads, window, dtype, False, dim + window, **MANY)
    for block in layer.blocks:
        first, second = block.mlp.linear1, block.mlp.linear2
        if variant == "no biases":
            first.bias = second.bias = None
        for p in {"frozen first layer": [first.weight, first.bias], "frozen second layer": [second.weight, second.bias],
                  "frozen biases": [first.bias, second.bias]}.get(variant, []):
            p.requires_grad_(False)
    results = []
    for single in (True, False):
        if not single:
            monkeypatch.setattr(layers, "_fused_dtype", lambda *a: None)
        layer.zero_grad(set_to_none=True)
        x = feats.clone().requires_grad_(True)
        with torch.autocast("cuda", dtype=torch.float16, enabled=mode == "amp"):
            y = run(x)
        gen = torch.Generator(device="cuda").manual_seed(1)
        up = torch.randn(y.shape, generator=gen, device="cuda").to(y.dtype)
        assert ("BlockNode" in y.grad_fn.name()) == single, y.grad_fn.name()
        assert y.dtype == dtype                                   # mixed precision: the residual stream stays fp32
        y.backward(up)
        results.append([("out", y.detach()), ("dx", x.grad)] + [(k, p.grad) for k, p in layer.named_parameters()])
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, enabled=mode == "amp"):
            assert not single or torch.equal(run(feats), y.detach()), "inference"
    tol = {"fp32": 2e-5, "bf16": 4e-2, "amp": 8e-3}[mode]
    for (k, a), (_, b) in zip(*results):
        assert (a is None) == (b is None), k
        if a is None:
            continue
        assert a.dtype == b.dtype and a.shape == b.shape, k
        rel = ((a.double() - b.double()).norm() / b.double().norm()).item()
        assert rel < tol, (k, rel)


@pytest.mark.parametrize("dim,heads,window,mode", [(96, 3, 5, "fp32"), (48, 3, 7, "amp"), (96, 3, 5, "bf16")])
def test_nodes_of_many_rows_on_other_streams(dim, heads, window, mode, monkeypatch):
    _takes_the_launches(dim, {"fp32": torch.float32, "bf16": torch.bfloat16, "amp": torch.float16}[mode])
    monkeypatch.setattr(nodes, "_stage_pieces", functools.partial(_stage_pieces, **MANY))
    nodes.test_nodes_on_other_streams(dim, heads, window, mode)
