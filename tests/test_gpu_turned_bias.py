"""Window-resident attention from a relative position table (its kernels read the bias turned as well) against the same attention
from the [H, n, n] bias gathered by torch: the same values meet in the same order, so every bit agrees."""
import numpy as np
import pytest
import torch

from helpers import ragged_window_indices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window,counts", [((1, 1, 1), [1, 1]), ((3, 3, 3), [1, 2, 15, 16, 17, 27]), ((4, 4, 8), [1, 128, 31, 32, 33, 64, 65, 96, 97, 127, 5])],
                         ids=["1", "27", "128"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("use_mask", [False, True], ids=["plain", "mask"])
def test_attention_from_the_table_equals_attention_from_the_bias(window, counts, dtype, use_mask):
    from sparseswin3d_amd import _lib
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    n, H, hd = int(np.prod(window)), 3, 32
    rng = np.random.default_rng(n)
    ind = torch.from_numpy(ragged_window_indices(rng, counts, n)).cuda()
    rows = int(np.prod([2 * w - 1 for w in window]))
    index = relative_position_index_3d(window).cuda()
    ti = BiasTableIndex.build(index, rows)
    torch.manual_seed(n)
    qkv, up = torch.randn(len(ind), 3, H, hd).to(dtype).cuda(), torch.randn(len(ind), H * hd).to(dtype).cuda()
    table = torch.randn(rows, H).to(dtype).cuda()
    mask = torch.from_numpy(rng.integers(0, 27, (len(counts), n)).astype(np.int8)).cuda() if use_mask else None
    results = []
    for bias, code in ((table, ti.code), (table.float()[index.reshape(-1).long()].view(n, n, H).permute(2, 0, 1).contiguous(), None)):
        x = qkv.clone().requires_grad_(True)
        plan = TokenPlan(ind, len(counts), n, H)
        out = _lib.native().attention(x, bias, plan.native, mask, code, ti.offset0, n, hd ** -0.5, "resident")
        out.backward(up)
        results.append((out.detach(), x.grad))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("coded", [True, False], ids=["table", "bias"])
def test_a_saved_bias_of_another_size_is_refused(coded):
    """The backward reads one or two biases by whether positions are coded: a hook on saved tensors that gives back the other number
    is an error, in front of the launch."""
    from sparseswin3d_amd import _lib
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    n, H, hd, rows = 27, 3, 32, 125
    ind = torch.from_numpy(ragged_window_indices(np.random.default_rng(0), [3, 27], n)).cuda()
    ti = BiasTableIndex.build(relative_position_index_3d((3, 3, 3)).cuda(), rows)
    bias = torch.randn(rows, H, device="cuda") if coded else torch.randn(H, n, n, device="cuda")

    def other(t):
        return t[0] if coded and t.dim() == 4 else torch.stack([t, t]) if not coded and t.shape == (H, n, n) else t
    x = torch.randn(len(ind), 3, H, hd, device="cuda", requires_grad=True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, other):
        out = _lib.native().attention(x, bias, TokenPlan(ind, 2, n, H).native, None, ti.code if coded else None, ti.offset0, n, hd ** -0.5, "resident")
    with pytest.raises(RuntimeError, match="saved bias"):
        out.backward(torch.ones_like(out))
