"""The flash backward with and without the table's gradient.  Chunks of 32 tokens: a frozen table takes the query side that forms the scores again, a
trained one dQ from the stored dS.  A wavefront a window and head: a frozen table leaves out the sums.  Both sum the same fp32 terms in another order (at most 384 of them: 2e-5 of the gradient's norm; 16-bit results
then differ where that crosses a rounding boundary, 1e-3 and 3e-3)."""
import numpy as np
import pytest
import torch

from helpers import ragged_window_indices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,n", [([1, 2, 31, 1, 33, 5, 16, 17, 1], 125), ([343, 129, 1, 31, 65, 5, 5, 256, 32, 64], 343)], ids=["small", "large"])
@pytest.mark.parametrize("hd,dtype,family", [(16, torch.float32, "flash_chunks"), (16, torch.float32, "flash_windows"), (16, torch.float16, "flash_chunks"),
                                             (16, torch.float16, "flash_windows"), (32, torch.bfloat16, "flash")], ids=lambda v: str(v).replace("torch.", ""))
@pytest.mark.parametrize("use_mask", [False, True], ids=["plain", "mask"])
def test_gradient_of_qkv_with_and_without_a_stored_ds(counts, n, hd, dtype, family, use_mask):
    from sparseswin3d_amd import _lib
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    w, H = round(n ** (1 / 3)), 3
    rng = np.random.default_rng(hd)
    ind = torch.from_numpy(ragged_window_indices(rng, counts, n)).cuda()
    ti = BiasTableIndex.build(relative_position_index_3d((w, w, w)).cuda(), (2 * w - 1) ** 3)
    torch.manual_seed(hd)
    qkv, up = torch.randn(len(ind), 3, H, hd).to(dtype).cuda(), torch.randn(len(ind), H * hd).to(dtype).cuda()
    table = torch.randn((2 * w - 1) ** 3, H).cuda()
    mask = torch.from_numpy(rng.integers(0, 27, (len(counts), n)).astype(np.int8)).cuda() if use_mask else None
    grads = []
    for trained in (True, False):
        x, t = qkv.clone().requires_grad_(True), table.clone().requires_grad_(trained)
        plan = TokenPlan(ind, len(counts), n, H)
        _lib.native().attention(x, t, plan.native, mask, ti.code, ti.offset0, n, hd ** -0.5, family).backward(up)
        assert (t.grad is not None) == trained
        grads.append(x.grad.double())
    rel = ((grads[0] - grads[1]).norm() / grads[1].norm()).item()
    assert rel < {torch.float32: 2e-5, torch.float16: 1e-3, torch.bfloat16: 3e-3}[dtype], rel
