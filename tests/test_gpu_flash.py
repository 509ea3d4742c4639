"""The attention kernels for heads of 16 / 32 channels and windows of any size (``sswin_flash_*``) against the block products
with the attention matrix in memory (the other implementation of the same softmax), all gradients included.  Heads of 16 have two
families, chunks of 32 tokens and a wavefront a window and head; each is asked for by its name.

fp32: both carry fp32 rounding of sums of at most 384 terms (2e-5 of a result's norm, bias gradient included).  16-bit tokens: P, dS
and all sums are fp32 in both, so results differ where 2e-5 crosses a rounding boundary: a share 2e-5 x 2^11 (fp16) or 2^8 (bf16) of
the values, by an ulp, 1e-4 or 3e-4 of the norm; dP - D subtracts such numbers, up to ten times their result."""
import numpy as np
import pytest
import torch

from helpers import random_window_indices, ragged_window_indices

pytestmark = pytest.mark.gpu

MIXES = {
    "tiny": ([1, 2, 3, 1, 0, 5, 31, 1, 1, 7, 9, 15, 16, 17, 2, 1], 125),          # many windows in one block
    "edges": ([32, 33, 31, 63, 64, 65, 16, 48, 1, 125, 0, 96, 97], 125),
    "large": ([343, 129, 1, 200, 31, 256, 257, 5, 5, 5, 30, 343, 128], 343),
    "one": ([1], 27),
}


BOTH = ["flash_chunks", "flash_windows"]


@pytest.mark.parametrize("mix", list(MIXES))
@pytest.mark.parametrize("hd,dtype,family", [(hd, dtype, f) for hd, dtype in ((16, torch.float32), (32, torch.float32), (16, torch.float16), (16, torch.bfloat16),
                                                                              (32, torch.bfloat16)) for f in (BOTH if hd == 16 else ["flash"])],
                         ids=lambda v: str(v).replace("torch.", ""))
@pytest.mark.parametrize("use_mask", [False, True], ids=["plain", "mask"])
def test_flash_against_block_products(mix, hd, dtype, family, use_mask):
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan, attention_path, fused_window_attention
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    counts, n = MIXES[mix]
    w = round(n ** (1 / 3))
    H = 3
    rng = np.random.default_rng(len(counts) + hd)
    ind = torch.from_numpy(ragged_window_indices(rng, counts, n)).cuda()
    ti = BiasTableIndex.build(relative_position_index_3d((w, w, w)).cuda(), (2 * w - 1) ** 3)
    assert attention_path(hd, n, ti, None) == ("flash" if hd == 16 or n > 128 else "resident")
    torch.manual_seed(hd)
    qkv = (torch.randn(len(ind), 3, H, hd) * 1.5).to(dtype).cuda()
    qkv[::7] *= 6                                                  # some rows with large scores: the running offset moves
    table = torch.randn((2 * w - 1) ** 3, H).cuda()
    mask = torch.from_numpy(rng.integers(0, 27, (len(counts), n)).astype(np.int8)).cuda() if use_mask else None
    up = torch.randn(len(ind), H * hd).to(dtype).cuda()
    got = []
    from sparseswin3d_amd import _lib
    for path in (family, "products"):
        x, t = qkv.clone().requires_grad_(True), table.clone().requires_grad_(True)
        plan = TokenPlan(ind, len(counts), n, H)
        out = _lib.native().attention(x, t, plan.native, mask, ti.code, ti.offset0, n, hd ** -0.5, path)
        out.backward(up)
        got.append((out.detach(), x.grad, t.grad))
        with torch.no_grad():
            assert torch.equal(_lib.native().attention(qkv, table, plan.native, mask, ti.code, ti.offset0, n, hd ** -0.5, path), out)
    tol = {torch.float32: 2e-5, torch.float16: 1e-3, torch.bfloat16: 3e-3}[dtype]
    for a, b, what in zip(*got, ("out", "d qkv", "d table")):
        assert not torch.isnan(a).any(), what
        # a lone token's dS is zero up to the rounding of dP - D, two numbers of order ten: held to the bound of a result of norm 1
        rel = ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1.0)).item()
        assert rel < tol, (what, rel)


@pytest.mark.parametrize("family", BOTH)
def test_flash_many_windows_and_heads(family):
    """Workgroups in whole rounds over the XCDs and in the remainder; head and chunk numbers of every workgroup."""
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    from sparseswin3d_amd import _lib
    rng = np.random.default_rng(0)
    ti = BiasTableIndex.build(relative_position_index_3d((5, 5, 5)).cuda(), 729)
    for N, H in ((2600, 5), (257, 2), (20000, 1)):
        ind = torch.from_numpy(random_window_indices(rng, 700, 125, N)).cuda()
        qkv, table = torch.randn(N, 3, H, 16).cuda(), torch.randn(729, H).cuda()
        plan = TokenPlan(ind, 700, 125, H)
        a, b = (_lib.native().attention(qkv, table, plan.native, None, ti.code, ti.offset0, 125, 0.25, p) for p in (family, "products"))
        assert ((a - b).norm() / b.norm()).item() < 1e-5, (N, H)


@pytest.mark.parametrize("family", BOTH)
def test_flash_fp16_gradients_outside_the_range_of_fp16(family):
    """dS beyond 65504 (two tokens a window, dO of 15000) while every result is finite in fp16: dS has to stay fp32."""
    from sparseswin3d_amd import _lib
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    ti = BiasTableIndex.build(relative_position_index_3d((5, 5, 5)).cuda(), 729)
    ind = torch.from_numpy(ragged_window_indices(np.random.default_rng(3), [2] * 400, 125)).cuda()
    torch.manual_seed(3)
    qkv = torch.randn(len(ind), 3, 2, 16)
    qkv[:, :2] *= 0.02
    qkv[:, 2] *= 2
    qkv, up = qkv.half().cuda(), (torch.randn(len(ind), 32) * 15000).clamp(-6e4, 6e4).half().cuda()
    table = torch.zeros(729, 2).cuda()
    got = []
    for path in (family, "products"):
        x = qkv.clone().requires_grad_(True)
        plan = TokenPlan(ind, 400, 125, 2)
        _lib.native().attention(x, table, plan.native, None, ti.code, ti.offset0, 125, 0.25, path).backward(up)
        got.append(x.grad.double())
    assert torch.isfinite(got[1]).all()
    assert ((got[0] - got[1]).norm() / got[1].norm()).item() < 1e-3     # an ulp of fp16 at most


def _float64(qkv, table, index, ind, scale, up):
    """Output and gradients of qkv in float64, window by window; what is not finite stays where the formulas put it."""
    N, _, H, hd = qkv.shape
    x, t, d_o = qkv.double().cpu(), table.double().cpu(), up.double().cpu().view(N, H, hd)
    out, d = torch.empty(N, H, hd, dtype=torch.float64), torch.empty_like(x)
    for w in ind[:, 0].unique():
        rows = (ind[:, 0] == w).nonzero()[:, 0]
        pos = ind[rows, 1].long()
        for h in range(H):
            q, k, v = (x[rows, i, h] for i in range(3))
            s = scale * (q @ k.T) + t[index[pos][:, pos], h]
            e = torch.exp(s - s.amax(1, keepdim=True).clamp_min(0))
            p = e / (e.sum(1, keepdim=True) + 1e-8)
            o, g = p @ v, d_o[rows, h]
            ds = p * (g @ v.T - (g * o).sum(1, keepdim=True))
            out[rows, h] = o
            d[rows, 0, h], d[rows, 1, h], d[rows, 2, h] = scale * ds @ k, scale * ds.T @ q, p.T @ g
    return out.view(N, -1), d


@pytest.mark.parametrize("which", ["q", "k", "v", "dO"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")], ids=["inf", "nan"])
@pytest.mark.parametrize("hd,dtype,family", [(hd, dtype, f) for hd, dtype in ((16, torch.float32), (32, torch.float32), (16, torch.float16), (32, torch.bfloat16))
                                             for f in (BOTH if hd == 16 else ["flash"])], ids=lambda v: str(v).replace("torch.", ""))
def test_flash_keeps_what_is_not_finite_where_it_belongs(which, value, hd, dtype, family):
    """One channel of one token of a few windows is not finite: other windows keep their results, whichever windows share a block
    with them, and inside the window infinities and NaN stand where float64 has them.  Bounds of finite values: as above, per
    result (5 x the norm's bound, at a norm of one token's row)."""
    from sparseswin3d_amd import _lib
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    counts, n, H = [3, 1, 2, 5, 31, 1, 7, 9, 15, 17, 1, 2, 4, 33, 40, 3, 3, 64, 100, 2, 2, 200], 343, 2
    index = relative_position_index_3d((7, 7, 7))
    ti = BiasTableIndex.build(index.cuda(), 13 ** 3)
    ind = torch.from_numpy(ragged_window_indices(np.random.default_rng(hd), counts, n))
    torch.manual_seed(hd)
    qkv, up = torch.randn(len(ind), 3, H, hd).to(dtype), torch.randn(len(ind), H * hd).to(dtype)
    table = torch.randn(13 ** 3, H) * 0.3
    hit = [int((ind[:, 0] == w).nonzero()[-1]) for w in (3, 6, 13, 15, 18, 21)]
    for r in hit:
        if which == "dO":
            up[r, hd + 3] = value                                 # of head 1
        else:
            qkv[r, "qkv".index(which), 1, 3] = value
    x = qkv.cuda().requires_grad_(True)
    plan = TokenPlan(ind.cuda(), len(counts), n, H)
    out = _lib.native().attention(x, table.cuda(), plan.native, None, ti.code, ti.offset0, n, hd ** -0.5, family)
    out.backward(up.cuda())
    ref = _float64(qkv, table, index, ind, hd ** -0.5, up)
    tol = {torch.float32: 1e-4, torch.float16: 5e-3, torch.bfloat16: 3e-2}[dtype]
    for got, want, what in zip((out.detach(), x.grad), ref, ("out", "d qkv")):
        got = got.double().cpu()
        finite = want.isfinite()
        assert got[finite].isfinite().all(), what
        assert ((got - want)[finite].abs() <= tol * (1 + want[finite].abs())).all(), what
        assert torch.equal(got[want.isinf()], want[want.isinf()]), what
        assert not got[want.isnan()].isfinite().any(), what
    if which != "dO":
        assert not torch.isfinite(out).all()


@pytest.mark.parametrize("counts,chosen", [([19] * 300, 0), ([21] * 300, 1), ([1] * 200 + [343] * 3, 1), ([1] * 400 + [343], 0), ([2] * 16385, 0), ([40] * 16385, 0)],
                         ids=["19", "21", "few-large", "one-large", "many-small", "many"])
def test_flash_family_by_the_tokens_of_windows(counts, chosen):
    """What the path takes by itself: a wavefront a window where that is faster, and at most 16 384 windows.  Its bits are those of that family."""
    from sparseswin3d_amd import _lib
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    ti = BiasTableIndex.build(relative_position_index_3d((7, 7, 7)).cuda(), 13 ** 3)
    ind = torch.from_numpy(ragged_window_indices(np.random.default_rng(0), counts, 343)).cuda()
    qkv, table, up = torch.randn(len(ind), 3, 1, 16).cuda(), torch.randn(13 ** 3, 1).cuda(), torch.randn(len(ind), 16).cuda()
    plan = TokenPlan(ind, len(counts), 343, 1)
    got = {}
    for path in ("flash", "flash_chunks") + (("flash_windows",) if len(counts) <= 16384 else ()):
        x, t = qkv.clone().requires_grad_(True), table.clone().requires_grad_(True)
        out = _lib.native().attention(x, t, plan.native, None, ti.code, ti.offset0, 343, 0.25, path)
        out.backward(up)
        got[path] = (out.detach(), x.grad, t.grad)
    assert all(torch.equal(a, b) for a, b in zip(got["flash"], got[BOTH[chosen]]))
    if "flash_windows" in got:
        assert not torch.equal(got["flash_chunks"][0], got["flash_windows"][0])
    else:
        with pytest.raises(RuntimeError):
            _lib.native().attention(qkv, table, plan.native, None, ti.code, ti.offset0, 343, 0.25, "flash_windows")


# chunks of 32 tokens: one, some threads without any, several a thread, the most an order holds; windows that fill, span and share
# chunks; more windows than an order takes, which leaves the chunks as they are
@pytest.mark.parametrize("N,sizes", [(1, "all"), (32, "all"), (33, "all"), (1000, "all"), (34001, "all"), (12288 * 32, "all"), (40000, "small")])
@pytest.mark.parametrize("H", [1, 3])
def test_flash_order_of_the_work(N, sizes, H):
    """The order holds every chunk once, by descending work, and results have the bits they have without one."""
    import ctypes as C
    from sparseswin3d_amd import _lib
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    lib, n = _lib.load(), 343
    rng = np.random.default_rng(N)
    counts, left = [], N
    while left:
        counts.append(int(min(rng.choice([1, 5, 20, 31, 32, 33, 64, 100, 250, 343] if sizes == "all" else [1, 2, 3]), left)))
        left -= counts[-1]
    ind = torch.from_numpy(ragged_window_indices(rng, counts, n)).cuda()
    ti = BiasTableIndex.build(relative_position_index_3d((7, 7, 7)).cuda(), 2197)
    plan = TokenPlan(ind, len(counts), n, H).native
    plan._finish()
    ptr = lambda t: C.c_void_p(t.data_ptr())
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    D = 16 * H
    qkv, d_o, table = torch.randn(N, 3 * D).cuda(), torch.randn(N, D).cuda(), torch.randn(2197, H).cuda()
    chunks, got = (N + 31) // 32, []
    assert lib.sswin_flash_order_ints(N, H) == (chunks if H * chunks > 12 * torch.cuda.get_device_properties(0).multi_processor_count else 0)
    for order in (None, torch.full((chunks,), -1, dtype=torch.int32, device="cuda")):
        words = torch.empty(2 * N, dtype=torch.int32, device="cuda")
        out, lse, d_qkv, delta = torch.empty(N, D).cuda(), torch.empty(H, N).cuda(), torch.empty(N, 3 * D).cuda(), torch.empty(H, N).cuda()
        d_s, o, sq = torch.empty(max(plan.A, 1)).cuda(), None if order is None else ptr(order), C.c_void_p(words.data_ptr() + 4 * N)
        _lib.check(lib.sswin_flash_tokens_ordered(ptr(plan.plan), plan.g_cap, plan.G, ptr(plan.tokens), N, H, n, ptr(ti.code), None, 0, ptr(words), sq, o, stream))
        _lib.check(lib.sswin_flash_forward_ordered(0, ptr(plan.tokens), ptr(words), o, N, H, 16, n, ptr(qkv), 0.25, ptr(table), 2197, ti.offset0, ptr(out), ptr(lse),
                                                   stream))
        _lib.check(lib.sswin_flash_backward_ordered(0, ptr(plan.tokens), ptr(words), sq, o, N, H, 16, n, ptr(qkv), 0.25, ptr(table), 2197, ti.offset0, ptr(out),
                                                    ptr(lse), ptr(d_o), ptr(d_qkv), ptr(delta), ptr(d_s), stream))
        got.append((words, out, lse, d_qkv, d_s[:plan.A]))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    assert torch.equal(order.sort()[0].cpu(), torch.arange(chunks, dtype=torch.int32))
    cost, T = np.zeros(chunks, dtype=np.int64), 0
    for c in counts:                                               # steps of 16 over the window: two, three with a second sub-tile, two a block
        if c < 32:
            cost[T // 32] += (c + 7) // 8
        else:
            for j in range(0, c, 32):
                cost[(T + j) // 32] += (c + 15) // 16 * (3 if c - j > 16 else 2) + 2
        T += c
    assert np.array_equal(order.cpu().numpy(), np.argsort(15 - np.minimum(cost // 4, 15), kind="stable") if len(counts) <= 16384 else np.arange(chunks))
    with pytest.raises(RuntimeError):
        big = 12288 * 32 + 1
        _lib.check(lib.sswin_flash_tokens_ordered(ptr(plan.plan), plan.g_cap, plan.G, ptr(plan.tokens), big, H, n, ptr(ti.code), None, 0, ptr(words), sq, o, stream))
