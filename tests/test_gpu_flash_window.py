"""The attention kernels that take a window and head a wavefront (``sswin_flash_window_*``) against float64, window by window: output, gradients of q, k
and v and of the bias table, where rows of a window lie far apart, where something is not finite, and at the edges of tiles and of a
wavefront's share.

Bounds: fp32 sums of at most 384 terms, 2e-5 of the norm of a window's result; 16-bit results carry half an ulp, at most 2^-11 (fp16) and 2^-8 (bf16) of
themselves.  D = dO . O is formed from the output as it was rounded, in float64 too."""
import numpy as np
import pytest
import torch

from helpers import ragged_window_indices

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 2e-5, torch.float16: 5e-4, torch.bfloat16: 4e-3}


def _case(counts, n, H, dtype, seed, regions=None, shape=None):
    from sparseswin3d_amd.fused import BiasTableIndex, TokenPlan
    from sparseswin3d_amd.window_attention import relative_position_index_3d
    shape = shape or (round(n ** (1 / 3)),) * 3
    rows = int(np.prod([2 * w - 1 for w in shape]))
    index = relative_position_index_3d(shape)
    ti = BiasTableIndex.build(index.cuda(), rows)
    ind = torch.from_numpy(ragged_window_indices(np.random.default_rng(seed), counts, n))
    torch.manual_seed(seed)
    qkv, up = torch.randn(len(ind), 3, H, 16).to(dtype), torch.randn(len(ind), H * 16).to(dtype)
    table = torch.randn(rows, H) * 0.5
    mask = torch.from_numpy(np.random.default_rng(seed).integers(0, regions, (len(counts), n)).astype(np.int8)) if regions else None
    return ti, index, ind, qkv, up, table, mask, TokenPlan(ind.cuda(), len(counts), n, H)


def _run(ti, ind, qkv, up, table, mask, plan, n):
    from sparseswin3d_amd import _lib
    x, t = qkv.cuda().requires_grad_(True), table.cuda().requires_grad_(True)
    out = _lib.native().attention(x, t, plan.native, None if mask is None else mask.cuda(), ti.code, ti.offset0, n, 0.25, "flash_windows")
    out.backward(up.cuda())
    return out.detach(), x.grad, t.grad


def _float64(index, ind, qkv, up, table, mask, rounded=None):
    """rounded: the output that D is formed from, float64's own if there is none."""
    N, _, H, hd = qkv.shape
    rounded = None if rounded is None else rounded.double().cpu().view(N, H, hd)
    x, t, d_o = qkv.double(), table.double(), up.double().view(N, H, hd)
    out, d, d_t = torch.zeros(N, H, hd, dtype=torch.float64), torch.zeros_like(x), torch.zeros_like(t)
    for w in ind[:, 0].unique():
        rows = (ind[:, 0] == w).nonzero()[:, 0]
        pos = ind[rows, 1].long()
        at = index[pos][:, pos].long()
        q, k, v = (x[rows, i].transpose(0, 1) for i in range(3))
        s = 0.25 * (q @ k.transpose(1, 2)) + t[at].permute(2, 0, 1)
        if mask is not None:
            r = mask[int(w)][pos]
            s = s - 100.0 * (r[:, None] != r[None]).double()
        e = torch.exp(s - s.amax(2, keepdim=True).clamp_min(0))
        p = e / (e.sum(2, keepdim=True) + 1e-8)
        o, g = p @ v, d_o[rows].transpose(0, 1)
        ds = p * (g @ v.transpose(1, 2) - (g * (o if rounded is None else rounded[rows].transpose(0, 1))).sum(2, keepdim=True))
        out[rows] = o.transpose(0, 1)
        for i, m in enumerate((0.25 * ds @ k, 0.25 * ds.transpose(1, 2) @ q, p.transpose(1, 2) @ g)):
            d[rows, i] = m.transpose(0, 1)
        d_t.index_put_((at.reshape(-1),), ds.permute(1, 2, 0).reshape(-1, H), accumulate=True)
    return out, d, d_t


def _check(got, want, ind, dtype, floor=0.0):
    """Per window, result and head: norm of the difference against the norm of the result (`floor`: against that at least)."""
    N, _, H, hd = want[1].shape
    out, d, d_t = got[0].double().cpu().view(N, H, hd), got[1].double().cpu().view(N, 3, H, hd), got[2].double().cpu()
    pairs = [(out, want[0], "out")] + [(d[:, i], want[1][:, i], name) for i, name in enumerate(("dq", "dk", "dv"))]
    for w in ind[:, 0].unique():
        rows = ind[:, 0] == w
        for a, b, name in pairs:
            diff, norm = (a[rows] - b[rows]).norm(dim=(0, 2)), b[rows].norm(dim=(0, 2)).clamp_min(floor)
            assert (diff <= TOL[dtype] * norm).all(), (name, int(w), (diff / norm).max().item())
    diff, norm = (d_t - want[2]).norm(dim=0), want[2].norm(dim=0)
    assert (diff <= TOL[dtype] * norm).all(), ("table", (diff / norm).max().item())


# tiles and their remainders, the most of one, two and four wavefronts and one more, the most there is; several windows of a kind in a workgroup
EDGES = [1, 2, 15, 16, 17, 31, 33, 64, 65, 80, 95, 96, 96, 97, 97, 97, 112, 191, 192, 193, 193, 255, 300, 343, 5, 5, 5, 5, 5]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("regions", [None, 1, 3], ids=["plain", "one-region", "regions"])
def test_windows_at_the_edges(dtype, regions):
    ti, index, ind, qkv, up, table, mask, plan = _case(EDGES, 343, 3, dtype, 1, regions)
    got = _run(ti, ind, qkv, up, table, mask, plan, 343)
    # a lone token's dS is zero up to the rounding of dP - D, two numbers of order ten
    _check(got, _float64(index, ind, qkv, up, table, mask, got[0]), ind, dtype, floor=10.0)
    for again in range(2):                                         # the table's sums too, whatever order the wavefronts add in
        assert all(torch.equal(a, b) for a, b in zip(got, _run(ti, ind, qkv, up, table, mask, plan, 343)))


@pytest.mark.parametrize("shape", [(6, 8, 8), (1, 1, 3), (2, 12, 16)])
def test_windows_of_other_shapes(shape):
    """The largest table of 384 positions, the most that two workgroups of a unit find LDS for; a few rows; sides far apart."""
    n = int(np.prod(shape))
    counts = [c for c in (1, 17, 96, 200, 384) if c <= n] + [n] * 3
    ti, index, ind, qkv, up, table, mask, plan = _case(counts, n, 3, torch.float32, 10, shape=shape)
    got = _run(ti, ind, qkv, up, table, mask, plan, n)
    _check(got, _float64(index, ind, qkv, up, table, mask, got[0]), ind, torch.float32, floor=10.0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("what", ["q row", "k row", "v row", "dO row", "dO rows", "windows", "zeros", "growing"])
def test_rows_far_apart(dtype, what):
    """Rows of a window, or whole windows, by powers of two apart: each window's results are held to its own norm."""
    counts = [40, 96, 97, 200, 16, 64, 33, 343]
    ti, index, ind, qkv, up, table, mask, plan = _case(counts, 343, 2, dtype, 2)
    big = 2.0 ** (24 if dtype != torch.float16 else 6)
    rows = [int((ind[:, 0] == w).nonzero()[c // 2]) for w, c in enumerate(counts)]
    if what == "q row":
        qkv[rows, 0] *= big
        qkv[:, 1] /= big                                           # scores of order one for that row, of none for the others
    elif what == "k row":
        qkv[rows, 1] *= big
        qkv[:, 0] /= big
    elif what == "v row":
        qkv[rows, 2] *= big
    elif what == "dO row":
        up[rows] *= big
    elif what == "dO rows":                                        # every other row 2^-14
        up[::2] *= 2.0 ** -14
    elif what == "windows":
        f = torch.tensor([1.0, big, 1.0 / big, 1.0, big, 1.0, 1.0 / big, 1.0])[ind[:, 0].long()]
        up *= f[:, None].to(dtype)
    elif what == "zeros":
        up[::3], qkv[::5, 0], qkv[::7, 1], qkv[::4, 2] = 0, 0, 0, 0
        up[ind[:, 0] == 1] = 0
        qkv[ind[:, 0] == 5] = 0
    else:                                                          # later rows larger: the scales follow
        rank = torch.arange(len(ind))[:, None] % 48
        up *= (2.0 ** (rank / 8)).to(dtype)
        qkv[:, 0] *= (2.0 ** (rank / 24)).to(dtype)[..., None]
    got = _run(ti, ind, qkv, up, table, mask, plan, 343)
    # the least that fp16 tells apart, 6e-8, of every value of a window
    _check(got, _float64(index, ind, qkv, up, table, mask, got[0]), ind, dtype, floor=1e-30 if dtype != torch.float16 else 6e-8 / TOL[dtype] * (343 * 16) ** 0.5)


# A row's own bound.  fp32: sums of at most 384 terms, dP - D of numbers up to ten times their difference, 1e-5; an ulp of a 16-bit result
ROW_TOL = {torch.float32: 1e-5, torch.float16: 2 ** -10, torch.bfloat16: 2 ** -7}


def _check_rows(got, want, rows, dtype, names):
    """Every row and head of the results named, against the norm of that row."""
    N, _, H, hd = want[1].shape
    a = {"out": got[0].double().cpu().view(N, H, hd), **{n: got[1].double().cpu().view(N, 3, H, hd)[:, i] for i, n in enumerate(("dq", "dk", "dv"))}}
    b = {"out": want[0], **{n: want[1][:, i] for i, n in enumerate(("dq", "dk", "dv"))}}
    for name in names:
        rel = ((a[name] - b[name])[rows].norm(dim=2) / b[name][rows].norm(dim=2)).max().item()
        assert rel <= ROW_TOL[dtype], (name, rel)


@pytest.mark.parametrize("dtype,bits", [(torch.float32, (0, 2, 6, 9, 11)), (torch.float16, (0, 6, 11, 17)), (torch.bfloat16, (0, 6, 11, 17, 21))], ids=["fp32", "fp16", "bf16"])
def test_rows_of_small_upstream_gradients(dtype, bits):
    """Every other row of dO 2^-bits of its neighbours, as those of voxels that are classified well: dQ of each row by itself."""
    for k in bits:
        ti, index, ind, qkv, up, table, mask, plan = _case([60, 17, 96, 200, 343], 343, 2, dtype, 5)
        up *= 2.0 ** 10                                            # (so that fp16 results stay above its least normal value)
        up[::2] *= 2.0 ** -k
        got = _run(ti, ind, qkv, up, table, mask, plan, 343)
        _check_rows(got, _float64(index, ind, qkv, up, table, mask, got[0]), slice(0, None), dtype, ("dq", "dk", "dv"))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
def test_mask_regions_of_small_upstream_gradients(dtype):
    """A whole region of a window with dO 2^-9 of the others': its keys meet small rows only.  bf16, whose range has room for it: dO and K 2^-21."""
    for k, keys in ((9, 0),) + (((21, 21),) if dtype == torch.bfloat16 else ()):
        ti, index, ind, qkv, up, table, mask, plan = _case([60, 96, 200, 343], 343, 2, dtype, 6, 2)
        small = mask[ind[:, 0].long(), ind[:, 1].long()] == 1
        up *= 2.0 ** 10
        up[small] *= 2.0 ** -k
        qkv[small, 1] *= 2.0 ** -keys
        got = _run(ti, ind, qkv, up, table, mask, plan, 343)
        _check_rows(got, _float64(index, ind, qkv, up, table, mask, got[0]), slice(0, None), dtype, ("dq", "dk", "dv"))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
def test_keys_that_no_query_attends(dtype):
    """A key in each window whose P is about 2^-20 for every query: its dK and dV; and the output where it alone has values (V = 0 elsewhere)."""
    counts = [60, 96, 200, 343]
    ti, index, ind, qkv, up, table, mask, plan = _case(counts, 343, 2, dtype, 7)
    rows = torch.tensor([int((ind[:, 0] == w).nonzero()[c // 2]) for w, c in enumerate(counts)])
    qkv[:, 0, :, 0] = 4
    qkv[rows, 1] = 0
    qkv[rows, 1, :, 0] = -8
    table *= 0.1
    up *= 2.0 ** 12
    got = _run(ti, ind, qkv, up, table, mask, plan, 343)
    _check_rows(got, _float64(index, ind, qkv, up, table, mask, got[0]), rows, dtype, ("dk", "dv"))
    other = torch.ones(len(ind), dtype=torch.bool)
    other[rows] = False
    qkv[other, 2] = 0
    qkv[rows, 2] *= 2.0 ** 12
    got = _run(ti, ind, qkv, up, table, mask, plan, 343)
    _check_rows(got, _float64(index, ind, qkv, up, table, mask, got[0]), slice(0, None), dtype, ("out",))


@pytest.mark.parametrize("dtype,bits", [(torch.float32, 20), (torch.float16, 12), (torch.bfloat16, 20)], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("head", [0, 1], ids=["same-head", "other-head"])
def test_table_where_single_rows_are_large(dtype, bits, head):
    """A row of dO in one window and one of V in another, 2^bits above the rest: what the table's gradient holds of other windows and heads."""
    counts = [4, 60, 200, 343, 4, 33]
    ti, index, ind, qkv, up, table, mask, plan = _case(counts, 343, 3, dtype, 8)
    first = [int((ind[:, 0] == w).nonzero()[0]) for w in range(len(counts))]
    up[first[0], 3] *= 2.0 ** bits
    qkv[first[4], 2, head, 3] *= 2.0 ** bits
    out, _, got = _run(ti, ind, qkv, up, table, mask, plan, 343)
    got, want = got.double().cpu(), _float64(index, ind, qkv, up, table, mask, out)[2]
    apart = torch.ones(len(table), dtype=torch.bool)               # rows that the two windows add nothing to
    for w in (0, 4):
        pos = ind[ind[:, 0] == w, 1].long()
        apart[index[pos][:, pos].reshape(-1).long()] = False
    for h in range(3):
        diff, norm = (got - want)[apart, h].norm(), want[apart, h].norm()
        assert diff <= TOL[dtype] * norm, (h, (diff / norm).item())


@pytest.mark.parametrize("heads", [1, 5, 24, 128])
def test_table_by_heads_of_all_sizes(heads):
    """Heads by powers of two apart, and voxel counts that do not divide by what a launch holds: each head's gradient by its own norm."""
    ti, index, ind, qkv, up, table, mask, plan = _case([60, 17, 96, 9], 343, heads, torch.float32, 9)
    size = 2.0 ** (torch.arange(heads) * 37 % 48 - 24).float()
    up *= size.repeat_interleave(16)
    qkv[:, 2] *= size.flip(0)[:, None]
    got = _run(ti, ind, qkv, up, table, mask, plan, 343)
    _check(got, _float64(index, ind, qkv, up, table, mask, got[0]), ind, torch.float32)


@pytest.mark.parametrize("which", ["q", "k", "v", "dO"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")], ids=["inf", "nan"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
def test_table_where_something_is_not_finite(which, value, dtype):
    """Rows of the table that no such dS is added to keep their sums; the others are not finite."""
    counts = [40, 96, 130, 343, 5]
    ti, index, ind, qkv, up, table, mask, plan = _case(counts, 343, 2, dtype, 3)
    for w in (0, 2):
        r = int((ind[:, 0] == w).nonzero()[-1])
        if which == "dO":
            up[r, 16 + 3] = value
        else:
            qkv[r, "qkv".index(which), 1, 3] = value
    out, _, got = _run(ti, ind, qkv, up, table, mask, plan, 343)
    got, want = got.double().cpu(), _float64(index, ind, qkv, up, table, mask, out)[2]
    finite = want.isfinite()
    assert finite[:, 0].all() and finite.any() and not finite.all()
    assert got[finite].isfinite().all() and not got[~finite].isfinite().any()
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    for h in range(2):
        f = finite[:, h]
        assert (got[f, h] - want[f, h]).norm() <= TOL[dtype] * want[f, h].norm()


def test_what_the_kernels_take():
    """Heads of 16, at most 384 positions, 128 heads, 16 384 windows; anything else is left to the other kernels, and refused here."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    size = lib.sswin_flash_window_list_ints
    assert size(0, 1000, 3, 16, 343, 2197, 20) > 0 and size(2, 1000, 128, 16, 384, 4096, 16384) > 0
    for dtype, N, H, hd, n, rows, windows in ((0, 1000, 3, 32, 343, 2197, 20), (0, 1000, 3, 16, 385, 2197, 20), (0, 1000, 129, 16, 343, 2197, 20),
                                              (0, 20000, 3, 16, 343, 2197, 16385), (0, 1000, 3, 16, 343, 4097, 20), (0, 0, 3, 16, 343, 2197, 0),
                                              (0, 8000000, 3, 16, 343, 2197, 20), (3, 1000, 3, 16, 343, 2197, 20)):
        assert size(dtype, N, H, hd, n, rows, windows) == 0
    assert lib.sswin_flash_window_forward(0, None, 60, 60, None, None, None, 1000, 3, 16, 343, None, 0.25, None, 2197, 1098, None, None, None) != 0


@pytest.mark.parametrize("windows,n,H", [(3000, 27, 1), (300, 27, 7), (200, 343, 128)])
def test_many_windows_and_heads(windows, n, H):
    """More pieces of work than a wavefront's lanes hold, heads that do not divide the workgroups, the most heads."""
    rng = np.random.default_rng(windows)
    counts = rng.integers(1, 4 if H == 128 else n + 1, windows).tolist()
    ti, index, ind, qkv, up, table, mask, plan = _case(counts, n, H, torch.float32, 4)
    got = _run(ti, ind, qkv, up, table, mask, plan, n)
    want = _float64(index, ind, qkv, up, table, mask)
    for a, b in zip(got, want):
        assert (a.double().cpu().view(b.shape) - b).norm() <= 2e-5 * b.norm()
