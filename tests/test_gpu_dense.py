"""GPU parity of the dense layers with a folded last step (``sswin_dense_*``), of the row norm (``sswin_layer_norm_*``) and
of the modules' compiled host path against float64 arithmetic on the same inputs.

Bounds: fp32 products are held to 1e-6 of the sum of the absolute products (what an fp32 GEMM reaches); 16-bit results to
one rounding of the result (2^-8 bf16, 2^-11 fp16) plus the same 1e-6; a last step adds its own value to the scale."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
ROUND = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
PLAIN, GELU, RESIDUAL, SCALE = range(4)


def _ptr(t):
    return C.c_void_p(t.data_ptr() if t is not None else None)


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _rand(gen, *shape, dtype=torch.float32, spread=3):
    # values over several binades, so that every piece of a split carries bits
    return (torch.randn(*shape, generator=gen) * torch.exp2(torch.randint(-spread, spread + 1, shape, generator=gen).float())).to(dtype).cuda()


def _check(got, ref, scale, dtype, what):
    assert not torch.isnan(got).any(), what
    err = (got.double() - ref).abs()
    bound = 1e-6 * scale + ROUND[dtype] * ref.abs() + (2.0 ** -24 if dtype == torch.float16 else 1e-30)
    assert (err <= bound).all(), f"{what}: {(err / bound).max().item():.2f} of the bound"


def _forward(lib, _lib, x, w, b, transposed, epi, extra, out):
    N, K = x.shape
    P = w.shape[1] if transposed else w.shape[0]
    y = torch.full((N, P), float("nan"), dtype=out, device="cuda")
    slope = torch.full((N, P), float("nan"), dtype=out, device="cuda") if epi == GELU else None
    nb = lib.sswin_dense_forward_workspace_bytes(CODE[x.dtype], N, K, P)
    ws = torch.empty(max(nb, 1), dtype=torch.uint8, device="cuda")
    _lib.check(lib.sswin_dense_forward(CODE[x.dtype], CODE[out], transposed, epi, _ptr(x), N, K, _ptr(w), _ptr(b), P,
                                       _ptr(extra), _ptr(y), _ptr(slope), _ptr(ws), nb, _stream()))
    return y, slope


# one row, part of a tile, tile edges, many tiles; reductions of one step, of odd counts of steps, of whole blocks; columns of
# part of a column block and of several; the few-rows kernel and the tiled ones; 96 channels: the kernel with W in LDS; 16 bit:
# shares of the reduction (ragged ones too), eight wavefronts a tile, tiles of 192 columns
SHAPES = [(1, 16, 16), (31, 48, 144), (33, 96, 96), (300, 384, 1152), (129, 1536, 48), (9000, 48, 192), (9001, 112, 208),
          (30000, 96, 288), (20001, 144, 48), (20000, 288, 96), (500, 1552, 384), (1300, 784, 368), (1364, 3072, 96), (8100, 400, 1536)]


@pytest.mark.parametrize("N,K,P", SHAPES)
@pytest.mark.parametrize("dtype,out", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                       (torch.float16, torch.float32)], ids=["fp32", "bf16", "fp16", "fp16-out32"])
def test_dense_forward_and_input_gradient(N, K, P, dtype, out):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(N + 3 * K + 7 * P)
    x, w, b = _rand(gen, N, K, dtype=dtype), (_rand(gen, P, K, spread=1) / K ** 0.5).to(dtype), _rand(gen, P, dtype=dtype)
    extra = _rand(gen, N, P, dtype=out)
    wd = w.double()
    pre = x.double() @ wd.T + b.double()
    mag = x.double().abs() @ wd.abs().T + b.double().abs()
    if out == dtype:
        y, _ = _forward(lib, _lib, x, w, b, 0, PLAIN, None, out)
        _check(y, pre, mag, out, "plain")
        y, slope = _forward(lib, _lib, x, w, b, 0, GELU, None, out)
        cdf = 0.5 * (1 + torch.erf(pre / 2 ** 0.5))
        # |gelu'| < 1.13 and |gelu''| < 0.8: an error of the product passes into both results at most at that size
        _check(y, pre * cdf, 1.13 * mag + pre.abs(), out, "gelu")
        _check(slope, cdf + pre * torch.exp(-0.5 * pre ** 2) / (2 * torch.pi) ** 0.5, 0.8 * mag + 1.2, out, "gelu'")
        dy, f = _rand(gen, N, P, dtype=dtype), _rand(gen, N, K, dtype=dtype)
        dx, _ = _forward(lib, _lib, dy, w, None, 1, PLAIN, None, out)
        ref, dmag = dy.double() @ wd, dy.double().abs() @ wd.abs()
        _check(dx, ref, dmag, out, "input gradient")
        dx, _ = _forward(lib, _lib, dy, w, None, 1, SCALE, f, out)
        _check(dx, ref * f.double(), dmag * f.double().abs(), out, "input gradient times a factor")
    y, _ = _forward(lib, _lib, x, w, b, 0, RESIDUAL, extra, out)
    _check(y, pre + extra.double(), mag + extra.double().abs(), out, "residual")


# rows at the line from which x is read once and in its last, moved tile; columns that end inside a step of 64 or 32
@pytest.mark.parametrize("K,N", [(48, 7999), (48, 8000), (48, 8001), (48, 8095), (96, 16000), (96, 16257), (192, 50000), (192, 50017)])
@pytest.mark.parametrize("P", [16, 48, 64, 144, 240])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
def test_dense_forward_that_reads_its_rows_once(K, N, P, dtype):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(N + 3 * K + 7 * P)
    x, w, b = _rand(gen, N, K, dtype=dtype), (_rand(gen, P, K, spread=1) / K ** 0.5).to(dtype), _rand(gen, P, dtype=dtype)
    pre, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    for bias in (b, None):
        add = 0 if bias is None else bias.double()
        y, _ = _forward(lib, _lib, x, w, bias, 0, PLAIN, None, dtype)
        _check(y, pre + add, mag + abs(add), dtype, "plain")


# 16 bit: on either side of the line up to which a layer takes the few-rows kernel: whole steps of 64 channels with and without GELU, up to 96
# channels, ragged steps, fewer than 96 columns
@pytest.mark.parametrize("K,P,epi,rows", [(192, 192, PLAIN, 56), (192, 768, GELU, 20), (96, 96, RESIDUAL, 260), (96, 384, GELU, 104), (144, 144, PLAIN, 173), (192, 48, RESIDUAL, 260)])
def test_dense_forward_around_the_lines_of_few_rows(K, P, epi, rows):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    dtype = torch.bfloat16
    gen = torch.Generator().manual_seed(K + 3 * P)
    for N in (rows * 128, rows * 128 + 1):
        x, w, b, extra = _rand(gen, N, K, dtype=dtype), (_rand(gen, P, K, spread=1) / K ** 0.5).to(dtype), _rand(gen, P, dtype=dtype), _rand(gen, N, P, dtype=dtype)
        y, _ = _forward(lib, _lib, x, w, b, 0, epi, extra if epi == RESIDUAL else None, dtype)
        pre = x.double() @ w.double().T + b.double()
        mag = x.double().abs() @ w.double().abs().T + b.double().abs()
        if epi == GELU:
            pre, mag = pre * 0.5 * (1 + torch.erf(pre / 2 ** 0.5)), 1.13 * mag + pre.abs()
        elif epi == RESIDUAL:
            pre, mag = pre + extra.double(), mag + extra.double().abs()
        _check(y, pre, mag, dtype, f"{N} rows")


# 16 bit, at most a workgroup a compute unit and a reduction of 768 and more: whole blocks of 64, a ragged last one, rows past a tile
@pytest.mark.parametrize("N,K,P", [(2048, 768, 768), (2113, 784, 768), (768, 1552, 1536), (7889, 1536, 384)])
@pytest.mark.parametrize("dtype,out", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16), (torch.float16, torch.float32)])
def test_dense_forward_of_long_reductions(N, K, P, dtype, out):
    test_dense_forward_and_input_gradient(N, K, P, dtype, out)
    test_dense_forward_and_input_gradient(N, P, K, dtype, out)


# fp32, fewer than 96 reduction channels: 64 columns a workgroup, or 96 where those cover the layer with fewer (272, 288; not with a second operand);
# parts of a tile, whole ones and one piece more; half steps of the reduction
@pytest.mark.parametrize("N,K", [(19201, 48), (19230, 80), (19313, 16)])
@pytest.mark.parametrize("P", [16, 48, 64, 80, 96, 112, 128, 144, 192, 272, 288, 304])
def test_dense_fp32_forward_of_short_reductions(N, K, P):
    test_dense_forward_and_input_gradient(N, K, P, torch.float32, torch.float32)


# a result in the place of its rows, where one workgroup of a tile holds them whole (96 columns at most, more rows than the few-rows kernel takes)
@pytest.mark.parametrize("K", [48, 96])
def test_dense_forward_in_place(K):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    N, dtype = 140001, torch.float16
    gen = torch.Generator().manual_seed(K)
    x, w, b = _rand(gen, N, K, dtype=dtype), (_rand(gen, K, K, spread=1) / K ** 0.5).to(dtype), _rand(gen, K, dtype=dtype)
    ref, mag = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs()
    _lib.check(lib.sswin_dense_forward(1, 1, 0, PLAIN, _ptr(x), N, K, _ptr(w), _ptr(b), K, None, _ptr(x), None, None, 0, _stream()))
    _check(x, ref, mag, dtype, "in place")


# fp32 in place with values that are not finite, whose results are formed again from rows that lie where results go; 32 and 96 columns a
# workgroup where the rows lie apart, a ragged last tile.  Up to 48 channels, 96, and with a workspace for pieces that in place has no use for
@pytest.mark.parametrize("N,K", [(19201, 96), (30001, 96), (140001, 48)])
@pytest.mark.parametrize("epi", [PLAIN, RESIDUAL])
@pytest.mark.parametrize("where", ["finite", "weight", "rows"])
def test_dense_fp32_forward_in_place(N, K, epi, where):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    for transposed in (0, 1):
        if transposed and epi == RESIDUAL:
            continue
        gen = torch.Generator().manual_seed(N + K)
        x, w, extra = torch.randn(N, K, generator=gen), torch.randn(K, K, generator=gen), torch.randn(N, K, generator=gen).cuda()
        if where == "weight":
            w[(K - 8, 40) if transposed else (40, K - 8)] = float("inf")
        elif where == "rows":
            x[N // 2, 40], x[N - 1, 3] = float("inf"), float("nan")
        x, w = x.cuda(), w.cuda()
        wd = w.double() if transposed else w.double().T
        ref, scale = x.double() @ wd, x.double().abs() @ wd.abs()
        if epi == RESIDUAL:
            ref, scale = ref + extra.double(), scale + extra.double().abs()
        ws = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
        _lib.check(lib.sswin_dense_forward(0, 0, transposed, epi, _ptr(x), N, K, _ptr(w), None, K, _ptr(extra) if epi == RESIDUAL else None, _ptr(x), None,
                                           _ptr(ws), ws.numel(), _stream()))
        _same_class(x, ref, scale, f"transposed {transposed}")
        assert ref.isfinite().all() == (where == "finite")


# 16 bit: the last rows of the few-rows kernel and the first of the tiles behind it, with a residual and as an input gradient
@pytest.mark.parametrize("N", [5376, 5377])
def test_dense_forward_where_the_tiles_take_over(N):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    K, P, dtype = 288, 144, torch.bfloat16                               # 42 row tiles x 2 x 288 = 24 192, 43: 24 768; the line: 26 400
    gen = torch.Generator().manual_seed(N)
    for n in (N, N + 384, N + 512):                                      # 45 row tiles: 25 920, 46: 26 496
        x, w, b, extra = _rand(gen, n, K, dtype=dtype), (_rand(gen, P, K, spread=1) / K ** 0.5).to(dtype), _rand(gen, P, dtype=dtype), _rand(gen, n, P, dtype=dtype)
        pre, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        y, _ = _forward(lib, _lib, x, w, b, 0, RESIDUAL, extra, dtype)
        _check(y, pre + b.double() + extra.double(), mag + b.double().abs() + extra.double().abs(), dtype, "residual")
        dx, _ = _forward(lib, _lib, x, w.T.contiguous(), None, 1, PLAIN, None, dtype)
        _check(dx, pre, mag, dtype, "input gradient")


@pytest.mark.parametrize("N,P,K", [(1, 16, 16), (17, 144, 48), (1024, 96, 96), (1025, 48, 208), (1100, 288, 96), (9001, 208, 192), (70001, 48, 144),
                                   (2000, 16, 16), (30001, 64, 48), (40001, 144, 48), (1100, 400, 64), (3003, 64, 400), (4501, 2304, 768)])
@pytest.mark.parametrize("dtype,out", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)],
                         ids=["fp32", "bf16", "fp16-out32"])
def test_dense_weight_gradient(N, P, K, dtype, out):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(N + P + K)
    dy, x = _rand(gen, N, P, dtype=dtype), _rand(gen, N, K, dtype=dtype)
    results = []
    for _ in range(2):
        dw, db = (torch.full(s, float("nan"), dtype=out, device="cuda") for s in ((P, K), (P,)))
        nb = lib.sswin_dense_weight_grad_workspace_bytes(CODE[dtype], N, P, K)
        ws = torch.empty(max(nb, 1), dtype=torch.uint8, device="cuda")
        _lib.check(lib.sswin_dense_weight_grad(CODE[dtype], CODE[out], _ptr(dy), _ptr(x), N, P, K, _ptr(dw), _ptr(db), _ptr(ws), nb, _stream()))
        results.append((dw, db))
    _check(results[0][0], dy.double().T @ x.double(), dy.double().abs().T @ x.double().abs(), out, "dW")
    _check(results[0][1], dy.double().sum(0), dy.double().abs().sum(0), out, "db")
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])       # fixed order of the sums


@pytest.mark.parametrize("N", [1025, 1033, 1057, 4111])
@pytest.mark.parametrize("P,K", [(96, 384), (112, 192), (128, 208), (400, 192), (64, 192), (192, 64), (80, 48), (64, 64), (16, 16), (144, 144), (48, 80)])
def test_fp32_weight_gradient_at_the_edges_of_its_tiles(N, P, K):
    """Every tile of dW, with columns that end inside one and rows that end inside the row groups of a step."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(N + P + K)
    dy, x = _rand(gen, N, P), _rand(gen, N, K)
    dw, db = (torch.full(s, float("nan"), device="cuda") for s in ((P, K), (P,)))
    nb = lib.sswin_dense_weight_grad_workspace_bytes(0, N, P, K)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    _lib.check(lib.sswin_dense_weight_grad(0, 0, _ptr(dy), _ptr(x), N, P, K, _ptr(dw), _ptr(db), _ptr(ws), nb, _stream()))
    _check(dw, dy.double().T @ x.double(), dy.double().abs().T @ x.double().abs(), torch.float32, "dW")
    _check(db, dy.double().sum(0), dy.double().abs().sum(0), torch.float32, "db")


@pytest.mark.parametrize("sizes", [(8,), (96 * 288, 288, 96 * 96, 96, 8, 16, 2056, 24)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_cast_parts(sizes, dtype):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(len(sizes))
    src = [_rand(gen, n) for n in sizes]
    dst = torch.full((sum(sizes),), float("nan"), dtype=dtype, device="cuda")
    _lib.check(lib.sswin_cast_parts(CODE[dtype], (C.c_void_p * len(src))(*[t.data_ptr() for t in src]), (C.c_int64 * len(src))(*sizes), len(src), _ptr(dst),
                                    _stream()))
    assert torch.equal(dst, torch.cat(src).to(dtype))
    assert lib.sswin_cast_parts(CODE[dtype], (C.c_void_p * 1)(src[0].data_ptr()), (C.c_int64 * 1)(4), 1, _ptr(dst), _stream()) != 0


def test_dense_refuses_what_it_does_not_take():
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    x = torch.zeros(4, 24, device="cuda")
    assert not lib.sswin_dense_supported(0, 16, 24) and lib.sswin_dense_supported(2, 16, 32) and not lib.sswin_dense_supported(3, 16, 16)
    assert lib.sswin_dense_forward(0, 0, 0, PLAIN, _ptr(x), 4, 24, _ptr(x), None, 16, None, _ptr(x), None, None, 0, _stream()) != 0
    assert b"multiples of 16" in lib.sswin_last_error()
    assert lib.sswin_dense_forward(0, 0, 0, SCALE, _ptr(x), 4, 16, _ptr(x), None, 16, _ptr(x), _ptr(x), None, None, 0, _stream()) != 0
    assert lib.sswin_dense_forward(0, 0, 0, RESIDUAL, _ptr(x), 4, 16, _ptr(x), None, 16, None, _ptr(x), None, None, 0, _stream()) != 0
    assert lib.sswin_dense_forward(0, 0, 0, PLAIN, None, 0, 16, None, None, 16, None, None, None, None, 0, _stream()) == 0


@pytest.mark.parametrize("N,D", [(1, 16), (7, 48), (1000, 96), (33, 192), (257, 768), (5, 80), (63, 1536), (4, 2048), (50000, 96)])
@pytest.mark.parametrize("dtype,out", [(torch.float32, torch.float32), (torch.float32, torch.float16), (torch.bfloat16, torch.bfloat16)],
                         ids=["fp32", "fp32-fp16", "bf16"])
def test_layer_norm(N, D, dtype, out):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    assert lib.sswin_layer_norm_supported(CODE[dtype], D)
    gen = torch.Generator().manual_seed(N + D)
    x, dy, dres = _rand(gen, N, D, dtype=dtype), _rand(gen, N, D, dtype=out), _rand(gen, N, D, dtype=dtype)
    g, b = _rand(gen, D, dtype=dtype, spread=1), _rand(gen, D, dtype=dtype, spread=1)
    y, stats = torch.full((N, D), float("nan"), dtype=out, device="cuda"), torch.empty(2, N, device="cuda")
    _lib.check(lib.sswin_layer_norm_forward(CODE[dtype], CODE[out], _ptr(x), N, D, _ptr(g), _ptr(b), 1e-5, _ptr(y), _ptr(stats), _stream()))
    xd, gd, dyd = x.double(), g.double(), dy.double()
    mean, var = xd.mean(1, keepdim=True), xd.var(1, unbiased=False, keepdim=True)
    rstd = (var + 1e-5).rsqrt()
    xh = (xd - mean) * rstd
    # the mean of a row carries an error of its magnitude times the sum's rounding, which the norm scales by 1 / deviation
    slack = 1 + xd.abs().amax(1, keepdim=True) * rstd
    _check(y, xh * gd + b.double(), gd.abs() * slack + b.double().abs(), out, "norm")
    nb = lib.sswin_layer_norm_backward_workspace_bytes(CODE[dtype], N, D)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    dx, dg, db = (torch.full(s, float("nan"), dtype=dtype, device="cuda") for s in ((N, D), (D,), (D,)))
    _lib.check(lib.sswin_layer_norm_backward(CODE[dtype], CODE[out], _ptr(dy), _ptr(x), _ptr(stats), N, D, _ptr(g), _ptr(dres), _ptr(dx), _ptr(dg),
                                             _ptr(db), _ptr(ws), nb, _stream()))
    gy = dyd * gd
    ref = rstd * (gy - gy.mean(1, keepdim=True) - xh * (gy * xh).mean(1, keepdim=True)) + dres.double()
    _check(dx, ref, rstd * (gy.abs() + gy.abs().mean(1, keepdim=True) * (1 + xh.abs() * xh.abs().amax(1, keepdim=True))) * slack + dres.double().abs(), dtype,
           "dx")
    _check(dg, (dyd * xh).sum(0), (dyd.abs() * (xh.abs() + slack)).sum(0), dtype, "d gain")
    _check(db, dyd.sum(0), dyd.abs().sum(0), dtype, "d offset")


def _stage_pieces(dim, heads, window, dtype, merge, seed, grid=(21, 18, 11), n=3000, qkv_bias=True):
    import numpy as np
    from sparseswin3d_amd.layers import BasicLayer, PoolDownsample
    from sparseswin3d_amd.window_attention import SparseVoxelTensor
    rng = np.random.default_rng(seed)
    cells = rng.choice(int(np.prod(grid)), size=n, replace=False)
    c4 = np.stack([np.zeros_like(cells), *np.unravel_index(cells, grid)], 1).astype(np.int32)
    torch.manual_seed(seed)
    layer = BasicLayer(dim, 2, heads, (window,) * 3, 0.0, qkv_bias=qkv_bias, downsample=PoolDownsample if merge else None)
    with torch.no_grad():
        for p in layer.parameters():
            p.add_(0.05 * torch.randn_like(p))
    layer = layer.cuda().to(dtype)
    feats = torch.randn(n, dim).cuda().to(dtype)
    return layer, lambda x: layer(SparseVoxelTensor(x, torch.from_numpy(c4).cuda(), grid, 1)).features, feats


@pytest.mark.parametrize("dim,heads,window,merge,qkv_bias", [(96, 3, 5, True, True), (48, 3, 7, False, True), (192, 6, 5, True, False), (80, 5, 5, False, True)])
@pytest.mark.parametrize("mode", ["fp32", "bf16", "amp"])
def test_stage_as_single_nodes_equals_its_composition(dim, heads, window, merge, qkv_bias, mode, monkeypatch):
    """BasicLayer with each block (and the merge) as one autograd node against the same layer composed of its modules, all
    gradients included.  fp32: both chains carry fp32 rounding only (2e-5 of the norm of a result); 16-bit: the composition
    rounds every intermediate to 16 bits, one node fewer of them, so the two differ by roundings of the type."""
    from sparseswin3d_amd import layers
    dtype = torch.bfloat16 if mode == "bf16" else torch.float32
    layer, run, feats = _stage_pieces(dim, heads, window, dtype, merge, dim + window, qkv_bias=qkv_bias)
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
        assert (("MergeNode" if merge else "BlockNode") in y.grad_fn.name()) == single, y.grad_fn.name()
        y.backward(up)
        results.append([("out", y.detach()), ("dx", x.grad)] + [(k, p.grad) for k, p in layer.named_parameters()])
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, enabled=mode == "amp"):
            # inference differs from the training forward in what it keeps, and where nothing rounds in between not in its result
            assert torch.equal(run(feats), y.detach()), "inference"
    tol = {"fp32": 2e-5, "bf16": 4e-2, "amp": 8e-3}[mode]
    for (k, a), (_, b) in zip(*results):
        assert a.dtype == b.dtype and a.shape == b.shape, k
        rel = ((a.double() - b.double()).norm() / b.double().norm()).item()
        assert rel < tol, (k, rel)


def test_blocks_with_dropout_or_hooks_run_their_modules():
    layer, run, feats = _stage_pieces(96, 3, 5, torch.float32, False, 5)
    calls = []
    handle = layer.blocks[0].norm2.register_forward_hook(lambda *a: calls.append(1))
    a = run(feats)
    assert calls == [1]
    handle.remove()
    b = run(feats)
    assert calls == [1] and torch.allclose(a, b, rtol=1e-4, atol=1e-5)
    layer.blocks[1].mlp.drop1.p = 0.5
    layer.train()
    torch.manual_seed(0)
    c = run(feats)
    assert not torch.allclose(b, c, rtol=1e-3, atol=1e-3)
    layer.eval()
    assert torch.allclose(run(feats), b, rtol=1e-4, atol=1e-5)


def test_modules_refuse_what_their_layers_do_not_fit():
    """Host checks of the compiled path: rows of another width, a plan of other voxels, forward-mode tangents."""
    import numpy as np
    from helpers import random_window_indices
    from sparseswin3d_amd.window_attention import SparseVoxelTensor, WindowAttentionSparse
    torch.manual_seed(0)
    attn = WindowAttentionSparse(96, 3, (5, 5, 5), qkv_bias=True).cuda()
    ind = torch.from_numpy(random_window_indices(np.random.default_rng(0), 40, 125, 700)).cuda()
    run = lambda f, i=ind: attn(SparseVoxelTensor(f, i, (125,), 40), None).features
    x = torch.randn(700, 96, device="cuda")
    for grad in (True, False):
        with torch.set_grad_enabled(grad):
            with pytest.raises(RuntimeError):
                run(torch.randn(700, 48, device="cuda"))
            with pytest.raises(RuntimeError):
                run(x[:600].contiguous())
            with torch.autograd.forward_ad.dual_level():
                with pytest.raises(RuntimeError, match="jvp"):
                    run(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
    layer, stage, feats = _stage_pieces(96, 3, 5, torch.float32, True, 7)
    with torch.no_grad(), torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError, match="jvp"):
        stage(torch.autograd.forward_ad.make_dual(feats, torch.ones_like(feats)))
    with pytest.raises(RuntimeError):
        stage(feats[:, :48].contiguous())


def test_projections_that_are_no_plain_linears_run_under_autocast():
    """Under autocast the projections are called as modules: a wrapper or a hook takes part."""
    import numpy as np
    from helpers import random_window_indices
    from sparseswin3d_amd.window_attention import SparseVoxelTensor, WindowAttentionSparse

    class Scaled(torch.nn.Linear):
        def forward(self, x):
            return 0 * super().forward(x)

    torch.manual_seed(0)
    attn = WindowAttentionSparse(96, 3, (5, 5, 5), qkv_bias=True).cuda()
    ind = torch.from_numpy(random_window_indices(np.random.default_rng(0), 40, 125, 700)).cuda()
    x = torch.randn(700, 96, device="cuda")
    with torch.autocast("cuda", dtype=torch.float16):
        plain = attn(SparseVoxelTensor(x, ind, (125,), 40), None).features
        calls = []
        handle = attn.qkv.register_forward_hook(lambda *a: calls.append(1))
        hooked = attn(SparseVoxelTensor(x, ind, (125,), 40), None).features
        handle.remove()
        assert calls == [1] and torch.allclose(plain, hooked, rtol=2e-2, atol=2e-2)
        attn.proj = Scaled(96, 96).cuda()
        assert not attn(SparseVoxelTensor(x, ind, (125,), 40), None).features.any()


@pytest.mark.parametrize("N,P,K", [(1, 16, 16), (33, 96, 384), (284, 208, 80), (500, 1536, 384), (1024, 48, 144)])
@pytest.mark.parametrize("dtype,out", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)],
                         ids=["fp32", "bf16", "fp16-out32"])
@pytest.mark.parametrize("factor", [False, True], ids=["plain", "factor"])
def test_dense_backward_of_few_rows_in_one_launch(N, P, K, dtype, out, factor):
    """Both gradients from one launch against the two launches: the same tiles, so the same bits."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    assert lib.sswin_dense_backward_small_supported(CODE[dtype], N, P, K) and not lib.sswin_dense_backward_small_supported(CODE[dtype], 1025, P, K)
    gen = torch.Generator().manual_seed(N + P + K)
    dy, x, w = _rand(gen, N, P, dtype=dtype), _rand(gen, N, K, dtype=dtype), _rand(gen, P, K, dtype=dtype)
    f = _rand(gen, N, K, dtype=dtype) if factor else None
    epi = SCALE if factor else PLAIN
    dx, dw, db = (torch.full(s, float("nan"), dtype=t, device="cuda") for s, t in (((N, K), dtype), ((P, K), out), ((P,), out)))
    _lib.check(lib.sswin_dense_backward_small(CODE[dtype], CODE[out], epi, _ptr(dy), _ptr(x), _ptr(w), N, P, K, _ptr(f), _ptr(dx), _ptr(dw), _ptr(db),
                                              _stream()))
    assert torch.equal(dx, _forward(lib, _lib, dy, w, None, 1, epi, f, dtype)[0])
    dw2, db2 = torch.empty_like(dw), torch.empty_like(db)
    nb = lib.sswin_dense_weight_grad_workspace_bytes(CODE[dtype], N, P, K)
    ws = torch.empty(max(nb, 1), dtype=torch.uint8, device="cuda")
    _lib.check(lib.sswin_dense_weight_grad(CODE[dtype], CODE[out], _ptr(dy), _ptr(x), N, P, K, _ptr(dw2), _ptr(db2), _ptr(ws), nb, _stream()))
    assert torch.equal(dw, dw2) and torch.equal(db, db2)
    dw.fill_(float("nan"))
    _lib.check(lib.sswin_dense_backward_small(CODE[dtype], CODE[out], epi, _ptr(dy), _ptr(x), _ptr(w), N, P, K, _ptr(f), _ptr(dx), _ptr(dw), None, _stream()))
    assert torch.equal(dw, dw2)


@pytest.mark.parametrize("N,D", [(1, 16), (33, 192), (5, 80), (5000, 96)])
@pytest.mark.parametrize("kind", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
def test_layer_norm_backward_with_a_16_bit_copy(N, D, kind):
    """dx in dy's type beside fp32 dx: the rounding of the same values, and nothing else changes."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(N + D)
    x, dres, g, dy = _rand(gen, N, D), _rand(gen, N, D), _rand(gen, D, spread=1), _rand(gen, N, D, dtype=kind)
    stats = torch.stack([x.mean(1), (x.var(1, unbiased=False) + 1e-5).rsqrt()]).contiguous()
    nb = lib.sswin_layer_norm_backward_workspace_bytes(0, N, D)
    results = []
    for with_copy in (True, False):
        ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
        dx, dg, db = (torch.full(s, float("nan"), device="cuda") for s in ((N, D), (D,), (D,)))
        copy = torch.full((N, D), float("nan"), dtype=kind, device="cuda") if with_copy else None
        _lib.check(lib.sswin_layer_norm_backward_copy(0, CODE[kind], _ptr(dy), _ptr(x), _ptr(stats), N, D, _ptr(g), _ptr(dres), _ptr(dx), _ptr(copy), _ptr(dg),
                                                      _ptr(db), _ptr(ws), nb, _stream()))
        results.append((dx, dg, db))
        if with_copy:
            assert torch.equal(copy, dx.to(kind))
    assert all(torch.equal(a, b) for a, b in zip(*results))


# the tiled kernel (half a step of the reduction and whole ones), the few-rows one; weight gradients: few rows and each tile shape
EXACT_ROWS = [(20000, 48, 96), (20000, 16, 112), (300, 384, 208), (33, 96, 96), (20001, 144, 48)]
EXACT_WGRAD = [(900, 144, 48), (9001, 208, 192), (20001, 48, 208), (30001, 64, 48), (40001, 144, 48), (9000, 208, 96)]


def _same_class(got, ref, scale, what):
    """Finite where float64 is (to the bound of the file), the same infinities, NaN where float64 has NaN."""
    got = got.double()
    finite = ref.isfinite()
    assert got[finite].isfinite().all(), what
    assert ((got - ref)[finite].abs() <= 1e-6 * scale[finite] + 1e-30).all(), what
    assert torch.equal(got[ref.isinf()], ref[ref.isinf()]), what
    assert got[ref.isnan()].isnan().all(), what


@pytest.mark.parametrize("N,K,P", EXACT_ROWS)
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4028234e38])
@pytest.mark.parametrize("where", ["rows", "weight"])
def test_dense_fp32_of_values_that_are_not_finite(N, K, P, value, where):
    """An infinity, a NaN or the largest number in a few places: the results that depend on them are those of plain fp32
    arithmetic.  (Rows or columns of the largest number are scaled down, so that the result is in range.)"""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(N + K)
    for transposed in (0, 1):
        rows, cols = (P, K) if transposed else (K, P)             # of the reduction and the result
        x, w = torch.randn(N, rows, generator=gen), torch.randn(P, K, generator=gen)
        if abs(value) < float("inf"):
            x, w = x * 2.0 ** -10, w * 2.0 ** -10
        for r, c in ((0, 1), (N // 2, rows - 1), (N - 1, 0)):
            if where == "rows":
                x[r, c] = value
            elif transposed:
                w[c, r % K] = value
            else:
                w[r % P, c] = value
        x[N // 3] = 0                                              # 0 x inf
        x, w = x.cuda(), w.cuda()
        y, _ = _forward(lib, _lib, x, w, None, transposed, PLAIN, None, torch.float32)
        wd = w.double() if transposed else w.double().T
        ref, scale = x.double() @ wd, x.double().abs() @ wd.abs()
        _same_class(y, ref, scale, f"transposed {transposed}")
        assert (abs(value) < float("inf")) == bool(ref.isfinite().all())


@pytest.mark.parametrize("N,P,K", EXACT_WGRAD)
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4028234e38])
@pytest.mark.parametrize("where", ["dy", "x"])
def test_dense_fp32_weight_gradient_of_values_that_are_not_finite(N, P, K, value, where):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(N + K)
    dy, x = torch.randn(N, P, generator=gen), torch.randn(N, K, generator=gen)
    if abs(value) < float("inf"):
        dy, x = dy * 2.0 ** -12, x * 2.0 ** -12
    t = dy if where == "dy" else x
    for r, c in ((0, 1), (N // 2, t.shape[1] - 1), (N - 1, 7)):
        t[r, c] = value
        (x if where == "dy" else dy)[r, :5] = 0
    dy, x = dy.cuda(), x.cuda()
    dw, db = torch.empty(P, K, device="cuda"), torch.empty(P, device="cuda")
    nb = lib.sswin_dense_weight_grad_workspace_bytes(0, N, P, K)
    ws = torch.empty(max(nb, 1), dtype=torch.uint8, device="cuda")
    _lib.check(lib.sswin_dense_weight_grad(0, 0, _ptr(dy), _ptr(x), N, P, K, _ptr(dw), _ptr(db), _ptr(ws), nb, _stream()))
    d, v = dy.double(), x.double()
    _same_class(dw, d.T @ v, d.abs().T @ v.abs(), "dW")
    _same_class(db, d.sum(0), d.abs().sum(0), "db")


# fp32 layers of at least 96 reduction channels (pairs of fp16): whole steps of 32 and a last one of 16, columns that end inside a tile, several
# column blocks; one row past a workgroup's
PAIRS = [(19201, 96, 112), (20001, 144, 48), (20001, 208, 304), (9601, 576, 192)]
# 96 channels (turned: 96 columns) and a multiple of 96 outputs: 32 or 96 columns a workgroup, one and several tiles of rows a wavefront
PAIRS += [(6401, 96, 288), (13825, 96, 288), (19233, 96, 96), (90001, 96, 96), (30001, 288, 96)]


@pytest.mark.parametrize("N,K,P", PAIRS)
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4028234e38])
def test_dense_fp32_pairs_of_values_that_are_not_finite(N, K, P, value):
    for where in ("rows", "weight"):
        test_dense_fp32_of_values_that_are_not_finite(N, K, P, value, where)


@pytest.mark.parametrize("span", [20, -20])
@pytest.mark.parametrize("N,K,P", PAIRS)
def test_dense_fp32_pairs_scales(N, K, P, span):
    """The pieces are scaled by row and by column: rows and columns of any size, values that grow or fall by 2^20 along the reduction and
    meet weights that do the opposite, so that each product counts the same; rows that begin with zeros.  Bound: the file's."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(K + P)
    two = lambda lo, hi, *s: torch.exp2(torch.randint(lo, hi + 1, s, generator=gen).float())
    for transposed in (0, 1):
        rows, cols = (P, K) if transposed else (K, P)             # of the reduction and the result
        ramp = torch.exp2(torch.linspace(-span / 2, span / 2, rows).round())
        x, wt = torch.randn(N, rows, generator=gen) * ramp * two(-40, 40, N, 1), torch.randn(cols, rows, generator=gen) / ramp * two(-40, 40, cols, 1)
        x[N // 2, :rows - 8] = 0
        x[N // 3] = 0
        x, w = x.cuda(), (wt.T.contiguous() if transposed else wt).cuda()
        y, _ = _forward(lib, _lib, x, w, None, transposed, PLAIN, None, torch.float32)
        wd = wt.double().cuda()
        _check(y, x.double() @ wd.T, x.double().abs() @ wd.abs().T, torch.float32, f"transposed {transposed}")


@pytest.mark.parametrize("span", [40, -40, 70])
@pytest.mark.parametrize("N,K,P", PAIRS)
def test_dense_fp32_pairs_scales_that_the_pieces_do_not_span(N, K, P, span):
    """Every result is small against what its row and column hold: all of them formed again."""
    test_dense_fp32_pairs_scales(N, K, P, span)


@pytest.mark.parametrize("power", [30, 36, 48])
@pytest.mark.parametrize("N,K,P", PAIRS)
def test_dense_fp32_pairs_of_a_channel_above_the_rest(N, K, P, power):
    """A channel 2^power above the others of its rows that meets zeros in some columns, whose results are those of the other channels: few
    results of a tile (the rows of a tile but one, one column), many (a block of rows that all have it); a row and a column of zeros."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(K + P + power)
    for transposed in (0, 1):
        rows, cols = (P, K) if transposed else (K, P)             # of the reduction and the result
        x, wt = torch.randn(N, rows, generator=gen), torch.randn(cols, rows, generator=gen)
        c = rows - 5
        x[7, c] = x[N // 2, c] = x[N - 1, c] = 2.0 ** power
        x[64:128, c] = -2.0 ** power
        x[9], wt[5] = 0, 0
        wt[3, c] = wt[cols - 1, c] = 0
        wt[cols // 2] *= 2.0 ** -power                            # one large weight in a column, met by zeros
        wt[cols // 2, 1] = 1
        x[N // 3:N // 3 + 3, 1] = 0
        x, w = x.cuda(), (wt.T.contiguous() if transposed else wt).cuda()
        wd = wt.double().cuda()
        for extra in (None, torch.zeros(N, cols, device="cuda") if transposed == 0 else torch.ones(N, cols, device="cuda")):
            y, _ = _forward(lib, _lib, x, w, None, transposed, PLAIN if extra is None else SCALE if transposed else RESIDUAL, extra, torch.float32)
            _check(y, x.double() @ wd.T, x.double().abs() @ wd.abs().T, torch.float32, f"transposed {transposed}")


@pytest.mark.parametrize("N,K,P", [(20001, 208, 304), (30001, 288, 96), (30001, 96, 288)])
def test_dense_fp32_pairs_rows_that_begin_with_zeros(N, K, P):
    """A row's results have the same bits whatever stands in the rows beside it: zeros at the beginning of every row or of some."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(K)
    x, w = torch.randn(N, K, generator=gen, device="cuda"), torch.randn(P, K, generator=gen, device="cuda")
    some, every = x.clone(), x
    some[::3, :K // 2] = 0
    every[:, :K // 2] = 0
    a, b = (_forward(lib, _lib, t, w, None, 0, PLAIN, None, torch.float32)[0] for t in (some, every))
    assert torch.equal(a[::3], b[::3])


# the last steps of 96 channels, on either side of the rows from which a workgroup takes 96 columns
@pytest.mark.parametrize("N,K,P", [(6400, 96, 288), (13633, 96, 288), (21761, 288, 96), (41217, 96, 96)])
def test_dense_fp32_pairs_of_96_channels(N, K, P):
    test_dense_forward_and_input_gradient(N, K, P, torch.float32, torch.float32)


# 2-norm of the error over that of the result, a twentieth above what was measured (three bf16 pieces: 2.0, 1.75, 2.5 and 6.0e-7)
@pytest.mark.parametrize("N,K,P,transposed,error", [(35569, 192, 192, 0, 1.27e-7), (20000, 48, 144, 1, 1.17e-7), (19201, 96, 288, 1, 1.43e-7), (9000, 384, 1536, 1, 2.75e-7)])
def test_dense_fp32_pairs_rounding(N, K, P, transposed, error):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(N + K)
    rows = P if transposed else K
    x, w = torch.randn(N, rows, generator=gen, device="cuda"), torch.randn(P, K, generator=gen, device="cuda") * rows ** -0.5
    y, _ = _forward(lib, _lib, x, w, None, transposed, PLAIN, None, torch.float32)
    ref = x.double() @ (w.double() if transposed else w.double().T)
    assert (y.double() - ref).norm() <= error * ref.norm()


def test_dense_fp32_without_a_workspace():
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(5)
    N, K, P = 20001, 208, 144
    x, w, y = _rand(gen, N, K), _rand(gen, P, K, spread=1), torch.full((N, P), float("nan"), device="cuda")
    assert lib.sswin_dense_forward_workspace_bytes(0, N, K, P) > 0
    _lib.check(lib.sswin_dense_forward(0, 0, 0, PLAIN, _ptr(x), N, K, _ptr(w), None, P, None, _ptr(y), None, None, 0, _stream()))
    _check(y, x.double() @ w.double().T, x.double().abs() @ w.double().abs().T, torch.float32, "plain")


# a null workspace with a size beside it: fp32 with pieces of W, 16 bit with shares of the reduction
@pytest.mark.parametrize("N,K,P,dtype", [(20001, 208, 144, torch.float32), (1364, 3072, 768, torch.bfloat16)])
def test_dense_null_workspace_with_a_size(N, K, P, dtype):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(5)
    x, w, y = _rand(gen, N, K, dtype=dtype), (_rand(gen, P, K, spread=1) / K ** 0.5).to(dtype), torch.full((N, P), float("nan"), dtype=dtype, device="cuda")
    nb = lib.sswin_dense_forward_workspace_bytes(CODE[dtype], N, K, P)
    assert nb > 0
    _lib.check(lib.sswin_dense_forward(CODE[dtype], CODE[dtype], 0, PLAIN, _ptr(x), N, K, _ptr(w), None, P, None, _ptr(y), None, None, nb, _stream()))
    _check(y, x.double() @ w.double().T, x.double().abs() @ w.double().abs().T, dtype, "plain")


# each tile shape where its sums are shortest or longest for their number; relative error of dW against float64 (2-norms).  The
# bounds are a twentieth above what tiles of 96 x 96 (64 x 64 up to 64 columns) with sums of at least 64 rows give there, averaged over
# as many inputs.
ROUNDING = [(14000, 80, 80, 1.78e-7), (30000, 48, 48, 2.12e-7), (20000, 144, 48, 1.90e-7), (30000, 144, 48, 2.13e-7), (112700, 144, 144, 5.08e-7),
            (112700, 96, 144, 3.85e-7), (14000, 240, 112, 1.90e-7)]


@pytest.mark.parametrize("N,P,K,error", ROUNDING)
def test_dense_fp32_weight_gradient_rounding(N, P, K, error):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    errors = []
    for seed in range(3):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        dy, x = torch.randn(N, P, generator=gen, device="cuda"), torch.randn(N, K, generator=gen, device="cuda")
        dw = torch.empty(P, K, device="cuda")
        nb = lib.sswin_dense_weight_grad_workspace_bytes(0, N, P, K)
        ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
        _lib.check(lib.sswin_dense_weight_grad(0, 0, _ptr(dy), _ptr(x), N, P, K, _ptr(dw), None, _ptr(ws), nb, _stream()))
        ref = dy.double().T @ x.double()
        errors.append(((dw.double() - ref).norm() / ref.norm()).item())
    assert sum(errors) / 3 <= 1.05 * error, [f"{e:.3e}" for e in errors]


# fp32 results of 16-bit rows: 2-norm of the error over that of the result, as the kernel for few rows has it (5.4, 5.5, 4.85 and 5.4e-8, three
# inputs within 1 %); the tiles give 6.0, 6.5 and 5.2e-8 for the first three, and 5.4e-8 for the last, where they are taken
@pytest.mark.parametrize("N,K,P,error", [(7296, 288, 288, 5.6e-8), (4096, 384, 384, 5.65e-8), (65920, 96, 96, 5.0e-8), (16384, 192, 192, 5.55e-8)])
def test_dense_fp32_results_of_16_bit_rows_rounding(N, K, P, error):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(N + K)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    x, w, b, extra = rand(N, K).half(), (rand(P, K) * K ** -0.5).half(), rand(P).half(), rand(N, P)
    y, _ = _forward(lib, _lib, x, w, b, 0, RESIDUAL, extra, torch.float32)
    ref = x.double() @ w.double().T + b.double() + extra.double()
    assert (y.double() - ref).norm() <= error * ref.norm()


@pytest.mark.parametrize("kind", ["rows", "few rows", "weight gradient", "weight gradient, few rows"])
def test_dense_fp32_keeps_the_bits_of_single_products(kind):
    """16 equal products of operands whose lower pieces are as large as they get (just below 1 + 2^-7; just below and above a
    half-way point of the pieces).  What the piece products leave out is at most 2^-23 of each product; adding up the kept ones rounds
    the result a few times more (the last additions: 2^-24 each): 2^-22 in all."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    ones = [1 + 2.0 ** -7 - 2.0 ** -15 - 2.0 ** -23, 1 + 2.0 ** -7 - 2.0 ** -23, 1 + 2.0 ** -8 + 2.0 ** -16 + 2.0 ** -23, 1 + 2.0 ** -8 + 2.0 ** -17,
            1.9999999, 1 + 2.0 ** -8 - 2.0 ** -17 - 2.0 ** -23]
    worst = 0.0
    for a in ones:
        for b in ones:
            for sign in (1.0, -1.0):
                ta, tb = torch.tensor(a, dtype=torch.float32), torch.tensor(b, dtype=torch.float32) * sign
                exact = 16 * ta.double().item() * tb.double().item()
                if kind in ("rows", "few rows"):
                    x, w = ta.expand(20000 if kind == "rows" else 64, 16).contiguous().cuda(), tb.expand(112, 16).contiguous().cuda()
                    y, _ = _forward(lib, _lib, x, w, None, 0, PLAIN, None, torch.float32)
                else:
                    N = 2000 if kind == "weight gradient" else 40
                    d, v = torch.zeros(N, 112), torch.zeros(N, 208)
                    d[8:24], v[8:24] = ta, tb
                    d, v, y = d.cuda(), v.cuda(), torch.empty(112, 208, device="cuda")
                    nb = lib.sswin_dense_weight_grad_workspace_bytes(0, N, 112, 208)
                    ws = torch.empty(max(nb, 1), dtype=torch.uint8, device="cuda")
                    _lib.check(lib.sswin_dense_weight_grad(0, 0, _ptr(d), _ptr(v), N, 112, 208, _ptr(y), None, _ptr(ws), nb, _stream()))
                err = (y.double() - exact).abs().max().item() / abs(exact)
                worst = max(worst, err)
                assert err <= 2.0 ** -22, (a, b, sign, err * 2 ** 24)
    print(f"{kind}: worst error {worst * 2 ** 24:.2f} x 2^-24")
