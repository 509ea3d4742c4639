"""GPU parity of the feed-forward part as one launch (``sswin_mlp_*``) against float64 arithmetic on the same inputs, and against
the two layers it stands for.

Bounds: a hidden value carries the error of its product (2e-6 of the sum of the absolute products, two chains of an fp32 GEMM) and of
GELU (4e-7 of the value's own size, 1e-6 near 0), rounded to the layers' type; the second layer adds its own, and passes on that of the
hidden values through the absolute weights."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
ROUND = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _ptr(t):
    return C.c_void_p(t.data_ptr() if t is not None else None)


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _empty(shape, dtype):
    return torch.full(shape, float("nan"), dtype=dtype, device="cuda")


def _workspace(lib, x, hidden, backward):
    nb = lib.sswin_mlp_workspace_bytes(CODE[x.dtype], x.shape[1], hidden, backward)
    return torch.empty(max(nb, 16), dtype=torch.uint8, device="cuda"), nb


def _check(got, ref, bound, what):
    assert not torch.isnan(got).any(), what
    err = (got.double() - ref).abs()
    assert (err <= bound).all(), f"{what}: {(err / bound).max().item():.2f} of the bound"


def _gelu(u):
    phi = 0.5 * torch.special.erfc(-u * 0.5 ** 0.5)
    return u * phi, phi + u * torch.exp(-0.5 * u * u) * 0.3989422804014327


# 32 rows, one more, parts of a workgroup, several workgroups with a ragged last tile; one and several steps of the hidden channels
SIZES = [(torch.float32, 96, 384), (torch.float32, 96, 64), (torch.float16, 48, 192), (torch.bfloat16, 96, 384), (torch.float16, 96, 128), (torch.float16, 48, 64)]


@pytest.mark.parametrize("N", [32, 33, 129, 3001, 140001])
@pytest.mark.parametrize("dtype,D,hidden", SIZES, ids=lambda v: str(v).split(".")[-1])
def test_mlp_against_float64(dtype, D, hidden, N):
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(N + D)
    rand = lambda *s, std=1.0: (torch.randn(*s, generator=gen) * std).to(dtype).cuda()
    x, w1, b1, w2, b2 = rand(N, D), rand(hidden, D, std=D ** -0.5), rand(hidden, std=0.5), rand(D, hidden, std=hidden ** -0.5), rand(D)
    round_ = ROUND[dtype]
    x64, w1d, w2d = x.double(), w1.double(), w2.double()
    u = x64 @ w1d.t() + b1.double()
    scale = x64.abs() @ w1d.abs().t() + b1.double().abs()
    g64, d64 = _gelu(u)
    g_err = 2e-6 * scale + 1e-6 + round_ * g64.abs() + (2.0 ** -24 if dtype == torch.float16 else 0)
    d_err = 2e-6 * scale + 1e-6 + round_ * d64.abs() + (2.0 ** -24 if dtype == torch.float16 else 0)
    for out in ([dtype] if dtype == torch.float32 else [dtype, torch.float32]):
        res = torch.randn(N, D, generator=gen).to(out).cuda()
        y64 = g64 @ w2d.t() + b2.double() + res.double()
        y_err = g_err @ w2d.abs().t() + 2e-6 * (g64.abs() @ w2d.abs().t() + b2.double().abs() + res.double().abs()) + ROUND[out] * y64.abs()
        for train in (True, False):
            y, g, d = _empty((N, D), out), _empty((N, hidden), dtype) if train else None, _empty((N, hidden), dtype) if train else None
            ws, nb = _workspace(lib, x, hidden, 0)
            _lib.check(lib.sswin_mlp_forward(CODE[dtype], CODE[out], _ptr(x), N, D, hidden, _ptr(w1), _ptr(b1), _ptr(w2), _ptr(b2), _ptr(res), _ptr(y),
                                             _ptr(g), _ptr(d), _ptr(ws), nb, _stream()))
            _check(y, y64, y_err, f"y {out} train {train}")
            if train:
                _check(g, g64, g_err, "act")
                _check(d, d64, d_err, "slope")
    # without biases and residual
    y = _empty((N, D), dtype)
    ws, nb = _workspace(lib, x, hidden, 0)
    _lib.check(lib.sswin_mlp_forward(CODE[dtype], CODE[dtype], _ptr(x), N, D, hidden, _ptr(w1), None, _ptr(w2), None, None, _ptr(y), None, None, _ptr(ws), nb,
                                     _stream()))
    g0 = _gelu(x64 @ w1d.t())[0]
    bound = 2e-6 * (x64.abs() @ w1d.abs().t()) + 1e-6 + round_ * g0.abs() + (2.0 ** -24 if dtype == torch.float16 else 0)
    y0 = g0 @ w2d.t()
    _check(y, y0, bound @ w2d.abs().t() + 2e-6 * (g0.abs() @ w2d.abs().t()) + round_ * y0.abs(), "y without biases")

    dy, slope = rand(N, D), d64.to(dtype)
    du64 = (dy.double() @ w2d) * slope.double()
    du_err = 2e-6 * (dy.double().abs() @ w2d.abs()) * slope.double().abs() + round_ * du64.abs() + (2.0 ** -24 if dtype == torch.float16 else 1e-30)
    dx64 = du64 @ w1d
    dx_err = du_err @ w1d.abs() + 2e-6 * (du64.abs() @ w1d.abs()) + round_ * dx64.abs() + (2.0 ** -24 if dtype == torch.float16 else 0)
    du, dx = _empty((N, hidden), dtype), _empty((N, D), dtype)
    ws, nb = _workspace(lib, x, hidden, 1)
    _lib.check(lib.sswin_mlp_backward(CODE[dtype], _ptr(dy), N, D, hidden, _ptr(w1), _ptr(w2), _ptr(slope), _ptr(du), _ptr(dx), _ptr(ws), nb, _stream()))
    _check(du, du64, du_err, "du")
    _check(dx, dx64, dx_err, "dx")


def test_mlp_refuses_what_it_does_not_take():
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    for dtype, n, d, hidden in [(0, 31, 96, 384), (0, 64, 48, 192), (0, 64, 96, 400), (2, 64, 96, 32), (2, 64, 96, 100), (2, 64, 112, 448), (2, 64, 192, 768), (2, 64, 96, 1056), (3, 64, 96, 384)]:
        assert not lib.sswin_mlp_supported(dtype, n, d, hidden)
        assert lib.sswin_mlp_backward(dtype, None, n, d, hidden, None, None, None, None, None, None, 1 << 30, None) != 0


def test_mlp_is_preferred_later_with_many_hidden_channels():
    """A wavefront's time grows with the hidden channels: 16 bit, beyond 384 of them the two layers are ahead up to 32 rows a channel."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    for d, hidden, rows in [(48, 192, 8192), (96, 384, 8192), (48, 384, 8192), (96, 416, 13312), (96, 768, 24576), (48, 1024, 32768)]:
        for dtype in (1, 2):
            assert lib.sswin_mlp_preferred(dtype, rows, d, hidden) and not lib.sswin_mlp_preferred(dtype, rows - 1, d, hidden)


def test_mlp_refuses_results_over_rows_it_reads():
    """The last rows are read twice: a result in the place of an input would change them in between.  Refused on the host."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    N, D, hidden = 65, 48, 192
    rows = lambda width, dtype=torch.float16: torch.zeros(N, width, dtype=dtype, device="cuda")
    x, y, w1, w2, act, slope = rows(D), rows(D), torch.zeros(hidden, D, device="cuda").half(), torch.zeros(D, hidden, device="cuda").half(), rows(hidden), rows(hidden)
    ws, nb = _workspace(lib, x, hidden, 1)
    wide = torch.zeros(N + 64, D, dtype=torch.float16, device="cuda")
    forward = lambda x, residual, y, act, slope: lib.sswin_mlp_forward(1, 1, _ptr(x), N, D, hidden, _ptr(w1), None, _ptr(w2), None, _ptr(residual), _ptr(y), _ptr(act),
                                                                       _ptr(slope), None, 0, _stream())
    backward = lambda dy, slope, du, dx: lib.sswin_mlp_backward(1, _ptr(dy), N, D, hidden, _ptr(w1), _ptr(w2), _ptr(slope), _ptr(du), _ptr(dx), _ptr(ws), nb, _stream())
    for args in [(x, y, y, None, None), (x, None, x, None, None), (wide, None, wide[64:], None, None), (wide[64:], None, wide, None, None), (act, None, y, act, slope),
                 (slope, None, y, act, slope)]:
        assert forward(*args) != 0 and b"overlap" in lib.sswin_last_error()
    for args in [(x, slope, act, x), (x, slope, slope, y), (act, slope, act, y)]:
        assert backward(*args) != 0 and b"overlap" in lib.sswin_last_error()
    assert forward(x, None, y, act, slope) == 0 and backward(x, slope, act, y) == 0


# behind the last full round of workgroups of 256 rows the tiles of 32 are dealt to all compute units: none, one, two and seven a
# workgroup, after no, one and two rounds
@pytest.mark.parametrize("rounds,tiles,extra", [(1, 0, 0), (0, 1, 1), (0, 2, -1), (1, 1, 31), (1, 7, 0), (2, 0, 1)])
def test_mlp_last_round(rounds, tiles, extra):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    test_mlp_against_float64(torch.float32, 96, 64, 32 * cus * (8 * rounds + tiles) + extra)


@pytest.mark.parametrize("N", [16385, 17001, 19072, 19073, 32768])
def test_mlp_fp32_sums_no_less_exactly_than_two_layers(N):
    """Where the launch is preferred, its error against float64 (2-norms) is at most that of the layers it stands for, up to 2 % for the
    spread of the inputs: they sum few rows in eight parts."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    D, hidden, gen = 96, 384, torch.Generator().manual_seed(N)
    assert lib.sswin_mlp_preferred(0, N, D, hidden) == (N > 19072)      # 149 tiles of 128 rows: few rows
    if N <= 19072:
        return
    rand = lambda *s, std=1.0: (torch.randn(*s, generator=gen) * std).cuda()
    x, w1, w2, dy, slope = rand(N, D), rand(hidden, D, std=D ** -0.5), rand(D, hidden, std=hidden ** -0.5), rand(N, D), rand(N, hidden)
    empty = lambda width: _empty((N, width), torch.float32)
    y, dx, du, act, y2, dx2, du2 = empty(D), empty(D), empty(hidden), empty(hidden), empty(D), empty(D), empty(hidden)
    nb = max(lib.sswin_mlp_workspace_bytes(0, D, hidden, 1), lib.sswin_mlp_workspace_bytes(0, D, hidden, 0), lib.sswin_dense_forward_workspace_bytes(0, N, hidden, D),
             lib.sswin_dense_forward_workspace_bytes(0, N, D, hidden), 16)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    layer = lambda turned, epilogue, a, k, w, p, extra, out: _lib.check(lib.sswin_dense_forward(0, 0, turned, epilogue, _ptr(a), N, k, _ptr(w), None, p, _ptr(extra), _ptr(out),
                                                                                              None, _ptr(ws), nb, _stream()))
    layer(0, 1, x, D, w1, hidden, None, act)                              # GELU
    layer(0, 0, act, hidden, w2, D, None, y2)
    layer(1, 3, dy, D, w2, hidden, slope, du2)                            # times the slope
    layer(1, 0, du2, hidden, w1, D, None, dx2)
    _lib.check(lib.sswin_mlp_forward(0, 0, _ptr(x), N, D, hidden, _ptr(w1), None, _ptr(w2), None, None, _ptr(y), None, None, _ptr(ws), nb, _stream()))
    _lib.check(lib.sswin_mlp_backward(0, _ptr(dy), N, D, hidden, _ptr(w1), _ptr(w2), _ptr(slope), _ptr(du), _ptr(dx), _ptr(ws), nb, _stream()))
    y64 = _gelu(x.double() @ w1.double().t())[0] @ w2.double().t()
    dx64 = ((dy.double() @ w2.double()) * slope.double()) @ w1.double()
    for one, two, ref, what in ((y, y2, y64, "y"), (dx, dx2, dx64, "dx")):
        errors = [((t.double() - ref).norm() / ref.norm()).item() for t in (one, two)]
        assert errors[0] <= 1.02 * errors[1], (what, errors)


@pytest.mark.parametrize("span", [20, -20])
@pytest.mark.parametrize("N,hidden", [(33, 64), (3001, 384)])
def test_mlp_fp32_scales(N, hidden, span):
    """fp32 operands are split into fp16 pieces, scaled by row: rows of any size; hidden values that grow or fall by 2^20 over the hidden
    channels, met by weights that fall or grow as much, so that each counts the same; rows whose first hidden values are zero.  Bounds as
    above: the sums of absolute products."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    D, gen = 96, torch.Generator().manual_seed(N)
    rand = lambda *s, std=1.0: torch.randn(*s, generator=gen) * std
    ramp = torch.exp2(torch.linspace(-span / 2, span / 2, hidden).round())
    size = torch.exp2(torch.randint(-60, 61, (N, 1), generator=gen).float())
    dy, w1, w2, slope = rand(N, D) * size, rand(hidden, D) / ramp[:, None], rand(D, hidden), rand(N, hidden) * ramp
    slope[N // 2, :hidden - 5] = 0
    dy, w1, w2, slope = (t.cuda() for t in (dy, w1, w2, slope))
    du64 = (dy.double() @ w2.double()) * slope.double()
    du_err = 2e-6 * (dy.double().abs() @ w2.double().abs()) * slope.double().abs()
    dx_err = du_err @ w1.double().abs() + 2e-6 * (du64.abs() @ w1.double().abs())
    du, dx = _empty((N, hidden), torch.float32), _empty((N, D), torch.float32)
    ws, nb = _workspace(lib, dy, hidden, 1)
    _lib.check(lib.sswin_mlp_backward(0, _ptr(dy), N, D, hidden, _ptr(w1), _ptr(w2), _ptr(slope), _ptr(du), _ptr(dx), _ptr(ws), nb, _stream()))
    _check(du, du64, du_err + 1e-30, "du")
    _check(dx, du64 @ w1.double(), dx_err + 1e-30, "dx")
    x, w1, w2 = dy / size.cuda() * torch.exp2(torch.randint(-8, 9, (N, 1), generator=gen).float()).cuda(), w1 * ramp[:, None].cuda() ** 2, w2 / ramp.cuda()
    g64 = _gelu(x.double() @ w1.double().t())[0]
    g_err = 2e-6 * (x.double().abs() @ w1.double().abs().t()) + 1e-6 * g64.abs().clamp(max=1)
    y = _empty((N, D), torch.float32)
    ws, nb = _workspace(lib, x, hidden, 0)
    _lib.check(lib.sswin_mlp_forward(0, 0, _ptr(x), N, D, hidden, _ptr(w1), None, _ptr(w2), None, None, _ptr(y), None, None, _ptr(ws), nb, _stream()))
    _check(y, g64 @ w2.double().t(), g_err @ w2.double().abs().t() + 2e-6 * (g64.abs() @ w2.double().abs().t()) + 1e-30, "y")


def test_mlp_fp32_hidden_values_that_begin_with_zeros():
    """A token's results have the same bits whatever stands beside it: zeros in the first hidden values of every token or of some."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    N, D, hidden, gen = 3001, 96, 384, torch.Generator(device="cuda").manual_seed(4)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    dy, w1, w2, slope = rand(N, D), rand(hidden, D), rand(D, hidden), rand(N, hidden)
    some, every = slope.clone(), slope
    some[::3, :100] = 0
    every[:, :100] = 0
    ws, nb = _workspace(lib, dy, hidden, 1)
    dxs = []
    for t in (some, every):
        du, dx = _empty((N, hidden), torch.float32), _empty((N, D), torch.float32)
        _lib.check(lib.sswin_mlp_backward(0, _ptr(dy), N, D, hidden, _ptr(w1), _ptr(w2), _ptr(t), _ptr(du), _ptr(dx), _ptr(ws), nb, _stream()))
        dxs.append(dx[::3])
    assert torch.equal(*dxs)


def test_mlp_fp32_inference_has_the_bits_of_training():
    """Rows enough for results that are small by chance, with and without weights that lose bits."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    N, D, hidden, gen = 100003, 96, 384, torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    x, w1, w2, b1, b2, res = rand(N, D), rand(hidden, D) * D ** -0.5, rand(D, hidden) * hidden ** -0.5, rand(hidden) * 0.1, rand(D) * 0.1, rand(N, D)
    ws, nb = _workspace(lib, x, hidden, 0)
    for k in range(3):
        if k == 1:
            w2[5, 7] = w1[9, 3] = 1e-12
        elif k == 2:
            b1[11] = 1e7                                          # a hidden channel above the rest, so that the others lose bits
            w2[:, 11] *= 1e-7
        ys = []
        for train in (False, True):
            y, act, slope = _empty((N, D), torch.float32), _empty((N, hidden), torch.float32), _empty((N, hidden), torch.float32)
            _lib.check(lib.sswin_mlp_forward(0, 0, _ptr(x), N, D, hidden, _ptr(w1), _ptr(b1), _ptr(w2), _ptr(b2), _ptr(res), _ptr(y), _ptr(act) if train else None,
                                             _ptr(slope) if train else None, _ptr(ws), nb, _stream()))
            ys.append(y)
        assert torch.equal(*ys), k


@pytest.mark.parametrize("span", [40, -40, 60])
@pytest.mark.parametrize("N,hidden", [(33, 64), (3001, 384)])
def test_mlp_fp32_scales_that_the_pieces_do_not_span(N, hidden, span):
    test_mlp_fp32_scales(N, hidden, span)


@pytest.mark.parametrize("power", [30, 40])
@pytest.mark.parametrize("where", ["token", "tokens", "weight", "ramp"])
@pytest.mark.parametrize("N,hidden", [(33, 64), (3001, 384)])
def test_mlp_fp32_of_a_channel_above_the_rest(N, hidden, where, power):
    """A channel of a token 2^power above its others, seen by one hidden channel alone, and that by all columns but some: hidden values and
    results that are small against what their rows hold, in one token of a tile or in most.  A weight of a hidden channel as much above its others, met
    by zeros in a few tokens; channels of a token that grow by as much and meet weights that fall, or fall and meet weights that grow."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    D, gen = 96, torch.Generator().manual_seed(N + power)
    rand = lambda *s: torch.randn(*s, generator=gen)
    x, wa, wb = rand(N, D), rand(hidden, D), rand(D, hidden)      # forward: w1 and w2, backward: w2^T and w1^T
    if where == "weight":
        wa[hidden - 7, 17] = 2.0 ** power
        x[N // 2, 17] = x[5, 17] = 0
    elif where == "ramp":
        ramp = torch.exp2(torch.linspace(-power, power, D).round() * (1 if hidden == 64 else -1))
        x, wa = x * ramp, wa / ramp
    else:
        x[0 if where == "tokens" else N // 2:N - 3 if where == "tokens" else N // 2 + 1, 17] = 2.0 ** power
        wa[:, 17], wa[hidden - 7, 17] = 0, 1
    wb[::5, hidden - 7] = 0
    wa[11], wb[20], x[N - 1] = 0, 0, 0
    slope = (rand(N, hidden) * 0.5 + 0.5).cuda()
    x, wa, wb = x.cuda(), wa.cuda(), wb.cuda()
    z64, mag = x.double() @ wa.double().t(), x.double().abs() @ wa.double().abs().t()
    g64, s64 = _gelu(z64)
    g_err = 2e-6 * mag + 1e-6 * g64.abs().clamp(max=1)
    y_err = g_err @ wb.double().abs().t() + 2e-6 * (g64.abs() @ wb.double().abs().t()) + 1e-30
    ws, nb = _workspace(lib, x, hidden, 0)
    ys = []
    for train in (False, True):
        y, act, slope_out = _empty((N, D), torch.float32), _empty((N, hidden), torch.float32), _empty((N, hidden), torch.float32)
        _lib.check(lib.sswin_mlp_forward(0, 0, _ptr(x), N, D, hidden, _ptr(wa), None, _ptr(wb), None, None, _ptr(y), _ptr(act) if train else None,
                                         _ptr(slope_out) if train else None, _ptr(ws), nb, _stream()))
        _check(y, g64 @ wb.double().t(), y_err, f"y, training {train}")
        ys.append(y)
    assert torch.equal(*ys)                                       # inference has the bits of training
    _check(act, g64, g_err + 1e-30, "act")
    _check(slope_out, s64, 2e-6 * mag + 1e-6, "slope")
    du64 = z64 * slope.double()
    du_err = 2e-6 * mag * slope.double().abs()
    dx_err = du_err @ wb.double().abs().t() + 2e-6 * (du64.abs() @ wb.double().abs().t())
    w2, w1 = wa.t().contiguous(), wb.t().contiguous()
    du, dx = _empty((N, hidden), torch.float32), _empty((N, D), torch.float32)
    ws, nb = _workspace(lib, x, hidden, 1)
    _lib.check(lib.sswin_mlp_backward(0, _ptr(x), N, D, hidden, _ptr(w1), _ptr(w2), _ptr(slope), _ptr(du), _ptr(dx), _ptr(ws), nb, _stream()))
    _check(du, du64, du_err + 1e-30, "du")
    _check(dx, du64 @ wb.double().t(), dx_err + 1e-30, "dx")


def _same_class(got, ref, bound, what):
    """Finite where float64 is (to the bound), the same infinities, NaN where float64 has NaN."""
    got, finite = got.double(), ref.isfinite()
    assert got[finite].isfinite().all(), what
    assert ((got - ref)[finite].abs() <= bound[finite]).all(), what
    assert torch.equal(got[ref.isinf()], ref[ref.isinf()]), what
    assert got[ref.isnan()].isnan().all(), what


@pytest.mark.parametrize("N,hidden", [(33, 64), (3001, 384), (16500, 64)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4028234e38])
@pytest.mark.parametrize("where", ["rows", "w1", "b1", "w2", "slope"])
def test_mlp_fp32_of_values_that_are_not_finite(N, hidden, value, where):
    """An infinity, a NaN or the largest number in a few places: hidden values, results and gradients are those of plain fp32
    arithmetic, as where the two layers run one by one.  (Everything else is small where the largest number is, so that results are in
    range.)  Bounds of finite results: as above."""
    from sparseswin3d_amd import _lib
    lib = _lib.load()
    D, gen = 96, torch.Generator().manual_seed(N)
    small = 2.0 ** -10 if abs(value) < float("inf") else 1.0
    rand = lambda *s, std=1.0: torch.randn(*s, generator=gen) * std * small
    x, w1, b1, w2, dy, slope = rand(N, D), rand(hidden, D, std=D ** -0.5), rand(hidden), rand(D, hidden, std=hidden ** -0.5), rand(N, D), rand(N, hidden)
    for t in {"rows": (x, dy), "w1": (w1,), "b1": (b1,), "w2": (w2,), "slope": (slope,)}[where]:
        if t.dim() == 1:
            t[hidden // 2 + 3] = value
        else:
            t[1, 0], t[t.shape[0] // 2, t.shape[1] - 1] = value, value
    x[N // 3], dy[N // 3] = 0, 0                                   # 0 x inf
    x, w1, b1, w2, dy, slope = (t.cuda() for t in (x, w1, b1, w2, dy, slope))
    w1d, w2d = w1.double(), w2.double()
    u, scale = x.double() @ w1d.t() + b1.double(), x.double().abs() @ w1d.abs().t() + b1.double().abs()
    g64, d64 = _gelu(u)
    err = 2e-6 * scale + 1e-6
    y64, y_err = g64 @ w2d.t(), err @ w2d.abs().t() + 2e-6 * (g64.abs() @ w2d.abs().t())
    for train in (True, False):
        y, g, d = _empty((N, D), torch.float32), *((_empty((N, hidden), torch.float32) if train else None) for _ in range(2))
        ws, nb = _workspace(lib, x, hidden, 0)
        _lib.check(lib.sswin_mlp_forward(0, 0, _ptr(x), N, D, hidden, _ptr(w1), _ptr(b1), _ptr(w2), None, None, _ptr(y), _ptr(g), _ptr(d), _ptr(ws), nb, _stream()))
        _same_class(y, y64, y_err, f"y train {train}")
        if train:
            _same_class(g, g64, err, "act")
            _same_class(d, d64, err, "slope")
    if where == "b1":
        return
    du64 = (dy.double() @ w2d) * slope.double()
    du_err = 2e-6 * (dy.double().abs() @ w2d.abs()) * slope.double().abs() + 1e-30
    dx64, dx_err = du64 @ w1d, du_err @ w1d.abs() + 2e-6 * (du64.abs() @ w1d.abs())
    du, dx = _empty((N, hidden), torch.float32), _empty((N, D), torch.float32)
    ws, nb = _workspace(lib, x, hidden, 1)
    _lib.check(lib.sswin_mlp_backward(0, _ptr(dy), N, D, hidden, _ptr(w1), _ptr(w2), _ptr(slope), _ptr(du), _ptr(dx), _ptr(ws), nb, _stream()))
    _same_class(du, du64, du_err, "du")
    _same_class(dx, dx64, dx_err, "dx")
    assert (abs(value) < float("inf")) == bool(y64.isfinite().all() and dx64.isfinite().all() if where != "slope" else dx64.isfinite().all())
