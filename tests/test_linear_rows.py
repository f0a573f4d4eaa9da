"""Products of few rows that stream their weights: edges of row tiles, channel
blocks, steps and parts of K, and the calls that stay with the library,
against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EXTENSIONS = ["_hip_ops", "_hip_layered"]


def _ext(name):
    import importlib
    return importlib.import_module(f"llm_d_inference_scheduler_amd.{name}")


def _draw(*shape, seed=0, scale=1.0):
    g = torch.Generator("cuda").manual_seed(seed)
    return (torch.randn(*shape, device="cuda", generator=g) *
            scale).bfloat16()


def _same(got, want, bits):
    """Sums of 32 bits over K products of size 1 / sqrt(K): far below 1e-5;
    the result is rounded to `bits` bits."""
    torch.testing.assert_close(got.double(), want, rtol=2.0 ** -bits,
                               atol=2e-5)


@pytest.mark.parametrize("rows", [1, 2, 15, 16, 17, 32, 33, 63, 64, 65, 96,
                                  97, 128, 129, 192, 193, 255, 256, 257])
@pytest.mark.parametrize("n,k", [(8, 8), (120, 64), (128, 136), (136, 520),
                                 (1032, 1000), (264, 4096), (33032, 72),
                                 (60008, 72), (4088, 256), (30000, 264)])
def test_product(rows, n, k):
    ext = _ext("_hip_ops")
    x, w = _draw(rows, k, seed=rows), _draw(n, k, seed=n, scale=k ** -0.5)
    want = x.double() @ w.double().t()
    _same(ext.linear(x, w), want, 8)
    wide = ext.linear32(x, w)
    assert (wide is None) == (not ext.few_rows(x, w))
    # not where 33032 channels need a second round for a few of them
    assert ext.few_rows(x, w) or rows > 64 or n == 33032
    if wide is not None:
        _same(wide, want, 16)


@pytest.mark.parametrize("name", EXTENSIONS)
@pytest.mark.parametrize("rows", [1, 16, 17, 64, 65, 128, 192, 193, 257])
@pytest.mark.parametrize("n,k", [(8, 64), (520, 128), (14400, 200),
                                 (16384, 48), (16400, 48)])
def test_gated(name, rows, n, k):
    """The last block partly empty; what the library does better gives
    None."""
    F = torch.nn.functional
    x = _draw(rows, k, seed=rows)
    w = _draw(2 * n, k, seed=n, scale=k ** -0.5)
    g, u = (x.double() @ w.double().t()).chunk(2, -1)
    for act, fn in enumerate([lambda z: F.gelu(z, approximate="tanh"), F.silu,
                              lambda z: z.relu().square()]):
        y = _ext(name).gated_linear(x, w, act)
        assert (y is None) == (rows > 192 or n not in (14400, 16384))
        if y is not None:
            _same(y, fn(g) * u, 8)


@pytest.mark.parametrize("rows", [192, 193, 255, 256])
@pytest.mark.parametrize("n,k,parts", [(4088, 8320, 8), (7304, 4224, 4),
                                       (7304, 4232, 4), (12576, 2048, 2)])
def test_parts_of_many_steps(rows, n, k, parts):
    """Ends of rows, channels and K of the loop for large parts (its K is a
    multiple of 128), and the bits of a row alone."""
    ext = _ext("_hip_ops")
    x, w = _draw(rows, k, seed=rows), _draw(n, k, seed=n, scale=k ** -0.5)
    y = ext.linear_parts(x, w)
    assert y.shape == (parts, rows, n) and y.dtype == torch.float32
    _same(y.sum(0), x.double() @ w.double().t(), 12)
    assert torch.equal(y[:, -1:], ext.linear_parts(x[-1:], w))


@pytest.mark.parametrize("rows", [65, 128, 129, 192, 193, 256])
@pytest.mark.parametrize("n,k,parts", [
    (16392, 1024, 1), (20488, 1152, 1), (16392, 1032, 1), (4088, 14336, 8),
    (9224, 5504, 3), (12576, 3968, 2)])
def test_whole_lines(rows, n, k, parts):
    """Ends of groups of 64 rows, of channels, and even and odd numbers of steps of
    128 of K; a K that is none goes by halves. With parts, the bits of a row alone."""
    ext = _ext("_hip_ops")
    x, w = _draw(rows, k, seed=rows), _draw(n, k, seed=n, scale=k ** -0.5)
    want = x.double() @ w.double().t()
    assert ext.few_rows(x, w) or parts > 1
    _same(ext.linear(x, w), want, 8)
    got = ext.linear_parts(x, w)
    if parts > 1:
        assert got.shape == (parts, rows, n)
        _same(got.sum(0), want, 16)
        for at in (0, rows - 1):
            assert torch.equal(got[:, at:at + 1],
                               ext.linear_parts(x[at:at + 1], w))
    half = n // 16 * 8
    gate, up = want[:, :half], want[:, half:2 * half]
    y = ext.gated_linear(x, w[:2 * half], 2)
    assert (y is None) == (half <= 64 * 159)
    if y is not None:
        _same(y, gate.relu().square() * up, 8)


@pytest.mark.parametrize("rows", [193, 256])
@pytest.mark.parametrize("n,k", [(14400, 1024), (16368, 1152), (14400, 1096)])
def test_gated_of_many_steps(rows, n, k):
    x, w = _draw(rows, k, seed=rows), _draw(2 * n, k, seed=n, scale=k ** -0.5)
    y = _ext("_hip_ops").gated_linear(x, w, 1)
    assert (y is None) == (k % 128 > 0)
    if y is not None:
        g, u = (x.double() @ w.double().t()).chunk(2, -1)
        _same(y, torch.nn.functional.silu(g) * u, 8)
        assert torch.equal(y[-1:], _ext("_hip_ops").gated_linear(x[-1:], w, 1))


@pytest.mark.parametrize("rows", [193, 256])
@pytest.mark.parametrize("n,k,one", [(16384, 1024, True), (14336, 8192, True),
                                     (14336, 8320, False), (14336, 896, False),
                                     (28744, 3584, False), (32768, 1024, False),
                                     (46168, 2176, False)])
def test_gated_of_one_round(rows, n, k, one):
    """More than a round of workgroups, or longer K: the library and the activation
    apart are faster."""
    x = torch.zeros(rows, k, device="cuda").bfloat16()
    w = torch.zeros(2 * n, k, dtype=torch.bfloat16, device="cuda")
    for name in EXTENSIONS:
        assert (_ext(name).gated_linear(x, w, 1) is not None) == one


@pytest.mark.parametrize("rows,one", [(192, True), (193, False), (256, False)])
@pytest.mark.parametrize("of_x", [False, True])
def test_gated_of_far_rows(rows, one, of_x):
    """Rows spread over 4 GiB and more: up to 192 of x in one kernel, with offsets of
    64 bits; more go to the library, as the kernel for them has 32."""
    n, k = 14400, 1024

    def far(t):
        row = ((1 << 31) // len(t) + 8) // 8 * 8
        out = torch.empty(len(t), row, dtype=t.dtype, device="cuda")[:, :k]
        return out.copy_(t)
    x, w = _draw(rows, k, seed=rows), _draw(2 * n, k, seed=n, scale=k ** -0.5)
    assert _ext("_hip_ops").gated_linear(x, w, 1) is not None
    y = _ext("_hip_ops").gated_linear(*((far(x), w) if of_x else (x, far(w))), 1)
    assert (y is not None) == one
    if one:
        g, u = (x.double() @ w.double().t()).chunk(2, -1)
        _same(y, torch.nn.functional.silu(g) * u, 8)


@pytest.mark.parametrize("name", EXTENSIONS)
@pytest.mark.parametrize("rows,n,k", [
    (257, 1024, 5120), (384, 1288, 5184), (385, 1032, 8192), (512, 4088, 14336),
    (513, 5120, 6400), (1000, 4096, 7168), (1300, 5120, 25600),
    (2560, 1024, 16384)])
def test_split_of_many_rows(name, rows, n, k):
    """Tiles of 192 and 256 rows that are partly empty, channels that end inside a
    tile, uneven parts of K, rows further apart than their length: each part is a
    sum of its own K, and all are the product. Sums as in _same."""
    ext = _ext(name)
    plan = ext.split_plan(rows, n, k)
    parts = plan >> 16
    assert parts > 1 and plan % 65536 in (192, 256)
    x = _draw(rows, k + 72, seed=rows)[:, 8:k + 8]
    w = _draw(n, k, seed=n, scale=k ** -0.5)
    want = x.double() @ w.double().t()
    _same(ext.linear(x, w), want, 8)
    got = ext.linear_parts(x, w)
    assert got.shape == (parts, rows, n) and got.dtype == torch.float32
    _same(got.double().sum(0), want, 16)
    ends = [k // 64 * i // parts * 64 for i in range(parts + 1)]
    for i in (0, parts - 1):
        a, b = ends[i:i + 2]
        _same(got[i], x[:, a:b].double() @ w[:, a:b].double().t(), 16)


@pytest.mark.parametrize("rows,n,k", [
    (256, 4096, 14336), (257, 4096, 5056), (257, 4096, 5128), (257, 1020, 8192),
    (257, 1016, 8192), (257, 0, 8192), (0, 4096, 8192), (257, 4096, 0),
    (2300, 5120, 25600), (2561, 1024, 16384), (1 << 62, 1 << 62, 1 << 62)])
def test_products_that_stay_whole(rows, n, k):
    """Few rows, short or odd K, odd or narrow widths, many rows, and what fills the
    compute units."""
    assert _ext("_hip_ops").split_plan(rows, n, k) == 0


def test_split_of_what_is_left():
    """Rows behind whole rounds of tiles, in a call of their own."""
    ext = _ext("_hip_ops")
    assert ext.whole_rounds(4400, 4096, 8192) == 4096
    assert ext.split_plan(304, 4096, 8192)
    x, w = _draw(4400, 8192, seed=1), _draw(4096, 8192, seed=2, scale=1 / 91)
    y = ext.linear(x, w)
    _same(y, x.double() @ w.double().t(), 8)
    assert torch.equal(y[4096:], ext.linear(x[4096:], w))


@pytest.mark.parametrize("name", EXTENSIONS)
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("rows,n,k,tile", [
    (640, 10880, 128, 256), (560, 10872, 192, 192), (897, 8192, 320, 256),
    (1024, 8136, 256, 256), (350, 14344, 128, 192), (300, 14344, 192, 192),
    (1153, 8128, 128, 192), (512, 16384, 64, 0), (640, 10880, 136, 0),
    (300, 8192, 128, 0)])
def test_act_of_many_rows(name, gated, rows, n, k, tile):
    """Tiles of 256 and 192 rows and a last one of up to 128 or more, channels that
    end inside a tile, even and odd numbers of steps, rows that lie apart; what does
    not fill its rounds of tiles and other sizes of K stay apart."""
    F, ext, one = torch.nn.functional, _ext(name), tile > 0
    assert ext.act_rows(rows, n if gated else 2 * n, k, gated) == tile
    n *= 1 if gated else 2
    x = _draw(rows, k + 8, seed=rows)[:, :k]
    w = _draw(2 * n if gated else n, k + 16, seed=n, scale=k ** -0.5)[:, 8:-8]
    z = x.double() @ w.double().t()
    call = ext.gated_linear if gated else ext.activated_linear
    for act, fn in enumerate([lambda z: F.gelu(z, approximate="tanh"), F.silu,
                              lambda z: z.relu().square()]):
        y = call(x, w, act)
        assert (y is not None) == one
        if one:
            g, u = z.chunk(2, -1) if gated else (z, 1)
            _same(y, fn(g) * u, 8)


@pytest.mark.parametrize("name", EXTENSIONS)
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("rows,n,tile", [
    (385, 24576, 256), (400, 24568, 256), (512, 24576, 256), (3400, 10000, 256),
    (5700, 4992, 256)])
def test_act_of_cut_tiles(name, gated, rows, n, tile):
    """Tiles behind whole rounds cut in two, up to half a round of them: a last row
    alone, a second half without rows and with some, channels that end inside a tile;
    a tile more than half a round, cut and whole."""
    F, ext, k = torch.nn.functional, _ext(name), 128
    n *= 1 if gated else 2
    assert ext.act_rows(rows, n, k, gated) == tile
    x, w = _draw(rows, k, seed=rows), _draw(n * (1 + gated), k, seed=n, scale=k ** -0.5)
    y = (ext.gated_linear if gated else ext.activated_linear)(x, w, 1)
    z = x.double() @ w.double().t()
    g, u = z.chunk(2, -1) if gated else (z, 1)
    _same(y, F.silu(g) * u, 8)


@pytest.mark.parametrize("name", EXTENSIONS)
@pytest.mark.parametrize("rows,n,k", [(1, 8, 512), (16, 4096, 520), (17, 7168, 4096),
                                      (64, 4088, 8192), (60, 30000, 264)])
def test_act_of_few_rows(name, rows, n, k):
    """The activation where the parts of K are summed; one part stays apart."""
    F, ext = torch.nn.functional, _ext(name)
    x, w = _draw(rows, k, seed=rows), _draw(n, k, seed=n, scale=k ** -0.5)
    z = x.double() @ w.double().t()
    for act, fn in enumerate([lambda z: F.gelu(z, approximate="tanh"), F.silu,
                              lambda z: z.relu().square()]):
        y = ext.activated_linear(x, w, act)
        assert (y is None) == (n == 30000)
        if y is not None:
            _same(y, fn(z), 8)


@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("rows_of_w,k", [
    (8192, 1024), (8208, 1032), (4112, 2048), (16384, 1152), (16400, 1280),
    (9232, 4104), (1024, 1064), (28672, 2080)])
def test_width_of_workgroups(rows, rows_of_w, k):
    """Ends of blocks of 64 and 128 rows of w, K in halves of which the second is shorter
    or ends inside a step: one part, its activation, 32-bit, gated."""
    F, ext = torch.nn.functional, _ext("_hip_layered")
    x = _draw(rows, k, seed=rows)
    w = _draw(rows_of_w, k, seed=rows_of_w, scale=k ** -0.5)
    z = x.double() @ w.double().t()
    _same(ext.linear(x, w), z, 8)
    _same(ext.linear32(x, w), z, 16)
    y = ext.activated_linear(x, w, 1)
    assert (y is not None) == (rows_of_w <= 16384)
    if y is not None:
        _same(y, F.silu(z), 8)
    g, u = z.chunk(2, -1)
    y = ext.gated_linear(x, w, 1)
    assert y is not None or k > 4096 or rows_of_w == 1024 and k > 2048
    if y is not None:
        _same(y, F.silu(g) * u, 8)


@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("rows_of_w,k", [
    (16400, 512), (16416, 520), (24576, 768), (28688, 640), (32784, 512), (41008, 1032),
    (47120, 512), (57344, 520), (65552, 640), (70016, 512)])
def test_even_rounds(rows, rows_of_w, k):
    """Blocks of 80 to 128 rows of w: waves without rows, the last block's end."""
    F, ext = torch.nn.functional, _ext("_hip_layered")
    x = _draw(rows, k, seed=rows)
    w = _draw(rows_of_w, k, seed=rows_of_w, scale=k ** -0.5)
    z = x.double() @ w.double().t()
    _same(ext.linear(x, w), z, 8)
    g, u = z.chunk(2, -1)
    _same(ext.gated_linear(x, w, 1), F.silu(g) * u, 8)


@pytest.mark.parametrize("rows", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("n,k", [(8, 8), (24, 128), (520, 136), (4096, 128), (4096, 520),
                                 (4104, 1024)])
def test_pair(rows, n, k):
    """Two products in a launch: columns of one tensor, the last block of the first."""
    ext = _ext("_hip_layered")
    x = _draw(rows, 2 * k + 8, seed=rows)
    w, w2 = (_draw(n, k, seed=n + i, scale=k ** -0.5) for i in range(2))
    pair = ext.linear_pair(x[:, 8:k + 8], w, x[:, k + 8:], w2)
    for y, a, b in zip(pair, (x[:, 8:k + 8], x[:, k + 8:]), (w, w2)):
        _same(y, a.double() @ b.double().t(), 8)
    assert ext.linear_pair(x[:, :k], w, x[:, :k], w2[:, :k - 8]) is None
    assert ext.linear_pair(x[:, :k], w, x[:, :k].contiguous(), w2) is None or rows == 1


@pytest.mark.parametrize("name", EXTENSIONS)
@pytest.mark.parametrize("rows,n", [(16, 4096), (8192, 8192)])
@pytest.mark.parametrize("act", [-1, 3, 1 << 32])
def test_no_such_act(name, rows, n, act):
    """Refused ahead of any kernel, of few rows and of many."""
    ext = _ext(name)
    x, w = _draw(rows, 512, seed=1), _draw(n, 512, seed=2)
    assert ext.activated_linear(x, w, 1) is not None
    with pytest.raises(RuntimeError, match="activation"):
        ext.activated_linear(x, w, act)


@pytest.mark.parametrize("act,low,high", [(0, -10.0, -6.0), (1, -88.5, -60.0)])
def test_act_of_small_results(act, low, high):
    """Down to where the exponential overflows: the result's rounding (half a step of 7
    bits behind the point, 2^-8) and the activation's own error, 2^-16 at most."""
    ext = _ext("_hip_layered")
    z = torch.linspace(low, high, 640, device="cuda").bfloat16()
    x = torch.zeros(640, 128, device="cuda").bfloat16()
    x[:, 0] = z
    w = torch.zeros(2 * 10880, 128, device="cuda").bfloat16()
    w[:, 0] = 1
    a = z.double()
    if act == 0:
        a = 2 * 0.7978845608028654 * (a + 0.044715 * a ** 3)
    want = z.double() / (1 + torch.exp(-a))
    got = ext.activated_linear(x, w, act).double()
    torch.testing.assert_close(got, want[:, None].expand_as(got),
                               rtol=2 ** -8 + 2 ** -16, atol=0)


@pytest.mark.parametrize("act", [0, 1, 2])
def test_act_of_large_sums(act):
    """Infinities and what overflows come out as they do apart."""
    ext = _ext("_hip_layered")
    x = torch.zeros(640, 128, device="cuda").bfloat16()
    x[:, 0] = torch.tensor([1, -1, 1e4, -1e4, 1e38, -1e38, 90, -90, 0, -0.0],
                           device="cuda").repeat(64).bfloat16()
    w = torch.zeros(2 * 10880, 128, device="cuda").bfloat16()
    w[::2, 0], w[1::2, 0] = 1, 1e4
    got, want = ext.activated_linear(x, w, act), ext.activate(x @ w.t(), act)
    assert torch.equal(got.isnan(), want.isnan())
    ok = ~want.isnan()
    torch.testing.assert_close(got[ok], want[ok], rtol=2 ** -7, atol=1e-30)


@pytest.mark.parametrize("rows,n,k,whole", [
    (2047, 4096, 4096, 0), (4096, 4096, 4096, 0), (4097, 4096, 96, 4096),
    (4096 + 2048, 4096, 96, 4096), (4096 + 2049, 4096, 96, 0),
    (4096 + 2049, 4096, 4096, 4096), (8192 + 2049, 4096, 96, 8192),
    (4096 + 3840, 4096, 4096, 4096), (4096 + 3841, 4096, 4096, 0),
    (8192 + 3072, 10240, 5120, 8192), (8192 + 3073, 10240, 5120, 0),
    (11456, 14336, 4096, 0), (8533, 14336, 4096, 8192),
    (7749, 12576, 4096, 0), (40000, 12576, 4096, 0)])
def test_which_rows_go_apart(rows, n, k, whole):
    """Up to half a round of tiles behind the whole ones; up to two of them
    that do not end full, where K or the whole ones are large."""
    assert _ext("_hip_ops").whole_rounds(rows, n, k) == whole


@pytest.mark.parametrize("rows", [2048, 4095, 4096, 4097, 4352, 4500, 8193])
@pytest.mark.parametrize("n,k", [(4096, 96), (4090, 72), (16384, 64),
                                 (300, 64)])
def test_whole_rounds_apart(rows, n, k):
    """Many rows in two calls, of which the second may have one row; rows that
    lie apart; errors and other types as ever."""
    ext = _ext("_hip_ops")
    x, w = _draw(rows, k + 8, seed=rows)[:, 8:], _draw(n, k, seed=n,
                                                       scale=k ** -0.5)
    _same(ext.linear(x, w), x.double() @ w.double().t(), 8)
    if n == 4096 and rows == 4500:
        y = ext.linear(x.float(), w.float())
        assert y.dtype == torch.float32
        with pytest.raises(RuntimeError):
            ext.linear(x, w[:, 1:])
        a = x.detach().clone().requires_grad_()
        ext.linear(a, w).float().sum().backward()
        assert a.grad.shape == x.shape


def test_rows_apart():
    """Slices of wider tensors, as the decay and gate projections take."""
    ext = _ext("_hip_layered")
    x, w = _draw(30, 400, seed=1), _draw(64, 304, seed=2)
    a, b = x[:, 16:16 + 136], w[:, 8:8 + 136]
    assert ext.few_rows(a, b)
    torch.testing.assert_close(ext.linear(a, b).double(),
                               a.double() @ b.double().t(), rtol=2 ** -8,
                               atol=1e-3)


def test_calls_that_stay_with_the_library():
    ext = _ext("_hip_layered")
    x, w = _draw(20, 256, seed=3), _draw(64, 256, seed=4, scale=1 / 16)
    want = x.double() @ w.double().t()
    flat = _draw(20 * 256 + 8, seed=5)
    odd = flat[1:1 + 20 * 256].view(20, 256).copy_(x)   # not 16-byte aligned
    across = x.t().contiguous().t()
    for a in (odd, across):
        assert not ext.few_rows(a, w)
        _same(ext.linear(a, w), want, 8)
    assert not ext.few_rows(x, w.t().contiguous().t())
    _same(ext.linear(x, w.t().contiguous().t()), want, 8)
    _same(ext.linear(x.view(4, 5, 256), w).view(20, 64), want, 8)
    _same(ext.linear(x[3], w), want[3], 8)
    assert ext.linear(x[:0], w).shape == (0, 64)
    f = ext.linear(x.float(), w.float())
    assert f.dtype == torch.float32 and not ext.few_rows(x.float(), w.float())
    for k, n in ((252, 64), (256, 60)):
        a, b = _draw(5, k, seed=6), _draw(n, k, seed=7, scale=1 / 16)
        assert not ext.few_rows(a, b)
        _same(ext.linear(a, b), a.double() @ b.double().t(), 8)
    with pytest.raises(RuntimeError):
        ext.linear(x, w[:, :128])
    with pytest.raises(RuntimeError):
        ext.linear(x, w.float())


def test_gradients_pass():
    ext = _ext("_hip_layered")
    x = _draw(6, 64, seed=8).requires_grad_()
    w = _draw(32, 64, seed=9).requires_grad_()
    ext.linear(x, w).float().sum().backward()
    assert x.grad.shape == x.shape and w.grad.shape == w.shape
    with torch.no_grad():
        assert ext.few_rows(x, w)


@pytest.mark.parametrize("name", EXTENSIONS)
@pytest.mark.parametrize("rows", [1, 20, 4500])
def test_calls_that_something_follows(name, rows):
    """A dispatch mode sees the product, a graph traced through one computes
    it anew, and autocast gives it its type."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils._python_dispatch import TorchDispatchMode
    ext, seen = _ext(name), []

    class Record(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func.overloadpacket)
            return func(*args, **(kwargs or {}))
    n, k = (4096, 64) if rows > 256 else (28672, 256)
    x, w = _draw(rows, k, seed=1), _draw(n, k, seed=2, scale=k ** -0.5)
    want = x.double() @ w.double().t()
    with Record():
        y = ext.linear(x, w)
        parts = ext.linear_parts(x, w)
        assert ext.linear32(x, w) is None
        assert ext.gated_linear(x, w, 1) is None
    assert seen.count(torch.ops.aten.mm) == 2
    _same(y, want, 8)
    _same(parts, want, 8)
    traced = make_fx(lambda a: ext.linear(a, w))(_draw(rows, k, seed=3))
    _same(traced(x), want, 8)
    with torch.autocast("cuda", dtype=torch.float16):
        assert ext.linear(x, w).dtype == torch.float16
    with torch.autocast("cuda", dtype=torch.bfloat16):
        _same(ext.linear(x, w), want, 8)


def test_zeros_without_memory():
    ext = _ext("_hip_ops")
    w = _draw(64, 256, seed=4)
    for rows in (20, 4500):
        x = torch._efficientzerotensor((rows, 256), dtype=torch.bfloat16,
                                       device="cuda")
        assert not ext.few_rows(x, w)
        y = ext.linear(x, w)
        assert y.shape == (rows, 64) and not y.any()


@pytest.mark.parametrize("rows,k", [(12, 4096), (60, 4096), (200, 4096),
                                    (300, 8192)])
def test_capture_and_replay(rows, k):
    """Partial sums are written anew by every replay."""
    ext = _ext("_hip_ops")
    x, w = _draw(rows, k, seed=10), _draw(4096, k, seed=11, scale=1 / 64)
    assert rows > 256 or ext.few_rows(x, w)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        ext.linear(x, w)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ext.linear(x, w)
    for i in range(3):
        x.copy_(_draw(rows, k, seed=20 + i))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ext.linear(x, w))


@pytest.mark.parametrize("r,c", [(8, 4), (64, 64), (72, 132), (200, 68),
                                 (12, 20), (8, 6)])
def test_lay_weights(r, c):
    w = _draw(r, c, seed=r).float() * 1.2345
    got = _ext("_hip_ops").lay_weights(w)
    assert got.is_contiguous() and torch.equal(got, w.bfloat16().t())


@pytest.mark.parametrize("rows", [1, 40, 128, 130, 256, 257])
def test_parts_in_norms(rows):
    """rmsnorm and stream_norm sum the parts of a product themselves."""
    from llm_d_inference_scheduler_amd.ops import layered
    hip = _ext("_hip_ops")
    x, w = _draw(rows, 2048, seed=1), _draw(520, 2048, seed=2, scale=1 / 45)
    gain = _draw(520, seed=3)
    y = hip.linear_parts(x, w)
    assert y.dim() == (3 if rows <= 256 else 2)
    if rows <= 256:
        assert y.shape[0] > 1 and y.dtype == torch.float32
    # a library product is rounded to bf16 before anything is added to it
    full = x.double() @ w.double().t() if y.dim() == 3 else y.double()
    for start in (None, _draw(rows, 520, seed=4)):
        residual = None if start is None else start.clone()
        got = hip.rmsnorm(y, gain, 1e-5, residual)
        src = full if start is None else full + start.double()
        if residual is not None:
            _same(residual, src, 8)
        _same(got, src * (src.square().mean(-1, keepdim=True) + 1e-5).rsqrt()
              * gain.double(), 8)
    wb, wn = gain.float(), _draw(520, seed=5).float()
    stream = _draw(rows, 520, seed=6).float()
    for post in (None, wb):
        z = full if post is None else full * (
            full.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * (
            post.double() + 0.5)
        s = stream.double() + z
        mine = stream.clone()
        h = layered.stream_norm(mine, layered.linear_parts(x, w), post, wn,
                                0.5, 1e-5, torch.bfloat16)
        torch.testing.assert_close(mine.double(), s, rtol=1e-5, atol=1e-4)
        _same(h, s * (s.square().mean(-1, keepdim=True) + 1e-5).rsqrt() *
              (wn.double() + 0.5), 8)


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5, 6, 7, 8, 9, 15, 16, 17])
@pytest.mark.parametrize("rows,width", [(3, 8), (2, 2040), (2, 2056), (2, 4104),
                                        (1, 8200), (2, 8192), (1, 16392)])
def test_norms_of_any_parts(rows, width, parts):
    """Whole and rest groups of 8 parts; threads that keep none, some or all of
    their vectors. Sums of up to 17 values of size 1: 32-bit ones within 1e-5; the
    rest as in _same."""
    from llm_d_inference_scheduler_amd.ops import layered
    hip = _ext("_hip_ops")
    g = torch.Generator("cuda").manual_seed(width + parts)
    y = torch.randn(parts, rows, width, device="cuda", generator=g)
    y /= parts ** 0.5
    full, gain = y.double().sum(0), _draw(width, seed=3)

    def normed(z):
        return z * (z.square().mean(-1, keepdim=True) + 1e-5).rsqrt()
    for start in (None, _draw(rows, width, seed=4)):
        residual = None if start is None else start.clone()
        got = hip.rmsnorm(y, gain, 1e-5, residual)
        src = full if start is None else full + start.double()
        if residual is not None:
            _same(residual, src, 8)
        # what does not stay in registers is read again from the residual, whose
        # rounding (2^-8) comes on top of the result's
        twice = residual is not None and width > 8192
        _same(got, normed(src) * gain.double(), 7 if twice else 8)
    wb, wn = gain.float(), _draw(width, seed=5).float()
    rows_of = _draw(2 * rows, width, seed=7)
    for post in (None, wb):
        for more in (None, rows_of):
            z = full if post is None else normed(full) * (post.double() + 0.5)
            if more is not None:
                z = z + more.double().view(rows, 2, width).sum(1)
            mine = _draw(rows, width, seed=6).float()
            s = mine.double() + z
            h = layered.stream_norm(mine, y, post, wn, 0.5, 1e-5,
                                    torch.bfloat16, more)
            torch.testing.assert_close(mine.double(), s, rtol=1e-5, atol=1e-5)
            _same(h, normed(s) * (wn.double() + 0.5), 8)


@pytest.mark.parametrize("parts", [0, 2])
@pytest.mark.parametrize("some", [None, [2, 0]])
def test_norms_of_no_channels(parts, some):
    from llm_d_inference_scheduler_amd import ops
    x = torch.empty(*[parts] * (parts > 0), 3, 0, device="cuda")
    x, gain = x if parts else x.bfloat16(), torch.empty(0, device="cuda").bfloat16()
    some = None if some is None else torch.tensor(some, device="cuda")
    for residual in (None, torch.empty(3, 0, device="cuda").bfloat16()):
        with pytest.raises(RuntimeError, match="no channels"):
            ops.rmsnorm(x, gain, 1e-5, residual, some)
    if some is not None and not parts:
        with pytest.raises(RuntimeError):
            ops.embed_rmsnorm(some, x, gain, 1e-5)


@pytest.mark.parametrize("parts", [0, 1, 8])
@pytest.mark.parametrize("rows,width", [(1, 8), (5, 2056), (300, 4096), (3, 4104),
                                        (600, 1024), (2, 16400), (2, 32776)])
def test_norms_of_some_rows(rows, width, parts):
    """The rows asked for, twice or from the end, as they come out among all; of a
    table, its rows and their norms. All the same bits: threads, sums and rounding are
    the same."""
    from llm_d_inference_scheduler_amd import ops
    x = _draw(max(parts, 1), rows, width, seed=rows)
    x = x.float() if parts else x[0]
    gain, start = _draw(width, seed=3), _draw(rows, width, seed=4)
    some = torch.tensor([rows - 1, 0, -1, rows // 2, 0], device="cuda")
    for residual in (None, start):
        want = ops.rmsnorm(x, gain, 1e-5,
                           None if residual is None else residual.clone())
        got = ops.rmsnorm(x, gain, 1e-5, residual, some)
        assert torch.equal(got, want[some])
        assert ops.rmsnorm(x, gain, 1e-5, residual, some[:0]).shape == (0, width)
    assert torch.equal(start, _draw(rows, width, seed=4))
    if not parts:
        rows_of, normed = ops.embed_rmsnorm(some, x, gain, 1e-5)
        assert torch.equal(rows_of, x[some])
        assert torch.equal(normed, ops.rmsnorm(x[some], gain, 1e-5))


@pytest.mark.parametrize("parts", [0, 3])
@pytest.mark.parametrize("rows,width", [(1, 8), (7, 2056), (3, 4104), (2, 32776)])
def test_norms_of_rows_that_do_not_exist(rows, width, parts):
    """They are no other row's, whatever stands beside the first and the last."""
    from llm_d_inference_scheduler_amd import ops
    x = _draw(max(parts, 1), rows, width, seed=rows)
    x = x.float() if parts else x[0]
    gain, start = _draw(width, seed=3), _draw(rows, width, seed=4)
    some = torch.tensor([0, rows, -rows - 1, rows - 1, 1 << 40, -(1 << 40), -rows],
                        device="cuda")
    there = torch.tensor([0, 3, 6], device="cuda")
    gone = torch.tensor([1, 2, 4, 5], device="cuda")
    for residual in (None, start):
        got = ops.rmsnorm(x, gain, 1e-5, residual, some)
        want = ops.rmsnorm(x, gain, 1e-5, residual, some[there])
        assert torch.equal(got[there], want) and got[gone].isnan().all()
    assert torch.equal(start, _draw(rows, width, seed=4))
    if not parts:
        for got, want in zip(ops.embed_rmsnorm(some, x, gain, 1e-5),
                             ops.embed_rmsnorm(some[there], x, gain, 1e-5)):
            assert torch.equal(got[there], want) and got[gone].isnan().all()


@pytest.mark.parametrize("width", [8, 1032, 2040, 2048])
@pytest.mark.parametrize("rows", [1, 300])
def test_norm_of_one_part(rows, width):
    """Rows of up to 256 vectors have 256 threads in parts too: to the bit what rows in
    bf16 come out as."""
    hip = _ext("_hip_ops")
    x, gain, start = (_draw(rows, width, seed=2), _draw(width, seed=3),
                      _draw(rows, width, seed=4))
    for residual in (None, start):
        a, b = (None if residual is None else residual.clone() for _ in range(2))
        assert torch.equal(hip.rmsnorm(x.float()[None], gain, 1e-5, a),
                           hip.rmsnorm(x, gain, 1e-5, b))
        assert residual is None or torch.equal(a, b)


@pytest.mark.parametrize("width", [1032, 2056, 4104, 8200])
@pytest.mark.parametrize("few,many,parts", [(256, 257, 9), (512, 513, 2)])
def test_norms_of_parts_of_many_rows(few, many, parts, width):
    """A row comes out alike whichever way its parts are asked for: the same bits; of
    the 32-bit stream, whose two forms join multiplications and additions otherwise,
    32-bit sums within 1e-5 as above, and one step of bf16 in what follows."""
    from llm_d_inference_scheduler_amd.ops import layered
    hip = _ext("_hip_ops")
    y = _draw(parts, many, width, seed=width).float()
    gain, start = _draw(width, seed=3), _draw(many, width, seed=4)
    outs = []
    for n in (few, many):
        mine, residual, x, z = y[:, :n].contiguous(), start[:n].clone(), *(
            start[:n].float() for _ in range(2))
        outs.append([hip.rmsnorm(mine, gain, 1e-5),
                     hip.rmsnorm(mine, gain, 1e-5, residual), residual,
                     layered.stream_norm(x, mine, gain.float(), gain.float(),
                                         0.5, 1e-5, torch.bfloat16), x,
                     layered.stream_norm(z, mine, None, gain.float(), 0.5,
                                         1e-5, torch.bfloat16), z])
    for i, (a, b) in enumerate(zip(*outs)):
        if i < 3:
            assert torch.equal(a, b[:few])
        elif a.dtype == torch.float32:
            torch.testing.assert_close(a, b[:few], rtol=1e-5, atol=1e-5)
        else:
            _same(a, b[:few].double(), 7)
        assert b[few:].isfinite().all() and b[few:].any()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("T,qh,kvh,d,bs", [(1, 4, 1, 128, 16),
                                           (37, 8, 8, 64, 16),
                                           (130, 6, 2, 32, 8),
                                           (5, 2, 1, 16, 4),
                                           (3, 3, 3, 96, 16)])
@pytest.mark.parametrize("parts", [0, 3])
def test_rope_and_cache(T, qh, kvh, d, bs, norm, fp8, parts):
    """One pass against its steps apart in float64; a slot below 0 is not
    cached; 96 channels have no normed form and go step by step."""
    from llm_d_inference_scheduler_amd import ops
    from llm_d_inference_scheduler_amd.ops import ref
    n = (qh + 2 * kvh) * d
    if parts:
        qkv = _draw(parts, T, n, seed=T).float() / 2
        x = qkv.double().sum(0)
    else:
        qkv = _draw(T, n, seed=T)
        x = qkv.double()
    pos = torch.randint(0, 300, (T,), device="cuda", dtype=torch.int32)
    cs = ref.rope_table(300, d, 1e4, device="cuda")
    blocks = T // bs + 2
    slots = torch.randperm(blocks * bs, device="cuda")[:T]
    slots[T // 2] = -1
    dtype = torch.float8_e4m3fn if fp8 else torch.bfloat16
    kc, vc = (torch.zeros(blocks, kvh, bs, d, device="cuda").to(dtype)
              for _ in range(2))
    qn, kn = (_draw(d, seed=7), _draw(d, seed=8)) if norm else (None, None)
    got = ops.rope_and_cache(qkv, qh, cs, pos, kc, vc, slots, qn, kn, 1e-5)
    q, k, v = (t.reshape(T, -1, d) for t in x.split(
        [qh * d, kvh * d, kvh * d], -1))
    if norm:
        q, k = (t * (t.square().mean(-1, keepdim=True) + 1e-5).rsqrt() *
                w.double() for t, w in ((q, qn), (k, kn)))
    c, s = (cs.double()[pos.long()][:, None, :, i] for i in (0, 1))

    def rotate(t):
        a, b = t[..., :d // 2], t[..., d // 2:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)
    # bf16, and the steps apart round twice; fp8: half a step of 2^-3
    torch.testing.assert_close(got.double(), rotate(q), rtol=2 ** -6,
                               atol=2e-2)
    keep = slots >= 0
    for cache, want in ((kc, rotate(k)), (vc, v)):
        rows = cache.float().permute(0, 2, 1, 3).reshape(-1, kvh, d)
        torch.testing.assert_close(
            rows[slots[keep]].double(), want[keep],
            rtol=2 ** -3.5 if fp8 else 2 ** -6, atol=2e-2)
        rows[slots[keep]] = 0
        assert not rows.any()            # nothing else was written


@pytest.mark.parametrize("n,k", [(4096, 4096), (264, 1000), (30000, 200),
                                 (60008, 136)])
def test_rows_come_out_alike(n, k):
    """One row alone and the same row among up to 256 give the same bits where K is in
    parts for the caller to sum, and in gated products of whole blocks. Not so where K is
    shared out inside a workgroup or parts are summed here (linear, linear32, an
    activation, narrow gated products): there the shares hang on the number of rows."""
    ext = _ext("_hip_ops")
    x, w = _draw(256, k, seed=1), _draw(n, k, seed=2, scale=k ** -0.5)
    one = ext.linear_parts(x[:1], w)
    for rows in (16, 17, 64, 100, 128, 192, 256):
        if ext.few_rows(x[:rows], w) or one.dim() == 3:
            y = ext.linear_parts(x[:rows], w)
            assert torch.equal(y[..., :1, :], one), rows
    if n % 2 == 0 and n >= 30000:
        one = ext.gated_linear(x[:1], w, 1)
        for rows in (16, 17, 128):
            y = ext.gated_linear(x[:rows], w, 1)
            assert (y is None) == (one is None)
            assert y is None or torch.equal(y[:1], one)


def test_rows_of_a_table_that_is_a_view():
    """As an index takes them."""
    from llm_d_inference_scheduler_amd import ops
    table, gain = _draw(50, 64)[::2, :40], _draw(40, seed=3)
    ids = torch.tensor([24, 0, -1], device="cuda")
    for some in (ids, ids.int(), ids.repeat(2)[::2]):
        rows, normed = ops.embed_rmsnorm(some, table, gain, 1e-5)
        assert torch.equal(rows, table[some])
        assert torch.equal(normed, ops.rmsnorm(table[some], gain, 1e-5))
