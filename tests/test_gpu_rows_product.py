"""Products of few rows (csrc/rows_product.hip) against f64: every kernel form at the edges of its tiles, remainders of the
depth and of the columns, strided rows, biases, f32 parts and the norms that read them, gated products, also of many rows
(csrc/gated_product.hip)."""

import pytest
import torch

from skyrl_amd.inference_engines import layer_kernels as lk

pytestmark = pytest.mark.gpu

# rows on both sides of every form's limit; columns: scalar tail, one tile, wide tiles with a remainder; depths below a
# piece, with a remainder, with unequal shares
SHAPES = [(1, 17, 8), (1, 203, 2072), (1, 8200, 520), (2, 16, 64), (3, 203, 72), (16, 40, 1000), (16, 8200, 136),
          (17, 50, 328), (32, 8192, 64), (33, 24, 712), (48, 96, 2048), (64, 8216, 200), (64, 1000, 1544), (65, 64, 264),
          (128, 4096, 72), (100, 136, 1088)]


def _data(dev, n, N, K, seed, pad=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(n, K + pad, device=dev, generator=g).bfloat16()[:, :K]
    w = torch.randn(N, K + pad, device=dev, generator=g).bfloat16()[:, :K]
    b = torch.randn(N, device=dev, generator=g).bfloat16()
    return x, w, b


def _bounds(x, w):
    """The exact product and what f32 sums of its exact terms, in any order, may be off by."""
    y = x.double() @ w.double().t()
    return y, x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 1e-30


@pytest.mark.parametrize("n,N,K", SHAPES)
@pytest.mark.parametrize("pad", (0, 24))
def test_products(dev, n, N, K, pad):
    x, w, b = _data(dev, n, N, K, n + N, pad)
    assert lk._rows_fit(x, w, parts=True) and lk._rows_fit(x, w) == (n <= 64)
    ref, off = _bounds(x, w)
    for bias in (None, b):
        want = ref if bias is None else ref + bias.double()
        y = lk.linear(x, w, bias)
        assert y.dtype == torch.bfloat16 and bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2 * off).all())
        parts = lk.linear(x, w, bias, parts=True)
        assert parts.dtype == torch.float32 and parts.shape[1:] == (n, N)
        assert bool(((lk.joined(parts).double() - want).abs() <= 2 * off + 2.0 ** -21 * want.abs()).all())


@pytest.mark.parametrize("act", ("silu", "gelu_tanh", "clamped"))
@pytest.mark.parametrize("n,N,K", [(1, 100, 264), (2, 8, 64), (16, 4100, 136), (17, 36, 200), (32, 72, 1032), (33, 132, 520),
                                   (64, 6144, 72), (513, 12288, 64), (1030, 6144, 192), (8200, 896, 128), (5000, 5120, 64)])
def test_gated(dev, n, N, K, act):
    x, w, _ = _data(dev, n, 2 * N, K, 5 * n)
    y = lk.gated_linear(x, w, act, 1.702, 7.0)
    z, off = _bounds(x, w)
    g, u = z[:, :N], z[:, N:]
    if act == "silu":
        ref = g * torch.sigmoid(g) * u
    elif act == "gelu_tanh":
        ref = torch.nn.functional.gelu(g, approximate="tanh") * u
    else:
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
        ref = g * torch.sigmoid(1.702 * g) * (u + 1)
    slack = 1.2 * off[:, :N] * (u.abs() + 1) + (g.abs() + 1) * off[:, N:]  # the gates' slopes are at most 1.2
    assert bool(((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2 * slack + 1e-5 * (g * u).abs() + 1e-6).all())


@pytest.mark.parametrize("n,N,K", [(65, 4096, 64), (128, 6144, 2048), (129, 4096, 256), (256, 8960, 320), (511, 4608, 384), (448, 4608, 1536)])
def test_gated_small_tiles(dev, n, N, K):
    """Tiles of 64 rows: one stage an item, fewer than are under way and more, items on their own and several a workgroup."""
    assert lk._ffi.query("skyrl_gated_product_fits", n, K, N)
    test_gated(dev, n, N, K, "silu")
    test_gated(dev, n, N, K, "gelu_tanh")


@pytest.mark.parametrize("n,N,K", [(128, 6144, 2048), (192, 4608, 1536), (256, 8960, 768), (448, 4608, 1536)])
def test_gated_rows_of_equal_tiles(dev, n, N, K):
    """A row has the same bits in every tile of 64 of its call, whichever of the tiles' items are halved."""
    x, w, _ = _data(dev, 64, 2 * N, K, n)
    assert lk._ffi.query("skyrl_gated_product_fits", n, K, N)
    y = lk.gated_linear(x.repeat(n // 64, 1), w, "silu").view(n // 64, 64, N)
    assert bool((y == y[0]).all())


@pytest.mark.parametrize("N", [4096, 4100, 8192, 8196, 12288, 12292, 16384, 16388])
@pytest.mark.parametrize("n,K", [(16, 264), (17, 136), (32, 520), (33, 264), (64, 1032)])
def test_rows_of_weights_a_workgroup(dev, n, N, K):
    """Both sides of each number of weight rows a workgroup, 16 to 64: rounded, capped, and gated pairs of as many rows."""
    test_products(dev, n, N, K, 24)
    test_gated(dev, n, N // 2, K, "silu")
    x, w, _ = _data(dev, n, N, K, n, 24)
    y = lk.linear(x, w).float()
    assert torch.allclose(lk.capped_linear(x, w, 3.0), 3.0 * torch.tanh(y / 3.0), rtol=2e-6, atol=1e-6)  # of the rounded product, in f32


@pytest.mark.parametrize("n,N,K", [(2113, 4096, 64), (2300, 6400, 128), (2113, 4096, 192), (2300, 6400, 256), (4161, 3968, 320)])
def test_gated_in_rounds(dev, n, N, K):
    """One to five stages an item, a second round of whole items and one of halves, a last tile of 65, 252 and 65 rows."""
    test_gated(dev, n, N, K, "silu")


@pytest.mark.parametrize("n,N,K", [(65, 40, 64), (129, 1000, 192), (200, 2040, 1088),            # tiles of 64 x 32
                                   (65, 8000, 64), (130, 5000, 320),                             # 64 x 64
                                   (300, 5000, 64), (700, 3400, 256), (65, 16384, 128),          # 64 x 128
                                   (300, 9000, 64), (1000, 4104, 192),                           # 128 x 128
                                   (2100, 520, 64), (1537, 5000, 640), (3000, 5000, 128), (3073, 6152, 192), (8200, 1032, 320)])  # 192, 256 rows
@pytest.mark.parametrize("pad", (0, 24))
def test_dense(dev, n, N, K, pad):
    """Many rows: one stage and several, more stages than are under way, the last tile's rows and columns."""
    x, w, _ = _data(dev, n, N, K, n + N, pad)
    ref, off = _bounds(x, w)
    for _ in range(2):
        y = lk._dense(x, w)
        assert y.shape == (n, N) and bool(((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2 * off).all())


@pytest.mark.parametrize("n,N,K", [(2560, 12352, 320), (4096, 6272, 512), (3072, 9224, 256)])
def test_dense_items_past_the_last_column(dev, n, N, K):
    """Full tiles of 256 rows in several rounds, whose last columns leave waves of an item without a store: the same bits every time."""
    x, w, _ = _data(dev, n, N, K, n + N)
    ref, off = _bounds(x, w)
    y = lk._dense(x, w)
    assert bool(((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2 * off).all())
    assert all(torch.equal(lk._dense(x, w), y) for _ in range(3))


@pytest.mark.parametrize("n,N,K", [(65, 28672, 64), (100, 28680, 320), (128, 30000, 256), (129, 28672, 512), (256, 66056, 128), (200, 28680, 768)])
def test_dense_one_tile_of_rows(dev, n, N, K):
    """One tile of 128 or 256 rows, halves of items and whole ones, depths with a start for each column and without."""
    test_dense(dev, n, N, K, 24)
    x, w, _ = _data(dev, n, N, K, n)
    assert lk._dense_fit(x, w) and torch.equal(lk._dense(x, w), lk._dense(x, w))


def test_many_rows_take_the_faster_form(dev):
    for n, N, K, own in ((65, 2048, 2048, True), (256, 2048, 2048, True), (256, 3408, 2048, True), (1024, 12352, 2048, True), (5637, 12352, 2048, True),
                         (5637, 3072, 768, True), (2048, 5824, 512, True), (1563, 2048, 2048, True), (3000, 2048, 2048, False), (8192, 2048, 2048, False),
                         (8192, 2048, 6144, False), (256, 32768, 2048, True), (300, 4096, 12288, False), (300, 2044, 2048, False),
                         (300, 2048, 2056, False)):
        x, w, b = _data(dev, n, N, K, 0)
        assert lk._dense_fit(x, w) == own, (n, N, K)
        assert not lk._dense_fit(x[:64], w) and not lk._dense_fit(x.float(), w.float())
        ref = torch.nn.functional.linear(x, w)
        y = lk.linear(x, w)
        assert float((y.float() - ref.float()).norm()) <= 1e-3 * float(ref.float().norm())  # the same rounding but where a sum's order differs
        assert torch.equal(lk.linear(x, w, b), torch.nn.functional.linear(x, w, b))
    x, w, _ = _data(dev, 256, 2048, 2048, 0, 4)
    assert not lk._dense_fit(x, w)  # row strides of 2052
    assert torch.equal(lk.linear(x, w), torch.nn.functional.linear(x, w))


@pytest.mark.parametrize("n,N,K", [(65, 2048, 512), (300, 2048, 2048), (5637, 3072, 768)])
def test_many_rows_that_need_gradients(dev, n, N, K):
    """The library's product, which has them, also where ours is the faster one."""
    x, w, _ = _data(dev, n, N, K, n)
    assert lk._dense_fit(x, w)
    dy = torch.randn(n, N, device=dev).bfloat16()
    for of_x, of_w in ((True, False), (False, True), (True, True)):
        got, want = [], []
        for f, to in ((lk.linear, got), (torch.nn.functional.linear, want)):
            a, b = x.clone().requires_grad_(of_x), w.clone().requires_grad_(of_w)
            y = f(a, b)
            y.backward(dy)
            to += [y, a.grad, b.grad]
        assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(got, want))
        with torch.no_grad():
            assert not lk.linear(x.clone().requires_grad_(of_x), w.clone().requires_grad_(of_w)).requires_grad


@pytest.mark.filterwarnings("ignore::DeprecationWarning")
def test_many_rows_that_are_transformed(dev):
    """Mapped, forward-differentiated and traced products are the library's too."""
    x, w, _ = _data(dev, 300, 2048, 512, 0)
    assert lk._dense_fit(x, w)
    taken = []
    for f in (torch.func.vmap, lambda f: lambda a: torch.func.jvp(f, (a,), (a,)), torch.func.grad):
        f(lambda a: taken.append(lk._dense_fit(a[0] if a.dim() == 3 else a, w)) or a.float().sum())(x.expand(2, 300, 512).contiguous())
    assert taken == [False] * 3
    with torch.autograd.forward_ad.dual_level():
        y = torch.autograd.forward_ad.unpack_dual(lk.linear(torch.autograd.forward_ad.make_dual(x, 2 * x), w))
    want = torch.nn.functional.linear(x, w)
    assert torch.equal(y.primal, want) and torch.equal(y.tangent, 2 * want)
    f = torch.jit.trace(lambda a: lk.linear(a, w), x)
    assert torch.equal(f(2 * x), 2 * want)


def test_what_the_library_takes(dev):
    x, w, _ = _data(dev, 129, 64, 64, 0)
    assert not lk._rows_fit(x, w)                                  # too many rows
    assert not lk._rows_fit(*_data(dev, 65, 4104, 64, 0)[:2])
    assert not lk._rows_fit(*_data(dev, 4, 64, 60, 0)[:2])         # depth no multiple of 8
    big = torch.randn(4, 132, device=dev).bfloat16()
    assert not lk._rows_fit(big[:, 1:65], w)                       # misaligned rows
    assert not lk._rows_fit(big[:, :64], w)                        # and row strides
    assert not lk._rows_fit(x[:4].float(), w.float())
    assert lk.gated_linear(x[:65], w, "silu") is None
    for n, N, K in ((511, 12288, 64), (1024, 5888, 64), (1024, 6208, 64), (1024, 6144, 72)):  # few rows, few items, remainders
        assert lk.gated_linear(*_data(dev, n, 2 * N, K, 0)[:2], "silu") is None
    # depths above 2048 where the library is the faster one: (rows, N, K, rounded, parts, gated of N / 2)
    for n, N, K, rounded, parts, gated in ((1, 4096, 4096, 1, 1, 1), (1, 4096, 8192, 0, 0, 0), (16, 2048, 6144, 1, 1, 1),
                                           (16, 2048, 8192, 0, 1, 0), (32, 8192, 4096, 0, 1, 0), (33, 4096, 4096, 1, 1, 1),
                                           (33, 4096, 12288, 0, 1, 0), (32, 8208, 4096, 1, 1, 1), (33, 8208, 4096, 0, 0, 0),
                                           (32, 8208, 3072, 0, 0, 0), (64, 32768, 2048, 1, 1, 1), (128, 2048, 2048, 0, 1, 0),
                                           (1, 4096, 16384, 0, 0, 0), (64, 4096, 18432, 1, 1, 1)):
        got = [bool(lk._ffi.query("skyrl_rows_product_fits", n, K, m, f)) for m, f in ((N, 0), (N, 2), (N // 2, 1))]
        assert got == [bool(rounded), bool(parts), bool(gated)], (n, N, K)
    for a, b in ((big[:, 1:65], w), (x, w), (x[:4].float(), w.float())):
        torch.testing.assert_close(lk.linear(a, b, parts=True), torch.nn.functional.linear(a, b))
    with pytest.raises(ValueError):
        lk.linear(x[:4], torch.zeros(8, 72, device=dev, dtype=torch.bfloat16))


@pytest.mark.parametrize("n,H", [(1, 40), (3, 203), (16, 2048), (64, 1536), (70, 4096)])
@pytest.mark.parametrize("parts", (1, 2, 3, 4, 8))
def test_norms_of_parts(dev, n, H, parts):
    g = torch.Generator(device=dev).manual_seed(parts)
    r = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
    d, h = r(parts, n, H), r(n, H)
    w, step, nxt, b = r(H).bfloat16(), r(H).bfloat16(), r(H).bfloat16(), r(H)
    full = h.double() + d.double().sum(0) + step.double()
    got = h.clone()
    y = lk.add_norm(d, got, w, 1e-6, "layer", step=step)
    c = full - full.mean(1, keepdim=True)
    torch.testing.assert_close(got.double(), full, atol=4e-6, rtol=1e-6)
    torch.testing.assert_close(y.double(), c / c.square().mean(1, keepdim=True).add(1e-6).sqrt() * w.double(), atol=1e-4, rtol=2 ** -8)
    for groups in (1, 4):
        if H % groups:
            continue
        norm = lambda v: (v.view(n, groups, -1) / v.view(n, groups, -1).square().mean(-1, keepdim=True).add(1e-6).sqrt()).view(n, H)  # noqa: E731
        z = r(n, H).bfloat16()
        full = h.double() + 0.5 * norm(d.double().sum(0) * torch.sigmoid(z.double() + b.double())) * w.double()
        got = h.clone()
        y = lk.gate_norm_add(d, got, w, nxt, 1e-6, groups=groups, mult=0.5, gate=z, gate_bias=b)
        torch.testing.assert_close(got.double(), full, atol=2e-5, rtol=1e-5)
        torch.testing.assert_close(y.double(), norm(full) * nxt.double(), atol=1e-4, rtol=2 ** -8)


@pytest.mark.parametrize("H,groups", [(2048, 256), (2048, 128), (2048, 64), (2048, 32), (2048, 16), (2048, 8), (2048, 4), (1536, 4), (4096, 2)])
def test_norms_in_parts_of_any_size(dev, H, groups):
    """Sums over 1, 2, 4, .. 64 neighbouring lanes, and over several such."""
    g = torch.Generator(device=dev).manual_seed(groups)
    r = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
    n = 5
    a, z, h, w, nxt, b = r(2 * n, H).bfloat16(), r(n, H).bfloat16(), r(n, H), r(H).bfloat16(), r(H).bfloat16(), r(H)
    norm = lambda v: (v.view(n, groups, -1) / v.view(n, groups, -1).square().mean(-1, keepdim=True).add(1e-6).sqrt()).view(n, H)  # noqa: E731
    full = h.double() + 0.5 * norm(a.double().view(n, 2, H).sum(1) * torch.sigmoid(z.double() + b.double())) * w.double()
    got = h.clone()
    y = lk.gate_norm_add(a, got, w, nxt, 1e-6, groups=groups, mult=0.5, parts=2, gate=z, gate_bias=b)
    torch.testing.assert_close(got.double(), full, atol=2e-5, rtol=1e-5)
    torch.testing.assert_close(y.double(), norm(full) * nxt.double(), atol=1e-4, rtol=2 ** -8)


@pytest.mark.parametrize("B,n,N,K", [(16, 1, 512, 128), (3, 2, 40, 24), (5, 17, 130, 264), (2, 33, 24, 136), (4, 64, 128, 512),
                                     (3, 65, 50, 200), (2, 200, 72, 328), (1, 256, 16, 64)])
def test_batch(dev, B, n, N, K):
    g = torch.Generator(device=dev).manual_seed(B + n)
    x = torch.randn(n, B, K + 8, device=dev, generator=g).bfloat16()[:, :, :K].transpose(0, 1)  # heads side by side in a row
    w = torch.randn(B, N, K, device=dev, generator=g).bfloat16()
    out = torch.full((n, B, N), float("nan"), device=dev, dtype=torch.bfloat16).transpose(0, 1)
    assert lk.rows_batch(x, w, out)
    for b in range(B):
        ref, off = _bounds(x[b], w[b])
        assert bool(((out[b].double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2 * off).all())
    assert not lk.rows_batch(x[:, :, 1:], w[:, :, 1:].contiguous(), out)  # a depth and rows that are not 16-byte pieces
    assert not lk.rows_batch(x.float(), w.float(), out.float())


@pytest.mark.parametrize("B,D,C", [(16, 128, 512), (12, 128, 512), (32, 128, 512), (8, 64, 256), (16, 96, 384)])
@pytest.mark.parametrize("n", [33, 48, 64, 65, 100, 191, 256])
def test_batch_in_order_is_the_librarys(dev, B, n, D, C):
    """Both up-projections of latent attention, from and to heads side by side in a row, bit for bit torch.bmm's."""
    g = torch.Generator(device=dev).manual_seed(B + n)
    q = torch.randn(n, B, D + 64, device=dev, generator=g).bfloat16()[:, :, :D].transpose(0, 1)
    for x, K, N in ((q, D, C), (torch.randn(B, n, C, device=dev, generator=g).bfloat16(), C, D)):
        w = (torch.randn(B, K, N, device=dev, generator=g) * 0.05).bfloat16()
        out = torch.full((n, B, N), float("nan"), device=dev, dtype=torch.bfloat16).transpose(0, 1)
        assert lk.rows_batch(x, w.transpose(1, 2).contiguous(), out, in_order=True)
        assert torch.equal(out, torch.bmm(x, w))


@pytest.mark.parametrize("n,N,K", [(33, 72, 328), (64, 130, 264), (200, 50, 72), (256, 24, 136), (100, 40, 512), (40, 16, 8)])
def test_batch_in_order(dev, n, N, K):
    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.randn(n, 3, K + 8, device=dev, generator=g).bfloat16()[:, :, :K].transpose(0, 1)
    w = torch.randn(3, N, K, device=dev, generator=g).bfloat16()
    out = torch.full((n, 3, N), float("nan"), device=dev, dtype=torch.bfloat16).transpose(0, 1)
    assert lk.rows_batch(x, w, out, in_order=True)
    for b in range(3):
        ref, off = _bounds(x[b], w[b])
        assert bool(((out[b].double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2 * off).all())
    assert not lk.rows_batch(x[:, :32], w, out[:, :32], in_order=True)
    big = torch.zeros(3, n, 520, device=dev, dtype=torch.bfloat16)
    assert not lk.rows_batch(big, torch.zeros(3, N, 520, device=dev, dtype=torch.bfloat16), out, in_order=True)


# n, columns, depth; what the form has: waves along the depth, slots of each wave's ring
DEEP = {"rounded": [(16, 3650, 2056, 4, 4), (20, 3650, 2056, 4, 3), (64, 3650, 2056, 4, 2),
                    (16, 8200, 2056, 4, 2), (32, 8200, 2040, 4, 2), (50, 8200, 2040, 2, 2), (1, 3650, 2056, 4, 4), (1, 8200, 2056, 4, 2),
                    (16, 8192, 2056, 4, 4), (16, 16392, 2056, 4, 2), (1, 16392, 2056, 4, 2)],
        "parts": [(16, 4104, 2056, 4, 4), (11, 2048, 6152, 4, 4), (32, 2050, 6152, 4, 2), (64, 2056, 6152, 4, 2), (100, 2056, 6152, 4, 1), (1, 2056, 6152, 4, 4)],
        "gated": [(16, 2056, 2040, 4, 2), (32, 2056, 2040, 4, 2), (64, 2056, 2040, 2, 2), (1, 2056, 2040, 2, 4), (64, 2056, 2040, 4, 2),
                  (16, 2056, 2040, 4, 3), (16, 4104, 2040, 2, 4), (1, 8192, 2040, 2, 4), (5, 8200, 2040, 4, 3), (9, 4104, 3080, 4, 3),
                  (40, 8200, 2040, 2, 2), (64, 16392, 2040, 4, 2)],
        "batch": [(16, 40, 1096, 4, 2), (32, 72, 1096, 4, 2), (100, 24, 1096, 4, 2)]}


@pytest.mark.parametrize("form,n,N,K,waves,slots", [(f, *s) for f, shapes in DEEP.items() for s in shapes])
def test_rings_are_refilled(dev, form, n, N, K, waves, slots):
    """Every wave's share goes round its ring of slots, with a remainder at the end; over and over, since a slot that is
    overwritten while it is read need not show at once."""
    x, w, _ = _data(dev, n, 2 * N if form == "gated" else N, K, n + K)
    shares = waves * (int(lk._ffi.query("skyrl_rows_product_splits", n, K, N)) if form == "parts" else 1)
    assert -(-K // 64) // shares >= slots + 2 and K % 64
    z, off = _bounds(x, w)
    if form == "batch":
        out = torch.empty(3, n, N, device=dev, dtype=torch.bfloat16)
        run = lambda: (lk.rows_batch(x.expand(3, n, K).contiguous(), w.expand(3, N, K).contiguous(), out.zero_()), out.clone())  # noqa: E731
        outs = [run() for _ in range(4)]
        assert all(took for took, _ in outs)
        outs = [y for _, y in outs]
    else:
        run = {"rounded": lambda: lk.linear(x, w), "parts": lambda: lk.linear(x, w, parts=True),
               "gated": lambda: lk.gated_linear(x, w, "silu")}[form]
        assert lk._rows_fit(x, w, gated=form == "gated", parts=form == "parts")
        outs = [run() for _ in range(4)]
    assert all(torch.equal(outs[0], y) for y in outs[1:])
    y = outs[0].double()
    if form == "gated":
        g, u = z[:, :N], z[:, N:]
        z, off = g * torch.sigmoid(g) * u, 1.2 * off[:, :N] * (u.abs() + 1) + (g.abs() + 1) * off[:, N:]
    if form == "parts":
        assert bool(((y.sum(0) - z).abs() <= 2 * off + 2.0 ** -21 * z.abs()).all())
    else:
        assert bool(((y - z).abs() <= 2.0 ** -8 * z.abs() + 2 * off + 1e-5).all())


@pytest.mark.parametrize("form,n,N", [("rounded", 33, 5000), ("rounded", 50, 8200), ("rounded", 64, 12296), ("rounded", 32, 8200), ("rounded", 17, 5000),
                                      ("rounded", 9, 12288), ("gated", 33, 4096), ("gated", 64, 6144), ("gated", 20, 2056), ("gated", 32, 6144),
                                      ("gated", 16, 6144)])
def test_rings_of_other_widths_are_refilled(dev, form, n, N):
    test_rings_are_refilled(dev, form, n, N, 2040, 4, 3 if form == "gated" and n <= 16 else 2)


@pytest.mark.parametrize("pairs", [100, 6144, 6148])
def test_gated_of_a_normed_row(dev, pairs):
    """Both sides of the number of weight rows a workgroup: the product of the norm's row, launched alone."""
    g = torch.Generator(device=dev).manual_seed(pairs)
    r = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
    w = (r(2 * pairs, 2048) * 0.02).bfloat16()
    delta, h, weight = r(4, 1, 2048), r(1, 2048), r(2048).bfloat16()
    rows = [lk.normed(delta, h, weight, 1e-5) for _ in range(3)]  # h is read: the residual leaves in another buffer
    y = [lk.gated_linear(row, w, "silu") for row in rows]
    row = rows[0]
    x = lk.rows_of(row)
    z, off = _bounds(x, w)
    a, u = z[:, :pairs], z[:, pairs:]
    slack = 1.2 * off[:, :pairs] * (u.abs() + 1) + (a.abs() + 1) * off[:, pairs:]
    assert all(torch.equal(y[0], t) for t in y) and bool(((y[0].double() - a * torch.sigmoid(a) * u).abs() <= 2.0 ** -8 * (a * u).abs() + 2 * slack + 1e-5).all())


def _close(y, x, w, want=None):
    ref, off = _bounds(x, w)
    want = ref if want is None else want
    y = lk.joined(y).double()
    return bool(((y - want).abs() <= 2.0 ** -8 * want.abs() + 2 * off).all())


@pytest.mark.parametrize("N,K", [(2048, 2048), (1536, 4608), (4096, 4096), (2048, 6144), (4096, 6144), (24, 2056)])
def test_shares_of_one_row_keep_their_bits(dev, N, K):
    """f32 shares of one row against 64 bits: within two roundings of the result (2^-23 in the 2-norm), at any depth; f32 sums along a
    wave's share of 1024 are off by three."""
    x, w, _ = _data(dev, 1, N, K, N + K)
    y = lk.linear(x, w, parts=True)
    ref = x.double() @ w.double().t()
    assert y.dim() == 3 and float((y.double().sum(0) - ref).norm()) <= 2.0 ** -23 * float(ref.norm())
    if K <= 4096:
        g = torch.Generator(device=dev).manual_seed(K)
        r = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
        row = lk.gate_normed(r(2, 1, K), r(1, K), r(K).bfloat16(), r(K).bfloat16(), 1e-6, gate=r(1, K).bfloat16(), gate_bias=r(K))
        y = lk.linear(row, w, parts=True)
        ref = lk.rows_of(row).double() @ w.double().t()
        assert row.alone is None and y.dim() == 3
        assert float((y.double().sum(0) - ref).norm()) <= 2.0 ** -23 * float(ref.norm())


# rows of one group of four, of a remainder of the last piece, of both register forms; wide and narrow products
@pytest.mark.parametrize("H,N", [(8, 16), (72, 203), (264, 8200), (1536, 96), (2048, 8192), (2056, 40), (4096, 12296), (4096, 24)])
@pytest.mark.parametrize("parts", (0, 1, 2, 4))
def test_norm_ahead_of_a_product(dev, H, N, parts):
    g = torch.Generator(device=dev).manual_seed(H + N + parts)
    _, w, b = _data(dev, 1, N, H, H)
    delta = torch.randn(parts, 1, H, device=dev, generator=g) if parts else None
    step = torch.randn(H, device=dev, generator=g).bfloat16() if parts % 2 == 0 else None
    weight = torch.randn(H, device=dev, generator=g).bfloat16()
    for kind, base in (("layer", 0.0), ("rms", 1.0)):
        h = torch.randn(1, H, device=dev, generator=g) + 3
        want_h = h.clone()
        want = lk.add_norm(delta, want_h, weight, 1e-3, kind, step, base=base)
        for gated in (False, True):
            before = h.clone()
            row = lk.normed(delta, before, weight, 1e-3, kind, step, base=base)
            assert isinstance(row, lk.NormedRow)
            y = lk.gated_linear(row, w, "silu") if gated and N % 2 == 0 else lk.linear(row, w, b)
            assert row.fused is None and torch.equal(before, h)  # the old residual is read by every workgroup
            assert torch.equal(lk.residual(row, before), want_h) and torch.equal(lk.rows_of(row), want)
            assert torch.equal(lk.linear(row, w, b), lk.linear(want, w, b))  # a second product: of the rows
            if gated and N % 2 == 0:
                z = want.double() @ w.double().t()
                ref = torch.nn.functional.silu(z[:, :N // 2]) * z[:, N // 2:]
                assert float((y.double() - ref).norm()) <= 2.0 ** -8 * float(ref.norm()) + 1e-6
            else:
                assert _close(y, want, w, want.double() @ w.double().t() + b.double())
    alone = lk.normed(delta, h, weight, 1e-3, "layer", step)
    want = lk.add_norm(delta, h.clone(), weight, 1e-3, "layer", step)
    assert torch.equal(lk.rows_of(alone), want)


@pytest.mark.parametrize("H,groups", [(64, 4), (1536, 4), (2048, 4), (2048, 1), (4096, 4), (4096, 2), (1048, 1), (2080, 4)])
@pytest.mark.parametrize("experts", (False, True))
def test_gate_and_norms_ahead_of_a_product(dev, H, groups, experts):
    g = torch.Generator(device=dev).manual_seed(H + groups)
    rand = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
    _, w, b = _data(dev, 1, 136, H, H)
    weight, nxt = rand(H).bfloat16(), rand(H).bfloat16()
    for parts in (1, 3) if not experts else (2, 8):
        a = rand(parts, H).bfloat16() if experts else rand(parts, 1, H)
        gate = rand(2, 1, H + 64) if experts else rand(1, H).bfloat16()
        args = dict(groups=groups, mult=0.5, parts=parts if experts else 1, gate=gate, gate_bias=rand(H))
        h = rand(1, H)
        want_h = h.clone()
        want = lk.gate_norm_add(a, want_h, weight, nxt, 1e-6, **args)
        row = lk.gate_normed(a, h, weight, nxt, 1e-6, **args)
        assert isinstance(row, lk.NormedRow)
        turn = (40, 103) if experts else None
        y = lk.linear(row, w, b, parts=not experts, turn=turn)
        assert row.fused is None
        assert torch.equal(lk.residual(row, h), want_h) and torch.equal(lk.rows_of(row), want)
        ref = lk.rows_of(row).double() @ w.double().t() + b.double()
        if experts:
            plain = lk.linear(lk.rows_of(row), w, b)
            assert torch.equal(y[:, :40], plain[:, :40]) and torch.equal(y[:, 103:], plain[:, 103:])
            assert torch.equal(y[:, 40:103], torch.tanh(plain[:, 40:103].float()).bfloat16())
        else:
            assert y.dim() == 3 and _close(y, lk.rows_of(row), w, ref)


def test_rows_that_are_normed_alone(dev):
    """More than one row, f32 models, longer rows and more shares than the joint launch takes."""
    for n, H, parts, dtype in ((2, 64, 2, torch.bfloat16), (1, 64, 0, torch.float32), (1, 4104, 1, torch.bfloat16), (1, 64, 5, torch.bfloat16)):
        h, w = torch.randn(n, H, device=dev), torch.randn(H, device=dev).to(dtype)
        delta = torch.randn(parts, n, H, device=dev) if parts else None
        want_h = h.clone()
        want = lk.add_norm(delta, want_h, w, 1e-6)
        x = lk.normed(delta, h, w, 1e-6)
        assert not isinstance(x, lk.NormedRow) and torch.equal(x, want) and torch.equal(h, want_h)


@pytest.mark.parametrize("n,N,K", [(1, 17, 8), (1, 8200, 136), (16, 203, 72), (17, 8192, 64), (33, 24, 712), (64, 8216, 200), (65, 40, 64)])
def test_what_follows_a_product(dev, n, N, K):
    """The cap of logits and the tanh of some columns are those of their own launches, bit for bit."""
    x, w, b = _data(dev, n, N, K, n + N)
    y = lk.linear(x, w)
    for cap in (30.0, None):
        assert torch.equal(lk.capped_linear(x, w, cap), lk.softcap(y, cap))
    for first, last in ((0, N), (5, 14), (N - 3, N), (7, 7)):
        if not lk.turns(x, w):
            assert n > 64
            continue
        t, plain = lk.linear(x, w, b, turn=(first, last)), lk.linear(x, w, b)
        assert torch.equal(t[:, :first], plain[:, :first]) and torch.equal(t[:, last:], plain[:, last:])
        if last > first:
            assert torch.equal(t[:, first:last], lk.tanh(plain[:, first:last]))


@pytest.mark.parametrize("H,N", [(8, 24), (264, 8200), (2048, 96), (4096, 40)])
def test_embedding_ahead_of_a_product(dev, H, N):
    g = torch.Generator(device=dev).manual_seed(H)
    rand = lambda *s: torch.randn(*s, device=dev, generator=g).bfloat16()  # noqa: E731
    table, w, weight, nxt, step = rand(50, H), rand(N, H), rand(H), rand(H), rand(H)
    for token, st in ((0, None), (49, step)):
        tok = torch.tensor([token], device=dev)
        h = lk.embed(tok, table, 1.75)
        want = lk.add_norm(None, h, weight, 1e-4, "layer", st)
        row = lk.normed_embedding(tok, table, 1.75, weight, 1e-4, "layer", st)
        y = lk.linear(row, w)
        assert row.fused is None and torch.equal(lk.residual(row, None), h) and torch.equal(lk.rows_of(row), want)
        assert _close(y, want, w)
        alone = lk.normed_embedding(tok, table, 1.75, weight, 1e-4, "layer", st)
        assert torch.equal(lk.rows_of(alone), want) and torch.equal(lk.residual(alone, None), h)
        groups = 1 if H == 8 else 4 if H > 300 else 3
        h = torch.empty(1, H, device=dev)
        want = lk.gate_norm_add(table, h, weight, nxt, 1e-6, groups, 0.5, rows=tok, fresh=True)
        for fuse in (True, False):
            row = lk.gate_normed_embedding(tok, table, weight, nxt, 1e-6, groups, 0.5)
            if fuse:
                assert _close(lk.linear(row, w), want, w)
            assert torch.equal(lk.rows_of(row), want) and torch.equal(lk.residual(row, None), h)
    assert lk.normed_embedding(torch.tensor([1, 2], device=dev), table, 1.0, weight, 1e-4) is None
