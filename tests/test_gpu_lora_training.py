"""GPU parity: the products of a trainable adapter with its activations and gradients (csrc/lora.hip) against float64 on the
same 16-bit operands, at the edges of their row chunks (16, 32), wavefronts (8 x 32 rows), column groups (32 and 64) and
ranks (padded to 16 and 32).

Tolerance: one rounding of the result (at most 2^-8 of it in bfloat16, 2^-11 in float16) and float32 sums of at most n
products of operands near 1 (n 2^-24 of the sum of magnitudes, below 2^-12 of the largest result of a row or column here)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _close(y, ref, dim):
    unit = 2.0 ** (-8 if y.dtype == torch.bfloat16 else -11)
    bound = (unit + 2.0 ** -12) * ref.abs().amax(dim=dim, keepdim=True)
    assert y.shape == ref.shape and bool(((y.double() - ref).abs() <= bound).all())


# 32 and 64 columns to a workgroup (64 where 32 make more workgroups than units), 8 and 16 rows (16 from 2049 on)
@pytest.mark.parametrize("M,K,N", [(17, 32, 64), (31, 64, 32), (32, 96, 8224), (33, 4128, 160), (255, 256, 8192), (257, 8224, 96),
                                   (520, 320, 640), (1100, 512, 12288), (2048, 96, 128), (2065, 8256, 64)])
@pytest.mark.parametrize("rank,scale,dtype", [(1, 1.0, torch.bfloat16), (6, 0.5, torch.bfloat16), (16, 1.0, torch.float16),
                                              (17, -2.0, torch.bfloat16), (32, 1.0, torch.bfloat16), (25, 0.25, torch.float16)])
def test_products_against_float64(M, K, N, rank, scale, dtype):
    from mflux_amd import _lib, lora

    ops = _lib.ops()
    gen = torch.Generator(device="cuda").manual_seed(95)
    make = lambda *shape: torch.randn(shape, generator=gen, device="cuda").to(dtype)
    a, b, x, g = make(K, rank), make(rank, N), make(M, K), make(M, N)
    R = 16 if rank <= 16 else 32
    pad = lambda t: torch.nn.functional.pad(t, (0, R - rank))
    af, bf, bs, ap = ops.low_rank_pack(a, b, scale)
    assert torch.equal(af, lora.down_fragments(pad(a))) and torch.equal(bf, lora.down_fragments(pad(b.t())))
    assert torch.equal(ap, pad(a)) and torch.equal(bs, pad((scale * b.float()).to(dtype).t()))

    def fragments(t):
        return lora.down_fragments(torch.nn.functional.pad(t, (0, 0, 0, -M % 32)))

    t, tf = ops.low_rank_forward(x, af, rank)
    _close(t[:, :rank], x.double() @ a.double(), 1)
    assert not bool(t[:, rank:].any()) and torch.equal(tf, fragments(t))
    gt, gtf, db = ops.low_rank_gradient(g, bf, tf, rank, scale, True, True)
    _close(gt[:, :rank], scale * (g.double() @ b.double().t()), 1)
    assert not bool(gt[:, rank:].any()) and torch.equal(gtf, fragments(gt))
    _close(db, scale * (t[:, :rank].double().t() @ g.double()), 1)
    _close(ops.low_rank_up(x, gtf, rank), x.double().t() @ gt[:, :rank].double(), 0)
    # each by itself: the same
    assert torch.equal(ops.low_rank_gradient(g, bf, tf, rank, scale, True, False)[0], gt)
    assert torch.equal(ops.low_rank_gradient(g, bf, tf, rank, scale, False, True)[2], db)


def test_an_infinite_row_stays_where_torch_has_it():
    """An infinity of x or of the gradient reaches the rows, columns and factors that the separate products let it reach, and
    not the columns a rank is padded by (zeros times infinity)."""
    from mflux_amd import lora, nn

    torch.manual_seed(96)
    lin = torch.nn.Linear(256, 320, bias=False, device="cuda", dtype=torch.bfloat16)
    layer = lora.LoRALinear.from_linear(nn.QuantizedLinear.from_linear(lin, 64, 4), r=4, scale=1.0)
    layer.lora_A.data.abs_()
    layer.lora_B.data.normal_(std=0.02).abs_()
    for where in ("x", "g"):
        x = torch.randn(50, 256, device="cuda").bfloat16()
        g = torch.randn(50, 320, device="cuda").bfloat16()
        (x if where == "x" else g)[33, 5] = float("inf")
        x.requires_grad_(True)
        inputs = (x, layer.lora_A, layer.lora_B)
        y = layer(x)
        got = [y, *torch.autograd.grad(y, inputs, g)]
        y = lora._composed(layer.linear, [layer], x)
        want = [y, *torch.autograd.grad(y, inputs, g)]
        for a, b in zip(got, want):
            assert torch.equal(torch.isfinite(a), torch.isfinite(b)) and torch.equal(torch.isnan(a), torch.isnan(b))


def test_gradients_that_are_not_wanted_or_not_contiguous():
    from mflux_amd import lora, nn

    torch.manual_seed(97)
    lin = torch.nn.Linear(256, 320, device="cuda", dtype=torch.bfloat16)
    layer = lora.LoRALinear.from_linear(nn.QuantizedLinear.from_linear(lin, 64, 8), r=16, scale=0.5)
    layer.lora_B.data.normal_(std=0.02)
    x = torch.randn(2, 24, 256, device="cuda").bfloat16().requires_grad_(True)
    inputs = (x, layer.lora_A, layer.lora_B)
    row = torch.randn(320, device="cuda").bfloat16()
    want = torch.autograd.grad(layer(x), inputs, row.expand(2, 24, 320).contiguous())
    for given in (row.expand(2, 24, 320), torch.cat([row.new_zeros(1), row.repeat(48)])[1:].view(2, 24, 320)):
        for a, b in zip(torch.autograd.grad(layer(x), inputs[1:], given), want[1:]):
            assert torch.equal(a, b)
    for i, one in enumerate(inputs):
        assert torch.equal(torch.autograd.grad(layer(x), one, row.expand(2, 24, 320))[0], want[i])
    frozen = x.detach()
    y = layer(frozen)
    for a, b in zip(torch.autograd.grad(y, inputs[1:], row.expand(2, 24, 320)), want[1:]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("rank", [6, 16, 32])
def test_packed_factors_are_copies(rank):
    """No output of the packing is a view of a factor, padded or not, so backward's input gradient is that of the factors
    that forward saw, also when one is written to behind autograd's back before it."""
    from mflux_amd import _lib, lora, nn

    torch.manual_seed(98)
    a, b = torch.randn(64, rank, device="cuda").bfloat16(), torch.randn(rank, 96, device="cuda").bfloat16()
    storages = {t.untyped_storage().data_ptr() for t in (a, b)}
    for t in _lib.ops().low_rank_pack(a, b, 1.0):
        assert t.untyped_storage().data_ptr() not in storages
    lin = torch.nn.Linear(256, 320, device="cuda", dtype=torch.bfloat16)
    layer = lora.LoRALinear.from_linear(nn.QuantizedLinear.from_linear(lin, 64, 4), r=rank, scale=1.0)
    layer.lora_B.data.normal_(std=0.5)
    x, g = torch.randn(40, 256, device="cuda").bfloat16().requires_grad_(True), torch.randn(40, 320, device="cuda").bfloat16()
    want, = torch.autograd.grad(layer(x), x, g)
    y = layer(x)
    layer.lora_A.data.zero_()
    layer.lora_B.data.zero_()
    assert torch.equal(torch.autograd.grad(y, x, g)[0], want)


@pytest.mark.parametrize("scale", [float("inf"), float("nan"), -3.0])
def test_a_scale_reaches_the_factor_alone(scale):
    """The columns a rank is padded by stay zero under any scale; with an infinite one they would make NaN of every output,
    where the composition has infinities."""
    from mflux_amd import _lib, lora, nn

    torch.manual_seed(99)
    a, b = torch.randn(64, 6, device="cuda").bfloat16(), torch.randn(6, 96, device="cuda").bfloat16()
    bs = _lib.ops().low_rank_pack(a, b, scale)[2]
    want = torch.nn.functional.pad((scale * b.float()).bfloat16().t(), (0, 10))
    assert torch.equal(bs.view(torch.int16)[:, 6:], torch.zeros_like(bs.view(torch.int16)[:, 6:]))
    assert torch.equal(torch.nan_to_num(bs), torch.nan_to_num(want))
    lin = torch.nn.Linear(256, 320, device="cuda", dtype=torch.bfloat16)
    layer = lora.LoRALinear.from_linear(nn.QuantizedLinear.from_linear(lin, 64, 4), r=6, scale=scale)
    layer.lora_A.data.abs_()
    layer.lora_B.data.normal_(std=0.02).abs_()
    x = torch.randn(50, 256, device="cuda").abs().bfloat16().requires_grad_(True)
    got, want = layer(x), lora._composed(layer.linear, [layer], x)
    assert torch.equal(torch.isfinite(got), torch.isfinite(want)) and torch.equal(torch.isnan(got), torch.isnan(want))
