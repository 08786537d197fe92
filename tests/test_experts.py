"""The routed experts' kernels alone, in every form an expert can have, against a plain sum over the chosen experts in float64:
the kernels for a decode step's rows, the grouped products whose operands cross LDS (sizes in whole cache lines, enough rows
an expert) and those that read their fragments from memory (other sizes, few rows an expert), with uneven choices (an expert
that everybody chose, one that nobody did), and rows of other branches added."""
import math

import pytest
import torch

gpu = pytest.mark.gpu
F64 = torch.float64
CAP = (1.3, 1.702, 1.0)


def plain_expert(form, z, ff):
    if form == "gelu":
        return 0.5 * z * (1 + torch.erf(z / math.sqrt(2.0)))
    if form == "relu_squared":
        return torch.clamp(z, min=0.0) ** 2
    g, u = z[..., :ff], z[..., ff:]
    if form == "gated_silu":
        return g * torch.sigmoid(g) * u
    limit, slope, shift = CAP
    g, u = torch.clamp(g, max=limit), torch.clamp(u, -limit, limit)
    return g * torch.sigmoid(slope * g) * (u + shift)


def plain_mixture(form, h, up, down, chosen, weight, ff):
    E, W = down.shape[0] // h.shape[1], h.shape[1]
    per = up.shape[0] // E
    out = torch.zeros(h.shape, dtype=F64)
    for e in range(E):
        for c in range(chosen.shape[1]):
            rows = (chosen[:, c] == e).nonzero().flatten()
            if rows.numel():
                z = h[rows].double() @ up[e * per:(e + 1) * per].double().T
                out[rows] += weight[rows, c, None].double() * (plain_expert(form, z, ff) @ down[e * W:(e + 1) * W].double().T)
    return out


def case(form, E, top, W, F, n, uneven, seed, dt):
    g = torch.Generator().manual_seed(seed)
    per = (2 if form in ("gated_silu", "capped_gated") else 1) * F
    up, down = (torch.randn(E * per, W, generator=g) * W ** -0.5).to(dt), (torch.randn(E * W, F, generator=g) * F ** -0.5).to(dt)
    h = torch.randn(n, W, generator=g).to(dt)
    chosen = torch.stack([torch.randperm(E - 1 if uneven and E > top else E, generator=g)[:top] for _ in range(n)]).to(torch.int32)
    if uneven:                                    # expert 0 is everybody's (once a token), the last one nobody's
        chosen = torch.where(chosen == 0, chosen[:, :1], chosen)
        chosen[:, 0] = 0
    weight = torch.rand(n, top, generator=g)
    return h, up, down, chosen, weight


@gpu
@pytest.mark.parametrize("form", ["gated_silu", "gelu", "capped_gated", "relu_squared"])
@pytest.mark.parametrize("E,top,W,F,n,uneven", [(4, 2, 64, 64, 300, False), (3, 1, 128, 192, 131, True), (8, 3, 320, 128, 400, True), (5, 5, 192, 320, 150, False),
                                                (2, 1, 64, 448, 700, False), (33, 2, 128, 64, 160, False), (6, 2, 72, 40, 200, True)])
def test_grouped_products(form, E, top, W, F, n, uneven):
    from palm_infra_amd.kernels import ops
    h, up, down, chosen, weight = case(form, E, top, W, F, n, uneven, E * n + F, torch.bfloat16)
    want = plain_mixture(form, h, up, down, chosen, weight, F)
    args = [t.cuda() for t in (h, up, down, chosen, weight)]
    got = ops.moe_grouped(*args, F, form, CAP if form == "capped_gated" else ops.NO_CAP)
    tol = 0.02 * float(want.abs().max())
    assert float((got.cpu().double() - want).abs().max()) <= tol
    y = torch.randn(n, W).to(torch.bfloat16)
    more = ops.moe_grouped(*args, F, form, CAP if form == "capped_gated" else ops.NO_CAP, add=[y.cuda()])
    assert torch.allclose(more - got, y.cuda().float(), atol=1e-4)


@gpu
@pytest.mark.parametrize("form", ["gated_silu", "relu_squared"])
@pytest.mark.parametrize("E,top,W,F,n,uneven", [(7, 3, 64, 128, 1, False), (4, 1, 1088, 64, 129, True), (3, 1, 192, 320, 200, False), (2, 2, 640, 576, 97, False),
                                                (2, 1, 128, 704, 290, True), (2, 1, 256, 64, 430, False)])
def test_grouped_tiles(form, E, top, W, F, n, uneven):
    """Tiles of 64 rows, with one stage and many, part tiles of features and of rows, and rows that start on no 16 bytes
    (which take the fragments' kernel): 32-bit sums of the same products, one rounding of the inner rows and one of the experts'."""
    from palm_infra_amd.kernels import ops
    h, up, down, chosen, weight = case(form, E, top, W, F, n, uneven, E * n + F, torch.bfloat16)
    want = plain_mixture(form, h, up, down, chosen, weight, F)
    tol = 0.02 * float(want.abs().max())
    args = [t.cuda() for t in (h, up, down, chosen, weight)]
    first = ops.moe_grouped(*args, F, form)
    assert float((first.cpu().double() - want).abs().max()) <= tol
    assert torch.equal(ops.moe_grouped(*args, F, form), first)
    odd = torch.empty(n * W + 1, dtype=torch.bfloat16, device="cuda")[1:].view(n, W).copy_(args[0])
    assert float((ops.moe_grouped(odd, *args[1:], F, form).cpu().double() - want).abs().max()) <= tol


@pytest.mark.parametrize("E,mean,W,F,gated,tile", [
    (4, 500, 4096, 2048, 0, 192), (8, 700, 2048, 1408, 1, 192), (16, 1000, 2048, 1024, 0, 192), (16, 700, 4096, 2048, 0, 192), (64, 500, 1024, 512, 0, 192),
    (16, 700, 2048, 1408, 1, 192), (32, 500, 4096, 2048, 0, 256), (32, 1000, 4096, 2048, 0, 256), (32, 600, 2048, 1408, 1, 256), (64, 1000, 2048, 768, 1, 256)])
def test_experts_of_many_rows_take_high_tiles_only_where_those_fill_the_chip(E, mean, W, F, gated, tile):
    from palm_infra_amd.kernels import ops
    assert ops.feedforward().palm_moe_tile_tokens(E * mean, E, W, F, gated, 1) == tile


@gpu
@pytest.mark.parametrize("form,E,top,W,F,n,uneven,tile", [
    ("gated_silu", 64, 2, 320, 1088, 640, True, 64), ("gated_silu", 64, 2, 1088, 320, 1920, True, 128), ("gated_silu", 64, 2, 320, 1088, 3520, False, 192),
    ("capped_gated", 64, 2, 1088, 320, 3520, True, 192), ("gated_silu", 64, 2, 1088, 320, 5440, True, 256), ("capped_gated", 36, 2, 1088, 1088, 3060, False, 256),
    ("relu_squared", 64, 2, 1088, 320, 1920, False, 128), ("gelu", 64, 2, 320, 1088, 7360, True, 192), ("relu_squared", 80, 2, 1088, 320, 6800, True, 256)])
def test_grouped_tiles_of_every_height_one_after_the_other(form, E, top, W, F, n, uneven, tile):
    """More tiles than compute units, so that blocks go on into another expert's, 5 and 17 stages that the walk begins inside and wraps
    around, an expert of many tiles and one that nobody chose."""
    from palm_infra_amd.kernels import ops
    gated = ops.expert_rows(form) > 1
    assert ops.feedforward().palm_moe_tile_tokens(n * top, E, W, F, int(gated), 1) == tile
    assert E * max(-(-F // (128 if gated else 256)), -(-W // 256)) > 256
    cap = CAP if form == "capped_gated" else ops.NO_CAP
    h, up, down, chosen, weight = case(form, E, top, W, F, n, uneven, E * n + F, torch.bfloat16)
    want = plain_mixture(form, h, up, down, chosen, weight, F)
    args = [t.cuda() for t in (h, up, down, chosen, weight)]
    for exact in (False, True):
        got = ops.moe_grouped(*args, F, form, cap, exact=exact)
        # the inner rows are rounded to bfloat16, 0.0017 of them in the mean square; so are the experts' results, unless they stay in 32 bits
        assert float((got.cpu().double() - want).norm() / want.norm()) < (0.003 if exact else 0.004)
        assert float((got.cpu().double() - want).abs().max()) <= 0.02 * float(want.abs().max())
        assert torch.equal(ops.moe_grouped(*args, F, form, cap, exact=exact), got)


@gpu
@pytest.mark.parametrize("form,E,W,F,rows", [("gated_silu", 320, 256, 320, (1, 31, 32, 33, 64, 127, 128, 129, 160, 161, 192, 193, 224, 225, 255, 256)),
                                             ("relu_squared", 320, 256, 320, (257, 320, 321, 384, 385, 512, 513, 576, 577, 700, 768, 769, 0, 900, 1024, 1025))])
def test_grouped_tiles_that_stop_early(form, E, W, F, rows):
    """Experts of as many rows as fill one to five tiles of 256 and a little more or less, one choice a row, the experts after those chosen by 700 or 500 each, so
    many that tiles of 256 rows are taken."""
    from palm_infra_amd.kernels import ops
    per = ops.expert_rows(form) * F
    g = torch.Generator().manual_seed(E + W)
    counts = list(rows) + [700 if form == "gated_silu" else 500] * (E - len(rows))
    chosen = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)]).to(torch.int32)
    chosen = chosen[torch.randperm(len(chosen), generator=g)][:, None]
    n = len(chosen)
    assert ops.feedforward().palm_moe_tile_tokens(n, E, W, F, int(ops.expert_rows(form) > 1), 1) == 256
    up, down = (torch.randn(E * per, W, generator=g) * W ** -0.5).to(torch.bfloat16), (torch.randn(E * W, F, generator=g) * F ** -0.5).to(torch.bfloat16)
    h, weight = torch.randn(n, W, generator=g).to(torch.bfloat16), torch.rand(n, 1, generator=g)
    want = plain_mixture(form, h, up, down, chosen, weight, F)
    args = [t.cuda() for t in (h, up, down, chosen, weight)]
    for exact in (False, True):
        got = ops.moe_grouped(*args, F, form, exact=exact).cpu().double()
        # the inner rows' rounding to bfloat16, 0.0017 in the mean square, and the experts' results' unless they stay in 32 bits
        assert float((got - want).norm() / want.norm()) < (0.003 if exact else 0.004)
        for e in range(len(rows)):                           # and in no expert's rows more than in others'
            of = chosen[:, 0] == e
            assert not of.any() or float((got[of] - want[of]).norm() / want[of].norm()) < 0.006


@gpu
@pytest.mark.parametrize("form", ["gated_silu", "gelu", "capped_gated", "relu_squared"])
@pytest.mark.parametrize("E,top,W,F,shared", [(4, 2, 64, 64, 40), (3, 1, 72, 24, None), (33, 4, 320, 264, 264), (5, 5, 8, 8, 16), (512, 3, 48, 16, None), (6, 2, 2056, 520, 1032)])
def test_few_rows(form, E, top, W, F, shared):
    """One row, a decode batch's rows, and as many as a recorded step holds: both kernels for few rows, with a shared expert and
    with planes of partial sums."""
    from palm_infra_amd.kernels import ops
    cap = CAP if form == "capped_gated" else ops.NO_CAP
    for n, uneven in ((1, False), (8, False), (17, True), (40, False), (70, True), (128, True), (128, False)):
        h, up, down, chosen, weight = case(form, E, top, W, F, n, uneven, E + F + n, torch.bfloat16)
        want = plain_mixture(form, h, up, down, chosen, weight, F)
        extra = None
        if shared:
            per = (2 if form in ("gated_silu", "capped_gated") else 1) * shared
            extra = ((torch.randn(per, W) * W ** -0.5).to(torch.bfloat16), (torch.randn(W, shared) * shared ** -0.5).to(torch.bfloat16))
            want += plain_expert(form, h.double() @ extra[0].double().T, shared) @ extra[1].double().T
            extra = tuple(t.cuda() for t in extra)
        args = [t.cuda() for t in (h, up, down, chosen, weight)]
        tol = 0.02 * float(want.abs().max())
        got = ops.moe_few(*args, F, form, cap, shared=extra)
        assert float((got.cpu().double() - want).abs().max()) <= tol, (n, uneven)
        again = ops.moe_few(*args, F, form, cap, shared=extra)
        assert torch.equal(got, again)
        assert torch.equal(ops.moe_few(*args, F, form, cap, shared=extra, once=True), got)          # (matrices marked as read once)
        planes = ops.moe_few(*args, F, form, cap, shared=extra, planes_ok=True)
        planes = planes if planes.dim() == 2 else planes.sum(0)
        assert torch.allclose(planes, got, atol=1e-4 * float(want.abs().max()), rtol=1e-4)
        exact = ops.moe_experts(*args, F, form, cap, shared=extra)
        assert float((exact.cpu().double() - want).abs().max()) <= tol, (n, uneven)
        y = [torch.randn(n, W).to(torch.bfloat16).cuda() for _ in range(2)]
        more = ops.moe_few(*args, F, form, cap, add=y, shared=extra)
        assert torch.allclose(more, got + y[0].float() + y[1].float(), atol=1e-3, rtol=1e-4)


@gpu
@pytest.mark.parametrize("form", ["gated_silu", "gelu", "capped_gated", "relu_squared"])
@pytest.mark.parametrize("E,top,W,F,shared", [(1, 1, 128, 128, None), (4, 2, 128, 384, 128), (33, 4, 1152, 256, None), (256, 32, 384, 128, 256),
                                              (6, 2, 2048, 640, 1280), (5, 5, 8192, 128, None), (40, 3, 4096, 128, 1152)])
def test_few_rows_as_one_stream(form, E, top, W, F, shared):
    """The kernels for up to 16 rows in whole lines: one step of a row of activations and all that a wave holds, waves without any,
    strips and steps that do not fill the blocks, eight rows and more, choices that repeat an expert, experts that nobody or everybody
    chose.  The inner rows and the result are rounded where the sum in float64 is not: as in the test above."""
    from palm_infra_amd.kernels import ops
    cap = CAP if form == "capped_gated" else ops.NO_CAP
    for n, uneven, repeats in ((1, False, False), (3, True, True), (8, False, False), (9, True, False), (16, False, True)):
        h, up, down, chosen, weight = case(form, E, top, W, F, n, uneven, E + F + n, torch.bfloat16)
        if repeats and top > 1:
            chosen[0, 1] = chosen[0, 0]
            chosen[n - 1, top - 1] = chosen[n - 1, 0]
        want = plain_mixture(form, h, up, down, chosen, weight, F)
        extra = None
        if shared:
            g = torch.Generator().manual_seed(n)
            per = (2 if form in ("gated_silu", "capped_gated") else 1) * shared
            extra = ((torch.randn(per, W, generator=g) * W ** -0.5).to(torch.bfloat16), (torch.randn(W, shared, generator=g) * shared ** -0.5).to(torch.bfloat16))
            want += plain_expert(form, h.double() @ extra[0].double().T, shared) @ extra[1].double().T
            extra = tuple(t.cuda() for t in extra)
        args = [t.cuda() for t in (h, up, down, chosen, weight)]
        assert ops.moe_ring_serves(*args[:3], top, E, W, F, shared or 0, extra)
        tol = 0.02 * float(want.abs().max())
        got = ops.moe_few(*args, F, form, cap, shared=extra)
        assert float((got.cpu().double() - want).abs().max()) <= tol, (n, uneven)
        assert torch.equal(ops.moe_few(*args, F, form, cap, shared=extra), got)
        y = [torch.randn(n, W).to(torch.bfloat16).cuda() for _ in range(2)]
        planes = ops.moe_few(*args, F, form, cap, add=y, shared=extra, planes_ok=True)
        planes = planes if planes.dim() == 2 else planes.sum(0)
        assert torch.allclose(planes, got + y[0].float() + y[1].float(), atol=1e-4 * float(want.abs().max()) + 1e-5, rtol=1e-4)


@gpu
@pytest.mark.parametrize("form,E,top,W,F", [("relu_squared", 6, 2, 256, 128), ("gated_silu", 4, 3, 1088, 64), ("capped_gated", 33, 4, 320, 192), ("gelu", 2, 1, 64, 704)])
def test_grouped_products_in_32_bits_are_as_near_as_the_kernels_for_few_rows(form, E, top, W, F):
    """A step of few rows may take either way: both round the inner rows to bfloat16 and nothing behind them, so their errors against
    64 bits are alike (the sums' order apart: 2^-24 against the inner rows' 2^-9); results in bfloat16 before the sum add two
    fifths.  With planes of another branch to add."""
    from palm_infra_amd.kernels import ops
    cap = CAP if form == "capped_gated" else ops.NO_CAP
    for n in (17, 40, 128):
        h, up, down, chosen, weight = case(form, E, top, W, F, n, False, E + F + n, torch.bfloat16)
        want = plain_mixture(form, h, up, down, chosen, weight, F)
        args = [t.cuda() for t in (h, up, down, chosen, weight)]
        error = lambda got: float((got.cpu().double() - want).norm() / want.norm())
        got = ops.moe_grouped(*args, F, form, cap, exact=True)
        assert error(got) <= 1.05 * error(ops.moe_few(*args, F, form, cap)), (n, error(got))
        assert torch.equal(ops.moe_grouped(*args, F, form, cap, exact=True), got)
        planes = torch.randn(3, n, W).cuda()
        more = ops.moe_grouped(*args, F, form, cap, exact=True, planes=planes)
        assert torch.allclose(more, got + planes.sum(0), atol=1e-5 * float(want.abs().max()), rtol=1e-5)
        assert torch.equal(ops.moe_grouped(*args, F, form, cap, exact=True, planes=planes[0]), ops.moe_grouped(*args, F, form, cap, exact=True, planes=planes[:1]))
    from palm_infra_amd.kernels import KernelError
    odd = torch.empty(n * W + 1, dtype=torch.bfloat16, device="cuda")[1:].view(n, W).copy_(args[0])
    with pytest.raises(KernelError, match="32-bit results"):
        ops.moe_grouped(odd, *args[1:], F, form, cap, exact=True)


@gpu
@pytest.mark.parametrize("planes,n,m", [(1, 3, 7), (2, 17, 64), (4, 128, 1030)])
def test_activation_of_a_product_in_planes(planes, n, m):
    from palm_infra_amd.kernels import ops
    z = torch.randn(planes, n, m)
    total = z.double().sum(0)
    for kind, want in (("relu_squared", torch.clamp(total, min=0.0) ** 2), ("gelu_erf", plain_expert("gelu", total, m))):
        exact = ops.activation_of_planes(z.cuda(), kind, torch.float32).cpu()
        assert torch.allclose(exact.double(), want, atol=1e-5, rtol=1e-5)
        assert torch.equal(ops.activation_of_planes(z.cuda(), kind, torch.bfloat16).cpu(), exact.to(torch.bfloat16))


def test_which_steps_go_through_the_grouped_products():
    from palm_infra_amd.kernels import ops

    def pays(n, W, F, E=1, top=1, dt=torch.bfloat16, form="gelu", shared=False, offset=0):
        h = torch.empty(n * W + 8, dtype=dt)[offset:offset + n * W].view(n, W)
        return ops.moe_grouped_pays(h, torch.empty(E * ops.expert_rows(form) * F, W, dtype=dt), torch.empty(E * W, F, dtype=dt), F, top, form, shared)
    assert pays(97, 64, 128, E=16) and pays(128, 4096, 64) and not pays(96, 64, 128, E=16)
    assert pays(48, 64, 128, E=8, top=2) and not pays(47, 64, 128, E=8, top=2) and pays(17, 64, 128)      # twelve rows an expert
    assert pays(17, 2048, 128, E=15, top=4) and not pays(17, 2048, 128, E=14, top=4)          # 135 and 126 tiles
    assert pays(17, 1792, 128, E=64, top=1) and not pays(17, 1536, 128, E=64, top=1)          # at most seventeen experts in use: 136 and 119
    assert not pays(17, 2048, 128, E=22, top=4, shared=True) and pays(17, 2048, 128, E=36, top=4, shared=True)
    assert pays(17, 1024, 512, E=32, top=4) and pays(17, 1024, 512, E=32, top=4, form="gated_silu")
    assert not pays(16, 2048, 128, E=22, top=4) and not pays(97, 72, 128) and not pays(97, 64, 40) and not pays(97, 64, 128, dt=torch.float32)
    # what the grouped products refuse or do from memory stays with the kernels for few rows: more experts, rows that start on no 16 bytes
    assert pays(97, 64, 128, E=512, top=4) and not pays(97, 64, 128, E=513, top=4)
    assert not pays(97, 64, 64, E=512, top=4) and pays(97, 64, 64, E=512, top=4, form="gated_silu")      # first matrices of a quarter of a tile
    assert not pays(97, 64, 128, offset=1) and pays(97, 64, 128, offset=8)


def test_tiles_of_the_grouped_products():
    """Low tiles as long as all run side by side, one tile an expert where the chip is full, fragments for narrow first matrices of few rows."""
    from palm_infra_amd.kernels import ops
    tile = lambda pairs, E, W, F, gated=0, aligned=1: ops.feedforward().palm_moe_tile_tokens(pairs, E, W, F, gated, aligned)
    assert tile(2000, 16, 512, 256) == 64 and tile(4000, 16, 512, 256) == 64          # 125 and 250 rows each
    assert [tile(4 * n, 32, 4096, 2048) for n in (200, 600, 850, 1500)] == [64, 128, 192, 256]
    assert tile(1200, 512, 512, 64) == tile(1200, 512, 512, 64, aligned=0) == 64 and not ops.feedforward().palm_moe_grouped_in_tiles(1200, 512, 512, 64, 0, 1)
    assert ops.feedforward().palm_moe_grouped_in_tiles(1200, 512, 512, 64, 1, 1) and ops.feedforward().palm_moe_grouped_in_tiles(320, 8, 512, 64, 0, 1)
