"""The shared launches of a backward pass (both phases of the transforms, both products) at the sizes where they can
go wrong: short Hadamard blocks with ragged tails, rows on either side of what a wave holds, jobs that round differently,
the edges of the paired products' tiles, values on and beside the boundary between two codes.  Bit-exact against the
oracle: integers, then the same fp32 operations in the same order."""
import numpy as np
import pytest
import torch

from oracle import hot_oracle as orc
from test_gpu_backward import fresh_args, make_case, run_both  # noqa: F401 (a fixture)
from test_gpu_random_cases import _options

pytestmark = pytest.mark.gpu

STOCH = dict(gx_round=orc.ROUND_STOCH, gw_round=orc.ROUND_STOCH, seed=21)


def check(gpu, L, O, I, dt, seed=3, **variant):
    x, w, gy = make_case(L, O, I, seed=seed, dtype=dt)
    ocfg = orc.HotConfig.python_rule(L, **variant)
    gx, gw, tr = run_both(x, w, gy, ocfg, _options(ocfg), gpu)
    assert torch.equal(gx.cpu(), torch.from_numpy(tr.g_x).to(dt)) and torch.equal(gw.cpu(), torch.from_numpy(tr.g_w).to(dt))


@pytest.mark.parametrize("n_o,O", [(1, 24), (2, 72), (4, 104), (8, 40), (8, 1000), (16, 272)])
@pytest.mark.parametrize("variant", [dict(), dict(gx_scale=orc.SCALE_ROW), dict(w_round=orc.ROUND_STOCH, seed=4), dict(w_scale=orc.SCALE_SAWB),
                                     dict(gx_bits=8, w_bits=8, **STOCH), dict(gx_round=orc.ROUND_STOCH, seed=9)])
def test_short_hadamard_blocks(gpu, n_o, O, variant):
    """W and the row-wise quantiser with blocks of 1 .. 16 along the out-features, the last group of 16 rows of W cut
    short; a last variant in which the two quantisers of g_y round differently."""
    check(gpu, 66, O, 40, torch.bfloat16 if O % 48 else torch.float32, n_o=n_o, **variant)


@pytest.mark.parametrize("L,O,I", [(2999, 2056, 24), (3006, 2064, 16), (6416, 2048, 8), (6464, 2056, 8), (13952, 2064, 8)])
@pytest.mark.parametrize("dt,variant", [(torch.bfloat16, dict()), (torch.float32, dict(gx_bits=8, w_bits=8, **STOCH)),
                                        (torch.float16, dict(gw_scale=orc.SCALE_ROW)), (torch.float32, dict())])
def test_row_quantiser_in_the_token_pass(gpu, L, O, I, dt, variant):
    """Tensors of 768 workgroups and more, whose token-wise pass runs the row-wise quantiser too: token blocks of 1, 2, 16, 64
    and 128, a last strip of 8 or 16 channels, row tails to clear, row groups cut short."""
    check(gpu, L, O, I, dt, n_o=min(16, O & -O), **variant)


@pytest.mark.parametrize("L", [2, 6, 12, 24, 40, 48, 160, 320])
@pytest.mark.parametrize("variant", [dict(), dict(gw_scale=orc.SCALE_ROW, act_scale=orc.SCALE_SAWB), STOCH])
def test_short_token_blocks(gpu, L, variant):
    """Token blocks of 2 .. 64, the short ones sixteen rows at a time with a tail."""
    check(gpu, L, 64, 264, torch.float32, **variant)


@pytest.mark.parametrize("O", [4096, 4112, 16384, 16400])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_row_quantiser_widths(gpu, O, dt):
    """A step per token: rows of a wave (up to 4096), of a workgroup (up to 16384) and of the kernel of their own."""
    check(gpu, 5, O, 8, dt, gx_scale=orc.SCALE_ROW)


# How the products of a shape are launched, with INT4 and with INT8 operands of g_x: apart, or together with g_x / g_W in tiles of
# 128 x 128 / 64 x 128, or of 192 x 128 both (ops.PRODUCTS_*).
APART, P128, P192 = 1, 2, 3


def launched(L, O, I, ocfg, launches):
    from hot_amd import ops
    assert (APART, P128, P192) == (ops.PRODUCTS_APART, ops.PRODUCTS_PAIR_128, ops.PRODUCTS_PAIR_192)
    return ops.backward_products(L, O, I, _options(ocfg)) == launches[ocfg.gx_bits == 8]


@pytest.mark.parametrize("L,O,I,launches", [
    (1, 16, 8, (P128, P128)), (127, 64, 128, (P128, P128)), (129, 80, 136, (P128, P128)), (192, 192, 128, (P128, P128)),
    (200, 400, 264, (P128, P128)), (300, 1664, 16, (P128, P128)),
    (64, 3072, 2048, (P192, APART)), (64, 3056, 2048, (P192, APART)), (64, 2880, 2048, (P128, APART)),
    (64, 1536, 4096, (P192, P192)), (64, 1536, 3968, (P128, P128)),
    (40, 3328, 136, (P128, APART)), (40, 3584, 136, (APART, APART)), (1800, 1792, 16, (P128, APART))])
@pytest.mark.parametrize("dt,bits", [(torch.float32, 4), (torch.bfloat16, 8), (torch.float16, 4)])
def test_paired_products(gpu, L, O, I, launches, dt, bits):
    """Tile edges of the paired products, K shorter than the ring, either side of the line between their two tilings (256 tiles of
    192 x 128 of g_W: 1536 x 4096, 3072 x 2048); g_x products of few tiles on either side of the length of K (14 stages, twice
    those of g_W) from which the two go apart."""
    assert launched(L, O, I, orc.HotConfig.python_rule(L, gx_bits=bits, w_bits=bits), launches)
    check(gpu, L, O, I, dt, gx_bits=bits, w_bits=bits)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("L,O,I,launches", [(200, 144, 264, (P128, P128)), (384, 144, 256, (P128, P128)),
                                            (208, 1552, 4104, (P192, P192)), (64, 3088, 2176, (P192, APART))])
@pytest.mark.parametrize("size", [1.0, 2.0 ** -12])
def test_epilogues_of_paired_products(gpu, dt, bits, L, O, I, launches, size):
    """Whole tiles (stored through LDS) and cut ones (stored directly) of both products in both tilings (first and third shape; the
    second has no cut tile of g_x, the last no whole one), with the powers of two folded into the steps: the values of the
    unfolded form, also where fp16 results are subnormal (gradients of 2^-12 size) and are rounded to fp32 first.  With INT8
    operands the last shape runs the products one after the other, unfolded."""
    x, w, gy = make_case(L, O, I, seed=5, dtype=torch.float32)
    ocfg = orc.HotConfig.python_rule(L, gx_bits=bits, w_bits=bits, n_o=16)
    assert launched(L, O, I, ocfg, launches)
    x, w, gy = x.to(dt), w.to(dt), (gy * size).to(dt)
    gx, gw, tr = run_both(x, w, gy, ocfg, _options(ocfg), gpu)
    assert torch.equal(gx.cpu(), torch.from_numpy(tr.g_x).to(dt)) and torch.equal(gw.cpu(), torch.from_numpy(tr.g_w).to(dt))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("L,O,I,launches", [(200, 144, 264, (P128, P128)), (208, 1552, 4104, (P192, P192))])
@pytest.mark.parametrize("case,dt", [(c, d) for c in ("g_x overflows", "g_w overflows", "g_w subnormal", "row steps")
                                     for d in (torch.float32, torch.bfloat16)] + [("row steps", torch.float16)])
def test_products_at_the_ends_of_the_range(gpu, dt, bits, L, O, I, launches, case):
    """Steps so large that a product of them overflows before the scale of the transform brings it back, and so small that
    results are subnormal (rounded once more): the paired launch, in both tilings, gives the values of the unfolded form there
    too, on whole tiles as on cut ones, and those of the products launched apart.  Last: rows whose steps lie on either side of
    what the folded form takes (2^-48, 2^47), and rows of zeros."""
    from dataclasses import replace
    from hot_amd import ops
    x, w, gy = make_case(L, O, I, seed=8)
    by_row = dict(gx_scale=orc.SCALE_ROW, gw_scale=orc.SCALE_ROW) if case == "row steps" else {}
    ocfg = orc.HotConfig.python_rule(L, gx_bits=bits, w_bits=bits, n_o=16, **by_row)
    opt = _options(ocfg)
    assert launched(L, O, I, ocfg, launches)
    xq_ref, sx_ref = orc.abc_forward(x.numpy(), ocfg)
    ref = lambda sx: orc.linear_backward(gy.to(dt).float().numpy(), w.to(dt).float().numpy(), xq_ref, sx, ocfg)
    top = lambda v: int(np.ceil(np.log2(np.abs(v).max())))
    tr = ref(sx_ref)
    sx = sx_ref
    if case == "g_x overflows":                     # the largest sum of scaled products reaches 2^129, the result 2^125
        k = 129 - top(tr.g_x) - 4
        gy, w = gy * 2.0 ** (k // 2), w * 2.0 ** (k - k // 2)
    elif case == "g_w overflows":                   # (a step of the caller's: 2^129 again, divided by the token block)
        sx = sx_ref * np.float32(2.0 ** (129 - top(tr.g_w) - int(np.log2(ocfg.hla_n))))
    elif case == "g_w subnormal":                   # results of at most 2^-124
        gy = gy * 2.0 ** -20
        sx = sx_ref * np.float32(2.0 ** (-124 - top(ref(sx_ref).g_w)))
    elif case == "row steps":
        e = torch.tensor([0, 50, 55, 60, -10, -20, -30, -48]) // (5 if dt == torch.float16 else 1)
        gy = gy * 2.0 ** e.repeat(L // 8)[:, None]
        gy[3::16] = 0.0
    with np.errstate(over="ignore"):
        tr = ref(sx)
    if case == "g_x overflows":
        assert np.isinf(tr.g_x).any() and np.isfinite(tr.g_x).mean() > 0.9
    elif case == "g_w overflows":
        assert np.isinf(tr.g_w).any() and np.isfinite(tr.g_w).mean() > 0.9
    args = (gy.to(dt).to(gpu), w.to(dt).to(gpu), torch.from_numpy(np.ascontiguousarray(_buffer(xq_ref))).to(gpu), torch.from_numpy(sx).to(gpu))
    gx, gw = ops.linear_backward(*args, opt)
    apart = ops.linear_backward(*args, replace(opt, streams=2))
    assert torch.equal(gx, apart[0]) and torch.equal(gw, apart[1])
    assert torch.equal(gx.cpu(), torch.from_numpy(tr.g_x).to(dt)) and torch.equal(gw.cpu(), torch.from_numpy(tr.g_w).to(dt))


@pytest.mark.parametrize("L,O,I,rows", [
    (1, 16, 8, 64), (63, 64, 64, 64), (65, 80, 72, 64), (128, 128, 128, 64), (449, 16, 72, 64),
    (64, 784, 128, 64), (64, 1040, 72, 64), (64, 1296, 64, 64), (64, 1808, 64, 64), (1153, 2048, 64, 64),
    (771, 80, 4104, 128), (1001, 64, 3992, 128), (896, 64, 4096, 128), (6304, 16, 3080, 128),
    (208, 1552, 4104, 192)])
@pytest.mark.parametrize("dt,bits", [(torch.float32, 4), (torch.bfloat16, 8), (torch.float16, 4)])
def test_tilings_of_paired_products(gpu, L, O, I, rows, dt, bits):
    """The three tilings of the paired launch: edges of their tiles, and with 64 x 64 as many stages of g_x and g_W as leave the
    ring of four unfilled, fill it, and take every remainder of its rounds."""
    from hot_amd import ops
    ocfg = orc.HotConfig.python_rule(L, gx_bits=bits, w_bits=bits)
    if not (bits == 8 and O > 1664):                # (those go apart)
        assert ops.backward_pair_rows(L, O, I, _options(ocfg)) == rows
    check(gpu, L, O, I, dt, gx_bits=bits, w_bits=bits)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("case,dt", [("g_x overflows", torch.float32), ("g_w subnormal", torch.bfloat16), ("row steps", torch.float16)])
def test_ends_of_the_range_in_wide_tiles(gpu, dt, bits, case):
    """The same in tiles of 128 x 128 / 64 x 128, whole ones and cut ones."""
    from hot_amd import ops
    L, O, I = 776, 80, 4104
    ocfg = orc.HotConfig.python_rule(L, gx_bits=bits, w_bits=bits, n_o=16)
    assert ops.backward_pair_rows(L, O, I, _options(ocfg)) == 128
    test_products_at_the_ends_of_the_range(gpu, dt, bits, L, O, I, (P128, P128), case)


def _buffer(xq):
    """The oracle's codes [L', I] as the activation buffer holds them: [I, L' rounded up to whole lines of 128 codes]."""
    out = np.zeros((xq.shape[1], -(-xq.shape[0] // 128) * 128), np.int8)
    out[:, :xq.shape[0]] = xq.T
    return out


@pytest.mark.parametrize("bits,O", [(8, 133144), (4, 171192)])
def test_longest_rows(gpu, bits, O):
    """As many out-features as an int32 accumulator takes: the zero codes that pad a row to whole lines do not count."""
    check(gpu, 3, O, 8, torch.bfloat16, n_o=8, gx_bits=bits, w_bits=bits)


@pytest.mark.parametrize("scale", [1.0, 3.1e-3, 7.7e4])
@pytest.mark.parametrize("bits", [4, 8])
def test_codes_on_the_boundary(gpu, scale, bits):
    """Values whose quotient by the step lies on a half-integer, or one ulp beside it: the code is that of the IEEE
    quotient rounded to even (np.rint), wherever the fast path cannot decide."""
    from hot_amd import ops
    qmax = 2 ** (bits - 1) - 1
    step = np.float32(scale)
    half = (np.arange(-qmax, qmax, dtype=np.float32) + np.float32(0.5)) * step
    v = np.concatenate([half, np.nextafter(half, np.float32(np.inf)), np.nextafter(half, np.float32(-np.inf))]).astype(np.float32)
    v = np.concatenate([v, np.full((-v.size - 8) % 16, 0, np.float32), np.full(8, step * np.float32(qmax), np.float32)])
    t = torch.from_numpy(np.tile(v, (4, 1)))
    codes, steps = ops.hq_rowwise(t.to(gpu), n=1, bits=bits, scale="row")
    d = np.float32(np.float32(np.max(np.abs(v))) / np.float32(qmax))
    assert np.array_equal(steps.cpu().numpy(), np.full(4, d))
    ref = np.rint(v / np.float32(d + np.float32(1e-11))).astype(np.int64)
    got = codes.cpu().numpy().astype(np.int64)
    if bits == 4:
        lo, hi = got & 15, (got >> 4) & 15
        got = np.stack([lo, hi], -1).reshape(4, -1)
        got = np.where(got > 7, got - 16, got)
    assert np.array_equal(got, np.tile(ref, (4, 1)))
    # the same values along the tokens (blocks of one): the column-wise body
    col, sc, kout = ops.hla_tokenwise(torch.from_numpy(np.tile(v[:, None], (1, 8))).to(gpu), 1, (0,), bits=bits)
    assert np.array_equal(col.cpu().numpy()[:, :kout].astype(np.int64), np.tile(ref, (8, 1)))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,O,variant", [(5, 197, 208, dict()), (3, 64, 192, dict(gx_scale=orc.SCALE_ROW, gw_scale=orc.SCALE_ROW)),
                                           (4, 196, 96, STOCH), (7, 6, 8, dict()), (2, 48, 264, dict()), (1, 128, 40, STOCH),
                                           (3, 640, 16, dict()), (130, 197, 128, dict()), (64, 2, 2056, dict(gx_scale=orc.SCALE_ROW))])
def test_batched_bias_gradient(gpu, dt, B, T, O, variant):
    """The column sums that leave the statistics pass of a batched backward: token blocks of 1 .. 128, the last strip of a
    sample cut short, strips of many samples.  Integers (below 2^24): every order gives the exact sum, a block dropped, doubled or
    misplaced shows.  Random values: within the fp32 accumulation bound of the 64-bit sum.  g_x and g_W stay as without it."""
    from hot_amd import ops
    ocfg = orc.HotConfig.python_rule(T, n_o=min(16, O & -O), **variant)
    opt = _options(ocfg)
    g = torch.Generator().manual_seed(B * T + O)
    w = ((torch.rand(O, 24, generator=g) * 2 - 1) / 5).to(dt).to(gpu)
    xq, sx = ops.abc_forward_batched(torch.randn(B, T, 24, generator=g).to(dt).to(gpu), opt)
    gy = torch.randn(B, T, O, generator=g).to(dt)
    gx, gw, gb = ops.linear_backward_batched(gy.to(gpu), w, xq, sx, opt, out_dtype=torch.float32, bias_grad=True)
    gx0, gw0 = ops.linear_backward_batched(gy.to(gpu), w, xq, sx, opt, out_dtype=torch.float32)
    assert torch.equal(gx, gx0) and torch.equal(gw, gw0)
    d = gy.double().reshape(-1, O)
    assert torch.all((gb.cpu().double() - d.sum(0)).abs() <= B * T * 2.0 ** -24 * d.abs().sum(0))
    gi = torch.randint(-8, 9, (B, T, O), generator=g).to(dt)
    gb = ops.linear_backward_batched(gi.to(gpu), w, xq, sx, opt, out_dtype=torch.float32, bias_grad=True)[2]
    assert torch.equal(gb.cpu(), gi.double().reshape(-1, O).sum(0).float())


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,O", [(8191, 2064), (12608, 3072), (16384, 768)])
def test_bias_gradient_of_one_long_sample(gpu, dt, T, O):
    """One sample with a step per channel and so many runs of token blocks that the statistics pass would rather take longer ones: the
    bias gradient adds up the rows that this call wrote, in both entry points.  NaN wherever the call has not written; integers, of
    which every order gives the exact sum."""
    from hot_amd import ops
    n, rows = orc.hla_rows(min(T & -T, 64))
    opt = ops.HotOptions(n_o=16, hla_n=n, hla_rows=tuple(int(v) for v in rows), gx_scale="row", gw_scale="row")
    g = torch.Generator(device=gpu).manual_seed(T)
    gy = torch.randint(-8, 9, (1, T, O), generator=g, device=gpu).to(dt)
    w, x = torch.rand(O, 16, generator=g, device=gpu).to(dt), torch.randn(1, T, 16, generator=g, device=gpu).to(dt)
    ref = gy[0].double().sum(0).float()
    ws = torch.empty(1 << 28, dtype=torch.uint8, device=gpu)
    for back, buf, v in ((ops.linear_backward_batched, ops.abc_forward_batched, gy), (ops.linear_backward, lambda t, o: ops.abc_forward(t[0], o), gy[0])):
        xq, sx = buf(x, opt)
        ws.view(torch.float32).fill_(float("nan"))
        gx, gw, gb = back(v, w, xq, sx, opt, out_dtype=torch.float32, workspace=ws, bias_grad=True)
        assert torch.equal(gb, ref)
        gx0, gw0 = back(v, w, xq, sx, opt, out_dtype=torch.float32, workspace=ws)      # (this one takes the longer runs)
        assert torch.equal(gx, gx0) and torch.equal(gw, gw0)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("O", [96, 100])
def test_layer_bias_gradient_per_sample(gpu, fresh_args, dt, O):
    """The bias gradient of a layer on 3-D activations with steps per sample, widths with and without padding: the 64-bit
    sum within the fp32 accumulation bound and one rounding of the type."""
    from hot_amd.quant_matmul import HQ_Linear
    fresh_args.hot_recipe()
    fresh_args.batched_mode = "per_sample"
    g = torch.Generator().manual_seed(O)
    lin = HQ_Linear(64, O).to(gpu).to(dt)
    gy = torch.randn(6, 197, O, generator=g).to(dt)
    lin(torch.randn(6, 197, 64, generator=g).to(dt).to(gpu)).backward(gy.to(gpu))
    d = gy.double().reshape(-1, O)
    bound = 6 * 197 * 2.0 ** -24 * d.abs().sum(0) + (2.0 ** -8 * d.sum(0).abs() if dt == torch.bfloat16 else 0)
    assert lin.bias.grad.dtype == dt and torch.all((lin.bias.grad.double().cpu() - d.sum(0)).abs() <= bound)


# An fp32 NaN with a payload (its low byte is no code), quiet and negative.
NAN = np.array([0x7FC12345, 0xFFC0007F], np.uint32).view(np.float32)


@pytest.mark.parametrize("n", [1, 2, 8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("rounding", ["nearest", "stoch"])
def test_nan_and_infinity_in_the_quantisers(gpu, n, rounding):
    """A NaN spoils the Hadamard block that holds it and nothing else: its codes are 0, like those of a block of zeros, whatever
    its payload.  An infinity makes the step infinite and every code 0."""
    from hot_amd import ops
    L, C = 512, 264
    x = np.random.default_rng(n).standard_normal((L, C)).astype(np.float32)
    x[300, 17] = 1000.0                                        # the absmax, in a block of its own
    bad, zeroed = x.copy(), x.copy()
    bad[70, 40], bad[511, 263] = NAN
    zeroed[70 // n * n:70 // n * n + n, 40] = zeroed[511 // n * n:, 263] = 0.0
    tok = lambda v: ops.hla_tokenwise(torch.from_numpy(v).to(gpu), n, tuple(range(n)), bits=8, rounding=rounding, seed=3)
    for got, ref in zip(tok(bad)[:2], tok(zeroed)[:2]):
        assert torch.equal(got, ref)
    bad[70, 40] = np.inf
    bad[511, 263] = 0.0
    q, step = tok(bad)[:2]
    assert torch.isinf(step).all() and not q.any()
    if n > 64:
        return
    for scale in ("tensor", "row"):
        w = x[:, :256].copy()
        bad, zeroed = w.copy(), w.copy()
        bad[70, 40], bad[511, 255] = NAN
        zeroed[70, 40 // n * n:40 // n * n + n] = zeroed[511, 255 // n * n:] = 0.0
        row = lambda v: ops.hq_rowwise(torch.from_numpy(v).to(gpu), n=n, bits=4, rounding=rounding, scale=scale, seed=3)
        for got, ref in zip(row(bad), row(zeroed)):
            assert torch.equal(got, ref)


@pytest.mark.parametrize("L,O", [(66, 272), (2999, 2064), (6464, 2064)])
@pytest.mark.parametrize("scale", ["tensor", "row"])
def test_nan_in_the_gradient(gpu, L, O, scale):
    """The same through the backward: g_x misses the row-wise block that holds the NaN, g_W the token-wise one.  The last two
    shapes join the row-wise quantiser to the token-wise pass (steps per tensor)."""
    from hot_amd import ops
    x, w, gy = make_case(L, O, 24, seed=5, dtype=torch.float32)
    ocfg = orc.HotConfig.python_rule(L, gx_scale=orc.SCALE_ROW if scale == "row" else orc.SCALE_TENSOR)
    opt, n = _options(ocfg), ocfg.hla_n
    gy = gy.numpy()
    gy[1, 3] = 100 * np.abs(gy).max()
    t, o = L - 1, O - 20                                        # (a Hadamard block other than the one of the absmax)
    bad, zero_row, zero_tok = gy.copy(), gy.copy(), gy.copy()
    bad[t, o] = NAN[0]
    zero_row[t, o // 16 * 16:o // 16 * 16 + 16] = 0.0
    zero_tok[t // n * n:t // n * n + n, o] = 0.0
    xq, sx = ops.abc_forward(x.to(gpu), opt)
    back = lambda v: ops.linear_backward(torch.from_numpy(v).to(gpu), w.to(gpu), xq, sx, opt)
    gx, gw = back(bad)[:2]
    assert torch.equal(gx, back(zero_row)[0]) and torch.equal(gw, back(zero_tok)[1])


@pytest.mark.parametrize("L,O,I,bits", [(4032, 5120, 640, 8), (4672, 11008, 256, 4)])
def test_long_products_that_leave_the_paired_launch(gpu, L, O, I, bits):
    """Few g_x tiles with a long K in a call long enough for a side stream: the default order keeps both products on the
    caller's stream (shorter INT8 tiles; INT4 in K ranges through the split workspace) and gives the bits of the forced orders."""
    from dataclasses import replace
    from hot_amd import ops
    x, w, gy = make_case(L, O, I, seed=6, dtype=torch.bfloat16)
    ocfg = orc.HotConfig.python_rule(L, gx_bits=bits, w_bits=bits)
    opt = _options(ocfg)
    assert ops.backward_streams(L, O, I, opt) == 2 and launched(L, O, I, ocfg, (APART, APART))
    gx, gw, tr = run_both(x, w, gy, ocfg, opt, gpu)
    assert torch.equal(gx.cpu(), torch.from_numpy(tr.g_x).to(gx.dtype)) and torch.equal(gw.cpu(), torch.from_numpy(tr.g_w).to(gw.dtype))
    xq, sx = ops.abc_forward(x.to(gpu), opt)
    for streams in (1, 2):
        other = ops.linear_backward(gy.to(gpu), w.to(gpu), xq, sx, replace(opt, streams=streams))
        assert torch.equal(gx, other[0]) and torch.equal(gw, other[1])
