"""The decoder language models' operators on the device, each mechanism alone, against the plain implementation."""
import ctypes as C
import importlib

import numpy as np
import pytest

import decoder_cases as cases
import decoder_oracle as plain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def decoder():
    return importlib.import_module("qingming-qwen3-tts_amd.decoder")


def put(a, dev, dtype=None):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev) if dtype is None else torch.from_numpy(np.ascontiguousarray(a)).to(dtype).to(dev)


def get(t):
    import torch
    torch.cuda.synchronize()
    return t.float().cpu().numpy()


def activation(f32):
    import torch
    return torch.float32 if f32 else torch.bfloat16


def close(got, want, f32, tol32=2e-6, tol16=4e-3):
    scale = np.abs(want).max() + 1e-30
    worst = np.abs(got.astype(np.float64) - want).max() / scale
    assert worst <= (tol32 if f32 else tol16), worst


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("width,ld,rows", [(96, 128, 3), (264, 384, 2), (1500, 1536, 2), (2048, 2048, 4), (4000, 4096, 2), (9000, 9088, 2)])
def test_residual_norm(decoder, dev, f32, width, ld, rows):
    import torch
    rng = np.random.default_rng(width)

    def padded(n):
        out = np.zeros((n, ld), np.float32)
        out[:, :width] = rng.standard_normal((n, width))
        return out

    x, y, step, norms = padded(7), [padded(7) for _ in range(3)], padded(1)[0], padded(3)
    embed = cases.bf16(padded(11))
    tokens = rng.integers(0, 11, 7).astype(np.int32)
    row_map = rng.permutation(7)[:rows].astype(np.int32)
    d = {n: put(v, dev) for n, v in (("x", x), ("y0", y[0]), ("y1", y[1]), ("y2", y[2]), ("step", step), ("norms", norms), ("tokens", tokens), ("map", row_map))}
    table = put(embed, dev, torch.bfloat16)
    eps, w = 0.01, slice(0, width)

    bigram = cases.bf16(padded(6))
    d["fed"], bigrams = put(np.concatenate([[-1], tokens]).astype(np.int32), dev), put(bigram, dev, torch.bfloat16)      # (no token before row 0's)

    def terms(src):
        return (0.5 * plain.rms_norm(y[0][src, w], norms[0, w], eps) - 0.25 * plain.rms_norm(y[1][src, w], norms[1, w], eps) + y[2][src, w])

    for mapped, embedded, count, stepped, pairs in ((False, False, 3, True, False), (True, False, 3, False, False), (True, True, 0, True, False),
                                                    (False, True, 2, False, False), (False, True, 0, False, True), (True, True, 2, False, True)):
        src = row_map if mapped else np.arange(rows)
        want = (embed[tokens[src]][:, w] if embedded else x[src, w]).astype(np.float64)
        if pairs:
            rows_of = [5 if i == 0 else (3 * int(tokens[i - 1]) + 4 * int(tokens[i])) % 5 for i in src]
            want = want + bigram[rows_of][:, w]
        if count == 3:
            want = want + terms(src)
        elif count == 2:
            want = want + 0.5 * plain.rms_norm(y[0][src, w], norms[0, w], eps) + y[2][src, w]
        if stepped:
            want = want + step[w]
        x_out = torch.full((rows, ld), 7.0, device=dev)
        h = torch.full((rows, ld), 7.0, device=dev, dtype=activation(f32))
        op = decoder.ResidualNorm(x_in=None if embedded else d["x"].data_ptr(), embed=table.data_ptr(), tokens=d["tokens"].data_ptr(),
                                  row_map=d["map"].data_ptr() if mapped else None, step_vec=d["step"].data_ptr() if stepped else None,
                                  norm_w=d["norms"].data_ptr() + 8 * ld, x_out=x_out.data_ptr(), h=h.data_ptr(), ld_h=ld, width=width, vocab=11,
                                  terms=count, eps=eps)
        if pairs:
            op.tokens, op.bigram = d["fed"].data_ptr() + 4, bigrams.data_ptr()
            op.buckets, op.mul_prev, op.mul_cur = 5, 3, 4
        chosen = [("y0", 0, 0.5), ("y1", 1, -0.25), ("y2", None, 1.0)] if count == 3 else [("y0", 0, 0.5), ("y2", None, 1.0)][:count]
        for i, (name, norm, scale) in enumerate(chosen):
            op.term[i] = decoder.ResidualTerm(d[name].data_ptr(), None if norm is None else d["norms"].data_ptr() + 4 * norm * ld, ld, scale, 0)
        assert decoder.lib().qm_residual_norm_rows(C.byref(op), rows, int(f32), torch.cuda.current_stream().cuda_stream) == 0
        got_x, got_h = get(x_out), get(h)
        close(got_x[:, w], want, True)
        close(got_h[:, w], plain.rms_norm(want, norms[2, w], eps), f32)
        assert np.all(got_x[:, width:] == 0) and np.all(got_h[:, width:] == 0)


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("groups,size,ld", [(1, 96, 128), (1, 2048, 2048), (1, 5000, 5120), (1, 70, 128), (3, 20, 128), (16, 128, 2048), (2, 160, 384), (1, 1, 128)])
@pytest.mark.parametrize("silu", [0, 1])
def test_gated_norm(decoder, dev, f32, groups, size, ld, silu):
    import torch
    rng = np.random.default_rng(size)
    n, rows = groups * size, 3
    o, gate, weight = rng.standard_normal((rows, n)).astype(np.float32), rng.standard_normal((rows, n + 12)).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    out = torch.full((rows, ld), 7.0, device=dev, dtype=activation(f32))
    d = [put(v, dev) for v in (o, weight, gate)]
    op = decoder.GatedNorm(o=d[0].data_ptr(), weight=None if silu else d[1].data_ptr(), silu=silu, gate=d[2].data_ptr(), out=out.data_ptr(), ld_o=n, ld_gate=n + 12, ld_out=ld,
                           groups=groups, size=size, eps=0.02)
    assert decoder.lib().qm_gated_norm_rows(C.byref(op), rows, int(f32), torch.cuda.current_stream().cuda_stream) == 0
    g = gate[:, :n].astype(np.float64)
    want = plain.rms_norm(o.astype(np.float64).reshape(rows, groups, size), 1.0, 0.02).reshape(rows, n) * (plain.silu(g) if silu else weight * plain.sigmoid(g))
    got = get(out)
    close(got[:, :n], want, f32)
    assert np.all(got[:, n:] == 0)


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("groups,size", [(4, 65), (5, 128), (5, 129), (8, 128), (8, 129), (9, 3), (9, 64), (9, 86), (16, 64), (17, 256), (8, 300)])
@pytest.mark.parametrize("rows", [1, 512, 513, 1025])
def test_gated_norm_in_slices_at_once(decoder, dev, f32, groups, size, rows):
    """Slices one by one and four at a time, around the lines between them in rows, slices and sizes."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(groups * size)
    n = groups * size
    ld = (n + 127) // 128 * 128
    o, gate, weight = torch.randn(rows, n, device=dev, generator=gen), torch.randn(rows, n, device=dev, generator=gen), torch.randn(n, device=dev, generator=gen)
    out = torch.full((rows + 1, ld), 7.0, device=dev, dtype=activation(f32))
    op = decoder.GatedNorm(o=o.data_ptr(), weight=weight.data_ptr(), gate=gate.data_ptr(), out=out.data_ptr(), ld_o=n, ld_gate=n, ld_out=ld, groups=groups,
                           size=size, eps=0.02)
    assert decoder.lib().qm_gated_norm_rows(C.byref(op), rows, int(f32), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    wide = o.double().reshape(rows, groups, size)
    want = (wide / (wide.square().mean(2, keepdim=True) + 0.02).sqrt()).reshape(rows, n) * weight.double() * torch.sigmoid(gate.double())
    close(out[:rows, :n].float().cpu().numpy(), want.cpu().numpy(), f32)
    assert bool((out[:rows, n:] == 0).all()) and bool((out[rows:] == 7).all())


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("n", [16, 48, 64, 80])
@pytest.mark.parametrize("rows,k,ldx,ldo", [(1, 128, 128, 128), (7, 256, 264, 132), (16, 128, 128, 128), (33, 384, 392, 140), (200, 2048, 2048, 128)])
def test_linear_of_few_columns(decoder, dev, f32, rows, k, ldx, ldo, n):
    import torch
    rng = np.random.default_rng(rows)
    x, w = cases.bf16(rng.standard_normal((rows, ldx))), cases.bf16(rng.standard_normal((n, k)) * k ** -0.5)
    xd, wd = put(x, dev, activation(f32)), put(w, dev, torch.bfloat16)
    out = torch.full((rows + 1, ldo), 7.0, device=dev)
    linear = decoder.DecoderLinear(x=xd.data_ptr(), w=wd.data_ptr(), out32=out.data_ptr(), ldx=ldx, ldo=ldo, n=n, k=k)
    assert decoder.lib().qm_decoder_linear_rows(C.byref(linear), 1, rows, int(f32), torch.cuda.current_stream().cuda_stream) == 0
    got = get(out)
    close(got[:rows, :n], x[:, :k].astype(np.float64) @ w.T, True, tol32=3e-6)
    assert np.all(got[rows:] == 7) and np.all(got[:, n:] == 7)


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("rows", [1, 2, 3, 5, 9, 15, 16, 40, 130])
def test_linears(decoder, dev, f32, rows):
    """Three linears of their own inputs and reductions in one launch, the last a gate/up pair."""
    import torch
    rng = np.random.default_rng(rows)
    shapes = [(256, 128), (128, 896), (384, 640)]
    x = [cases.bf16(rng.standard_normal((rows, k))) for _, k in shapes]
    w = [cases.bf16(rng.standard_normal((n, k)) * k ** -0.5) for n, k in shapes]
    up = cases.bf16(rng.standard_normal(shapes[2]) * shapes[2][1] ** -0.5)
    xd = [put(v, dev, activation(f32)) for v in x]
    wd = [put(v, dev, torch.bfloat16) for v in w + [up]]
    outs = [torch.full((rows, shapes[i][0]), 7.0, device=dev, dtype=torch.float32 if i < 2 else activation(f32)) for i in range(3)]
    linears = (decoder.DecoderLinear * 3)()
    for i, (n, k) in enumerate(shapes):
        linears[i] = decoder.DecoderLinear(x=xd[i].data_ptr(), w=wd[i].data_ptr(), w_up=wd[3].data_ptr() if i == 2 else None,
                                           out32=outs[i].data_ptr() if i < 2 else None, out=outs[i].data_ptr() if i == 2 else None, ldx=k, ldo=n, n=n, k=k)
    assert decoder.lib().qm_decoder_linear_rows(linears, 3, rows, int(f32), torch.cuda.current_stream().cuda_stream) == 0
    for i in range(2):
        close(get(outs[i]), x[i].astype(np.float64) @ w[i].T, True, tol32=3e-6)
    gate = x[2].astype(np.float64) @ w[2].T
    close(get(outs[2]), plain.silu(gate) * (x[2].astype(np.float64) @ up.T), f32, tol32=3e-6, tol16=2e-2)


@pytest.mark.parametrize("rows,k", [(5, 4096), (8, 6144), (9, 256), (12, 2048), (15, 640)])
@pytest.mark.parametrize("pair", [False, True])
def test_few_bf16_rows_give_the_same_bits_together_and_alone(decoder, dev, rows, k, pair):
    """Up to 15 rows a row is the dot products': fp32 sums in one order, a pair rounded once behind its product."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(rows)
    n = 256
    x = torch.randn(rows, k, device=dev, generator=gen).bfloat16()
    w, up = ((torch.randn(n, k, device=dev, generator=gen) * k ** -0.5).bfloat16() for _ in range(2))
    dtype = torch.bfloat16 if pair else torch.float32

    def run(first, count):
        out = torch.full((count, n), 7.0, device=dev, dtype=dtype)
        linear = decoder.DecoderLinear(x=x.data_ptr() + 2 * k * first, w=w.data_ptr(), w_up=up.data_ptr() if pair else None, out32=None if pair else out.data_ptr(),
                                       out=out.data_ptr() if pair else None, ldx=k, ldo=n, n=n, k=k)
        assert decoder.lib().qm_decoder_linear_rows(C.byref(linear), 1, count, 0, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return out

    assert torch.equal(run(0, rows), torch.cat([run(i, 1) for i in range(rows)]))


@pytest.mark.parametrize("rows", [1, 8, 9, 15])
def test_a_reduction_too_long_for_the_dot_products_is_refused(decoder, dev, rows):
    import torch
    n, k = 128, 65536 + 128
    x, w = torch.zeros(rows, k, device=dev, dtype=torch.bfloat16), torch.zeros(n, k, device=dev, dtype=torch.bfloat16)
    out = torch.full((rows, n), 7.0, device=dev)
    linear = decoder.DecoderLinear(x=x.data_ptr(), w=w.data_ptr(), out32=out.data_ptr(), ldx=k, ldo=n, n=n, k=k)
    assert decoder.lib().qm_decoder_linear_rows(C.byref(linear), 1, rows, 0, torch.cuda.current_stream().cuda_stream) == -2
    assert bool((out == 7).all())


SPLIT_LINEARS = [
    # every tile of the 32-bit mode's matrix-core linears: columns that end inside a tile, reductions of an odd number of steps per share
    (16, 2128, 2048, False), (9, 3600, 2176, False), (33, 1040, 2048, False), (40, 1040, 1664, False), (129, 6640, 128, False),
    (300, 6640, 128, False), (10, 1664, 2176, True), (33, 1024, 1152, True), (150, 4096, 128, True), (257, 4096, 128, True),
    # (and those of the above that a single round of the dot products' blocks covers, with more rows or columns)
    (81, 1040, 2048, False), (81, 1040, 1664, False), (81, 1024, 1152, True), (10, 4096, 2176, True)]


@pytest.mark.parametrize("rows,n,k,pair", SPLIT_LINEARS)
def test_linears_of_many_fp32_rows(decoder, dev, rows, n, k, pair):
    """Against 64 bits, per output: a sum of k exact products through at most k / 64 + 80 roundings of partial sums that sum |x w| bounds.
    Columns of x differ by up to 2^40; the last row holds an infinity."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(rows)
    ldx, ldo = k + 8, n + 12
    x = torch.randn(rows, ldx, device=dev, generator=gen) * torch.exp2(torch.randint(-20, 21, (ldx,), device=dev, generator=gen).float())
    w, up = ((torch.randn(n, k, device=dev, generator=gen) * k ** -0.5).bfloat16() for _ in range(2))
    if pair:
        x /= x.abs().amax(1, keepdim=True)
    else:
        x[-1, 3] = float("inf")
    out = torch.full((rows + 1, ldo), 7.0, device=dev)
    linear = decoder.DecoderLinear(x=x.data_ptr(), w=w.data_ptr(), w_up=up.data_ptr() if pair else None, out32=None if pair else out.data_ptr(),
                                   out=out.data_ptr() if pair else None, ldx=ldx, ldo=ldo, n=n, k=k)
    assert decoder.lib().qm_decoder_linear_rows(C.byref(linear), 1, rows, 1, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert bool((out[rows:] == 7).all()) and bool((out[:, n:] == 7).all())
    got, wide = out[:rows, :n].double().cpu(), x[:, :k].double().cpu()
    unit = (k / 64 + 80) * 2.0 ** -24
    gate, most = wide @ w.double().cpu().T, wide.abs() @ w.double().cpu().abs().T
    if pair:
        other, other_most = wide @ up.double().cpu().T, wide.abs() @ up.double().cpu().abs().T
        want = torch.nn.functional.silu(gate) * other
        # (silu's slope is at most 1.1; its exponential, reciprocal and product are good to a few units in the last place)
        bound = unit * (1.1 * most * other.abs() + torch.nn.functional.silu(gate).abs() * other_most) + 8 * 2.0 ** -24 * want.abs() + 1e-12
    else:
        assert torch.equal(got[-1].isinf(), w[:, 3].cpu() != 0) and torch.equal(got[-1].sign(), w[:, 3].double().cpu().sign())
        want, bound, got = gate[:-1], unit * most[:-1], got[:-1]
    assert bool(((got - want).abs() <= bound).all()), float(((got - want).abs() / bound).max())


@pytest.mark.parametrize("rows,n,k,pair", SPLIT_LINEARS)
def test_many_fp32_rows_meet_infinite_weights(decoder, dev, rows, n, k, pair):
    """Infinities and NaNs stand where the dot products of few rows have them: infinite weights against inputs with nothing behind their
    upper bits, zeros, subnormals and infinities."""
    import torch
    inf = float("inf")
    gen = torch.Generator(device=dev).manual_seed(rows)
    x = torch.randn(rows, k, device=dev, generator=gen)
    x[0], x[1], x[2, 3], x[3, :64], x[-2] = 1.0, 0.5, 0.0, 1e-41, x[-2].bfloat16().float()
    x[-1, 3] = inf
    w, up = ((torch.randn(n, k, device=dev, generator=gen) * k ** -0.5).bfloat16() for _ in range(2))
    w[5, 3], w[7, 2], w[9, 4], w[11, 0], w[11, 1], w[n - 1, k - 1], w[n // 2, 100] = inf, -inf, float("nan"), inf, -inf, -inf, inf
    up[5, 9], up[6, 3], up[n // 2 + 1, 5] = -inf, inf, inf

    def run(first, count):
        out = torch.full((count, n), 7.0, device=dev)
        linear = decoder.DecoderLinear(x=x.data_ptr() + 4 * k * first, w=w.data_ptr(), w_up=up.data_ptr() if pair else None, out32=None if pair else out.data_ptr(),
                                       out=out.data_ptr() if pair else None, ldx=k, ldo=n, n=n, k=k)
        assert decoder.lib().qm_decoder_linear_rows(C.byref(linear), 1, count, 1, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return out

    got, want = run(0, rows), torch.cat([run(i, min(8, rows - i)) for i in range(0, rows, 8)])
    assert bool(want.isinf().any()) and bool(want.isnan().any())
    for same in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(same(got), same(want))


@pytest.mark.parametrize("exponent", [-122, -112, -108, -60])
@pytest.mark.parametrize("rows,n,k", [shape[:3] for shape in SPLIT_LINEARS if not shape[3]])
def test_many_fp32_rows_of_small_inputs(decoder, dev, rows, n, k, exponent):
    """Rows of normal numbers down to the smallest keep all their bits: one small input among others does as well."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(rows)
    x = (torch.rand(rows, k, device=dev, generator=gen) + 1) * torch.randint(0, 2, (rows, k), device=dev, generator=gen).mul(2).sub(1).float() * 2.0 ** exponent
    x[rows // 2, k // 2] = 1.0
    w = (torch.randn(n, k, device=dev, generator=gen) * k ** -0.5).bfloat16()
    out = torch.full((rows, n), 7.0, device=dev)
    linear = decoder.DecoderLinear(x=x.data_ptr(), w=w.data_ptr(), out32=out.data_ptr(), ldx=k, ldo=n, n=n, k=k)
    assert decoder.lib().qm_decoder_linear_rows(C.byref(linear), 1, rows, 1, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    want = x.double() @ w.double().T
    # (2-norms: the errors of a chain of k roundings scatter like the root of k: 2^-24 sqrt(2176) = 2.8e-6 at most; twice that)
    assert bool(((out.double() - want).norm(dim=1) <= 6e-6 * want.norm(dim=1)).all())


@pytest.mark.parametrize("rows,n,k,pair,dots", [
    (32, 1024, 3072, False, True), (33, 1024, 3072, False, False), (16, 2048, 6144, False, True), (17, 2048, 6144, False, False),
    (32, 2048, 2048, False, True), (33, 2048, 2048, False, False), (33, 1024, 2048, True, True), (57, 1024, 2048, True, False), (16, 4096, 2048, False, False), (10, 1664, 2176, True, True), (9, 6144, 2048, True, False)])
def test_fp32_rows_that_the_dot_products_end_first(decoder, dev, rows, n, k, pair, dots):
    """Long reductions to few columns stay with the dot products while their blocks fit a round: the bits of eight rows at a time."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn(rows, k, device=dev, generator=gen)
    w, up = ((torch.randn(n, k, device=dev, generator=gen) * k ** -0.5).bfloat16() for _ in range(2))

    def run(first, count):
        out = torch.full((count, n), 7.0, device=dev)
        linear = decoder.DecoderLinear(x=x.data_ptr() + 4 * k * first, w=w.data_ptr(), w_up=up.data_ptr() if pair else None, out32=None if pair else out.data_ptr(),
                                       out=out.data_ptr() if pair else None, ldx=k, ldo=n, n=n, k=k)
        assert decoder.lib().qm_decoder_linear_rows(C.byref(linear), 1, count, 1, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return out

    got, want = run(0, rows), torch.cat([run(i, min(8, rows - i)) for i in range(0, rows, 8)])
    assert torch.equal(got, want) == dots
    assert float((got - want).abs().max()) <= 4e-6 * float(want.abs().max())


@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_many_fp32_rows_into_any_float_address(decoder, dev, pair, shift):
    """Outputs that are no multiple of 16 bytes are the dot products', which store single floats."""
    import torch
    rows, n, k, ldo = 104, 1024, 2048, 1028
    gen = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn(rows, k, device=dev, generator=gen)
    w, up = ((torch.randn(n, k, device=dev, generator=gen) * k ** -0.5).bfloat16() for _ in range(2))

    def run(first, count, shift):
        out = torch.full((count * ldo + 8,), 7.0, device=dev)
        at = out.data_ptr() + 4 * shift
        linear = decoder.DecoderLinear(x=x.data_ptr() + 4 * k * first, w=w.data_ptr(), w_up=up.data_ptr() if pair else None, out32=None if pair else at,
                                       out=at if pair else None, ldx=k, ldo=ldo, n=n, k=k)
        assert decoder.lib().qm_decoder_linear_rows(C.byref(linear), 1, count, 1, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        assert bool((out[:shift] == 7).all()) and bool((out[shift + count * ldo:] == 7).all())
        return out[shift:shift + count * ldo].reshape(count, ldo)

    got, want = run(0, rows, shift), torch.cat([run(i, 8, 0) for i in range(0, rows, 8)])
    assert bool((got[:, n:] == 7).all())
    assert torch.equal(got, want) == (shift != 0)
    assert float((got - want).abs().max()) <= 4e-6 * float(want[:, :n].abs().max())


class ThroughPlanes:
    """The decoder library with fp32 linears of more than eight rows by qm_decoder_linear_rows_planes."""

    def __init__(self, decoder, dev):
        self.decoder, self.dev = decoder, dev

    def __getattr__(self, name):
        return getattr(self.decoder, name)

    def lib(self):
        return self

    def qm_decoder_linear_rows(self, linears, count, rows, f32, stream):
        import torch
        lib = self.decoder.lib()
        if rows <= 8:
            return lib.qm_decoder_linear_rows(linears, count, rows, f32, stream)
        nbytes = lib.qm_decoder_linear_planes_bytes(linears, count, rows)
        planes = torch.full((nbytes // 4 + 4,), float("nan"), device=self.dev)
        assert lib.qm_decoder_linear_rows_planes(linears, count, rows, planes.data_ptr(), nbytes - 1, stream) == -4
        rc = lib.qm_decoder_linear_rows_planes(linears, count, rows, planes.data_ptr(), nbytes, stream)
        torch.cuda.synchronize()
        assert bool(planes[nbytes // 4:].isnan().all())
        return rc


# (the last ones: grids that take blocks of 256 weight rows; a reduction of a single pair of steps; a last row tile of one row and of all but one)
@pytest.mark.parametrize("rows,n,k,pair", SPLIT_LINEARS + [(600, 4112, 128, False), (577, 2176, 384, True), (64, 128, 128, False), (191, 256, 256, True)])
def test_linears_of_fp32_rows_split_beforehand(decoder, dev, rows, n, k, pair):
    """As the linears that split their inputs themselves: bounds against 64 bits, infinities, inputs down to the smallest normal numbers."""
    planes = ThroughPlanes(decoder, dev)
    test_linears_of_many_fp32_rows(planes, dev, rows, n, k, pair)
    test_many_fp32_rows_meet_infinite_weights(planes, dev, rows, n, k, pair)
    if not pair:
        for exponent in (-122, -112, -108, -60):
            test_many_fp32_rows_of_small_inputs(planes, dev, rows, n, k, exponent)


class InnerTypes:
    """The decoder kernels' launchers as the engine calls them: structures of qm_decoder_ops.h, and functions by their C++ names."""

    class Linears(C.Structure):
        pass

    class Planes(C.Structure):
        _fields_ = [("at", C.c_void_p), ("elements", C.c_int64), ("split", C.c_bool)]

    class Cut(C.Structure):
        _fields_ = [("sums", C.c_void_p), ("room", C.c_int64), ("plane", C.c_int64), ("planes", C.c_int)]

    class More(C.Structure):
        _fields_ = [("sums", C.c_void_p), ("plane", C.c_int64), ("planes", C.c_int)]

    def __init__(self, decoder):
        if not hasattr(self.Linears, "_fields_"):
            self.Linears._fields_ = [("group", decoder.DecoderLinear * 3), ("groups", C.c_int), ("rows", C.c_int), ("streaming", C.c_int)]
        handle = C.CDLL(decoder.lib_path())
        self.linears = handle._ZN2qm22launch_decoder_linearsERKNS_15DecLinearParamsEiP12ihipStream_tPNS_12ReductionCutERKNS_11PlaneMemoryE
        self.linears.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
        self.norm = handle._ZN2qm20launch_residual_normERK16qm_residual_normiiP12ihipStream_tRKNS_10MoreOfTermEPt
        self.norm.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]


def upper_parts(x):
    """The three bf16 parts of fp32 numbers, as floats: eight significant bits each, cut off."""
    parts = []
    for _ in range(3):
        upper = (x.view(np.uint32) & 0xffff0000).view(np.float32)
        parts.append(upper)
        x = x - upper
    return parts


@pytest.mark.parametrize("width,ld,rows,pieces", [(1000, 1024, 5, 1), (1024, 1024, 3, 3), (1500, 1536, 2, 1), (4000, 4096, 2, 2), (9000, 9088, 2, 1)])
def test_norms_leave_the_parts_of_their_rows(decoder, dev, width, ld, rows, pieces):
    """A norm that leaves its rows split as well: the rows and the stream with the bits that it has alone, and the parts of those rows, bit for bit; the last
    term in pieces, too."""
    import torch
    inner, gen = InnerTypes(decoder), torch.Generator(device=dev).manual_seed(width)
    x, y, w = [torch.randn(n, ld, device=dev, generator=gen) for n in (rows, rows, 1)]
    more = torch.randn(2, rows, ld, device=dev, generator=gen)
    for t in (x, y, w, more):
        t[..., width:] = 0.0
    left = []
    for split in (False, True):
        x_out, h = torch.full((rows, ld), 7.0, device=dev), torch.full((rows, ld), 7.0, device=dev)
        parts = torch.full((3 * rows * ld + 8,), 7.0, device=dev, dtype=torch.bfloat16)
        op = decoder.ResidualNorm(x_in=x.data_ptr(), x_out=x_out.data_ptr(), norm_w=w.data_ptr(), h=h.data_ptr(), ld_h=ld, width=width, eps=1e-5, terms=1)
        op.term[0] = decoder.ResidualTerm(y=y.data_ptr(), ld=ld, scale=0.5)
        pending = inner.More(more.data_ptr() if pieces > 1 else None, rows * ld, pieces - 1)
        assert inner.norm(C.addressof(op), rows, 1, torch.cuda.current_stream().cuda_stream, C.addressof(pending), parts.data_ptr() if split else None) == 0
        left.append([get(t) for t in (x_out, h, parts)])
    (x_alone, h_alone, untouched), (x_out, h, parts) = left
    assert np.array_equal(x_out, x_alone) and np.array_equal(h, h_alone) and np.all(untouched == 7.0) and np.all(parts[3 * rows * ld:] == 7.0)
    want = (x.double() + 0.5 * (y.double() + more[:pieces - 1].double().sum(0))).cpu().numpy()
    assert np.abs(x_out - want).max() <= 1e-6 * np.abs(want).max()
    for got, part in zip(parts[:3 * rows * ld].reshape(3, rows, ld), upper_parts(h)):
        assert np.array_equal(got, part)


@pytest.mark.parametrize("rows,sizes,pieces", [(300, [(1024, 1024), (1024, 3072)], 3), (400, [(1024, 1024), (1024, 1024), (1024, 3072)], 2),
                                               (70, [(1024, 3072), (1024, 9216)], 3)])
def test_pieces_of_a_fp32_reduction(decoder, dev, rows, sizes, pieces):
    """The engine's launch with memory for split inputs and for pieces of the last reduction: so many pieces, whose sums come to the linear, and the bits
    of the others as they are without a cut.  A linear whose input is there already, split, takes the parts and not the rows."""
    import torch
    inner, gen = InnerTypes(decoder), torch.Generator(device=dev).manual_seed(rows)
    x = [torch.randn(rows, k, device=dev, generator=gen) for _, k in sizes]
    w = [(torch.randn(n, k, device=dev, generator=gen) * k ** -0.5).bfloat16() for n, k in sizes]
    stream = torch.cuda.current_stream().cuda_stream
    planes = torch.full((3 * rows * sum(k for _, k in sizes),), float("nan"), device=dev, dtype=torch.bfloat16)

    def launch(which, cut, split=False):
        outs = [torch.full((rows, sizes[i][0]), 7.0, device=dev) for i in which]
        p = inner.Linears(groups=len(which), rows=rows)
        for g, (i, out) in enumerate(zip(which, outs)):
            p.group[g] = decoder.DecoderLinear(x=x[i].data_ptr(), w=w[i].data_ptr(), out32=out.data_ptr(), ldx=sizes[i][1], ldo=sizes[i][0], n=sizes[i][0], k=sizes[i][1])
        memory = inner.Planes(planes.data_ptr(), planes.numel(), split)
        assert inner.linears(C.addressof(p), 1, stream, C.addressof(cut) if cut else None, C.addressof(memory)) == 0
        torch.cuda.synchronize()
        return outs

    sizes, every = list(sizes), list(range(len(sizes)))
    n = sizes[-1][0]
    more = torch.full((2, rows, n), float("nan"), device=dev)
    cut = inner.Cut(more.data_ptr(), more.numel(), 0, 0)
    outs = launch(every, cut)
    assert (cut.planes, cut.plane) == (pieces - 1, rows * n)
    assert bool(more[pieces - 1:].isnan().all())
    small = inner.Cut(more.data_ptr(), (pieces - 1) * rows * n - 1, 0, 0)          # no room for them: whole
    uncut = launch(every, small)
    assert small.planes == 0
    for i in every:
        want = x[i].double() @ w[i].double().T
        got = outs[i] + more[:pieces - 1].sum(0) if i == every[-1] else outs[i]
        # (pieces of 1024 to 3072 inputs, each 8e-8 to 9.6e-8 of its own sums, and their sum's roundings)
        assert float((got.double() - want).norm() / want.norm()) <= 1.1e-7
        assert float((uncut[i].double() - want).norm() / want.norm()) <= 1.5e-7
        assert i == every[-1] or torch.equal(outs[i], uncut[i])
    if rows == 400:
        sizes[:] = [(4096, 1024)]
        w[0] = (torch.randn(4096, 1024, device=dev, generator=gen) / 32).bfloat16()
        before = launch([0], None)[0]
        x[0].normal_(generator=gen)
        assert torch.equal(launch([0], None, split=True)[0], before)
        assert not torch.equal(launch([0], None)[0], before)


def test_more_rows_than_a_grid_is_high_are_split_beforehand(decoder, dev):
    import torch
    rows, n, k = 65600, 16, 128
    gen = torch.Generator(device=dev).manual_seed(29)
    x, w = torch.randn(rows, k, device=dev, generator=gen), (torch.randn(n, k, device=dev, generator=gen) * k ** -0.5).bfloat16()
    out = torch.full((rows, n), 7.0, device=dev)
    linear = decoder.DecoderLinear(x=x.data_ptr(), w=w.data_ptr(), out32=out.data_ptr(), ldx=k, ldo=n, n=n, k=k)
    assert ThroughPlanes(decoder, dev).qm_decoder_linear_rows(C.byref(linear), 1, rows, 1, torch.cuda.current_stream().cuda_stream) == 0
    want = x.double() @ w.double().T
    assert float((out.double() - want).abs().max()) <= 2e-6 * float(want.abs().max())


@pytest.mark.parametrize("rows", [70, 300])
def test_three_linears_of_fp32_rows_split_beforehand(decoder, dev, rows):
    """Several linears in one launch, two of them of one input: the bits of one launch each, and where prompts go this way errors no larger than the other
    kernel's."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(rows)
    shapes = [(1024, 1024, 0), (256, 1024, 0), (1040, 3072, 1)]
    x = [torch.randn(rows, k, device=dev, generator=gen) for k in (1024, 3072)]
    w = [(torch.randn(n, k, device=dev, generator=gen) * k ** -0.5).bfloat16() for n, k, _ in shapes]

    def run(library, which):
        outs = [torch.full((rows, shapes[i][0]), 7.0, device=dev) for i in which]
        linears = (decoder.DecoderLinear * len(which))(*[
            decoder.DecoderLinear(x=x[shapes[i][2]].data_ptr(), w=w[i].data_ptr(), out32=out.data_ptr(), ldx=shapes[i][1], ldo=shapes[i][0], n=shapes[i][0], k=shapes[i][1])
            for i, out in zip(which, outs)])
        assert library.lib().qm_decoder_linear_rows(linears, len(which), rows, 1, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return outs

    together, alone, plain_way = run(ThroughPlanes(decoder, dev), [0, 1, 2]), [run(ThroughPlanes(decoder, dev), [i])[0] for i in range(3)], run(decoder, [0, 1, 2])
    for i in range(3):
        assert torch.equal(together[i], alone[i])
        want = x[shapes[i][2]].double() @ w[i].double().T
        errors = [float((got.double() - want).norm() / want.norm()) for got in (together[i], plain_way[i])]
        # (of 70 rows four groups of waves share a reduction, 7.5e-8 of 1024 inputs, and prompts keep to that; here 7.9e-8, as two groups of 300 rows have it.
        # Of the same inputs, 300 x 256 sums and more: both errors scatter by 0.3 %)
        if rows == 300:
            assert errors[0] <= 1.01 * errors[1], errors


ATTENTION = [
    # heads, kv_heads, dim, vdim, chunk, rot_dims
    (4, 2, 16, 16, 50, 8), (3, 3, 24, 40, 37, 24), (5, 1, 36, 20, 64, 10), (6, 2, 64, 64, 200, 16), (2, 1, 136, 144, 300, 64), (8, 2, 128, 128, 256, 128),
    (4, 4, 8, 256, 33, 0), (16, 1, 32, 48, 70, 32), (7, 1, 20, 28, 5, 4),
]


class AttentionCase:
    """Projections of a sequence with a needle: at some positions one far key is made to stand out."""

    def __init__(self, shape, tokens, seed=0):
        self.heads, self.kv, self.dim, self.vdim, self.chunk, self.rot = shape
        rng = np.random.default_rng(seed)
        self.n, self.ld = tokens, self.heads * self.dim + self.kv * (self.dim + self.vdim) + 8
        self.k_at = self.heads * self.dim
        self.v_at = self.k_at + self.kv * self.dim
        self.proj = rng.standard_normal((tokens, self.ld)).astype(np.float32)
        # keys that many queries of their chunk point at: the first and the last of each chunk, one just outside for the next
        q = self.proj[:, :self.k_at].reshape(tokens, self.heads, self.dim)
        for p in range(0, tokens, self.chunk):
            for at in (p, min(p + self.chunk, tokens) - 1):
                self.proj[at, self.k_at:self.v_at] *= 6.0
        q *= 2.0
        self.base, self.scale = 500.0, self.dim ** -0.5

    def want(self, chunk=None):
        p = self.proj.astype(np.float64)
        heads = lambda a, count: a.reshape(self.n, count, -1)
        q = plain.rotate(heads(p[:, :self.k_at], self.heads), 0, self.rot, self.base)
        k = plain.rotate(heads(p[:, self.k_at:self.v_at], self.kv), 0, self.rot, self.base)
        v = heads(p[:, self.v_at:self.v_at + self.kv * self.vdim], self.kv)
        return plain.softmax_attention(q, k, v, self.scale, plain.chunk_visible(self.n, chunk or self.chunk)).reshape(self.n, -1)

    def run(self, decoder, dev, f32, portions, ring=None, rows_only=False, splits=4):
        import torch
        dtype = activation(f32)
        r8 = lambda n: (n + 7) // 8 * 8
        ks, vs, n_out = r8(self.dim), r8(self.vdim), self.heads * self.vdim
        ld_out = (n_out + 127) // 128 * 128
        ring = ring or self.n
        freq = put(self.base ** (-2.0 * np.arange(max(1, self.rot // 2)) / max(1, self.rot)), dev)
        kc = torch.full((self.kv, ring, ks), float("nan"), device=dev, dtype=dtype)
        vc = torch.full((self.kv, ring, vs), float("nan"), device=dev, dtype=dtype)
        proj = put(self.proj, dev)
        most = max(portions)
        per_split = -(-self.chunk // splits)
        ml = torch.zeros(most * self.heads * splits * 2, device=dev)
        acc = torch.zeros(most * self.heads * splits * self.vdim, device=dev)
        q_rot = torch.zeros(most * self.heads * ks, device=dev, dtype=dtype)
        got, at = [], 0
        for rows in portions:
            out = torch.full((rows, ld_out), 7.0, device=dev, dtype=dtype)
            op = decoder.ChunkAttention(proj=proj.data_ptr() + 4 * self.ld * at, frequency=freq.data_ptr(), q_rot=q_rot.data_ptr(), k_cache=kc.data_ptr(),
                                        v_cache=vc.data_ptr(), out=out.data_ptr(),
                                        part=decoder.AttentionPartials(ml.data_ptr(), acc.data_ptr(), self.heads, self.vdim, splits, per_split),
                                        ld_proj=self.ld, ld_out=ld_out, position=at, rows=rows, heads=self.heads, kv_heads=self.kv, dim=self.dim,
                                        vdim=self.vdim, k_stride=ks, v_stride=vs, ring=ring, chunk=self.chunk, rot_dims=self.rot, k_column=self.k_at,
                                        v_column=self.v_at, scale=self.scale, options=1 if rows_only else 0)
            assert decoder.lib().qm_chunk_attention_rows(C.byref(op), int(f32), torch.cuda.current_stream().cuda_stream) == 0
            out = get(out)
            assert np.all(out[:, n_out:] == 0)
            got.append(out[:, :n_out])
            at += rows
        return np.concatenate(got)


@pytest.mark.parametrize("shape", ATTENTION)
def test_chunk_attention(decoder, dev, shape):
    case = AttentionCase(shape, 230)
    want = case.want()
    if shape[4] < 230:       # the inputs tell a chunk from one that is a position longer or shorter
        scale = np.abs(want).max()
        assert min(np.abs(case.want(shape[4] + d) - want).max() for d in (1, -1)) > 0.1 * scale
    cuts = [230], [100, 2, 28, 1, 1, 17, 3, 16, 62], [1] * 8 + [222], [60, 15, 2, 2, 2, 2] + [1] * 60 + [87]
    for portions in cuts:
        close(case.run(decoder, dev, True, portions), want, True, tol32=2e-5)
        for rows_only in (False, True):
            close(case.run(decoder, dev, False, portions, rows_only=rows_only), want, False, tol16=3e-2)


@pytest.mark.parametrize("shape", [ATTENTION[0], ATTENTION[2], ATTENTION[8]])
def test_chunk_attention_over_a_ring(decoder, dev, shape):
    """A ring of chunk + portion - 1 positions: slots are used again while their old keys have just left the chunk."""
    case = AttentionCase(shape, 410, seed=5)
    want = case.want()
    for most in (1, 2, 20, 33):
        portions = [most] * (410 // most) + ([410 % most] if 410 % most else [])
        ring = case.chunk + most - 1
        close(case.run(decoder, dev, True, portions, ring=ring), want, True, tol32=2e-5)
        close(case.run(decoder, dev, False, portions, ring=ring), want, False, tol16=3e-2)


@pytest.mark.parametrize("shape", [(2, 2, 192, 128, 1250, 64), (4, 2, 64, 64, 1300, 16), (3, 1, 128, 120, 1000, 128), (2, 1, 32, 32, 1201, 0), (2, 1, 250, 136, 1290, 6)])
def test_chunk_attention_of_few_blocks_that_walk_far(decoder, dev, shape):
    """Prompts behind 1200 keys and more, whose few blocks take eight waves where these fit, on both sides of that line and with a ring that wraps
    inside a wave's tile; tolerance and plain attention as above."""
    case = AttentionCase(shape, 1290, seed=13)
    want = case.want()
    for portions in ([1290], [1199, 17, 74], [1100, 33, 31, 126]):
        for ring in (1290, min(1290, case.chunk + max(portions) - 1)):
            close(case.run(decoder, dev, False, portions, ring=ring), want, False, tol16=3e-2)


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("heads,kv,dim,vdim,rot", [(4, 2, 64, 64, 64), (16, 8, 128, 128, 128), (3, 1, 24, 8, 16), (2, 1, 256, 136, 0), (36, 9, 64, 40, 8), (1, 1, 8, 8, 8),
                                                   (64, 32, 64, 128, 64), (2, 2, 256, 256, 256)])
def test_chunk_attention_rotates_in_vectors(decoder, dev, heads, kv, dim, vdim, rot, f32):
    """Queries and keys that are turned four channels at a time, and values, as the kernel for any alignment leaves them: the same projections, begun a
    float later in memory."""
    import torch
    rng = np.random.default_rng(heads + dim)
    rows, position, ring = 19, 5, 21
    k_at = heads * dim + 4
    v_at = k_at + kv * dim + 4
    ld = v_at + kv * vdim
    flat = rng.standard_normal(rows * ld).astype(np.float32)
    freq = put(700.0 ** (-2.0 * np.arange(max(1, rot // 2)) / max(1, rot)), dev)
    left = []
    for shift in (0, 1):
        proj = torch.zeros(rows * ld + 4, device=dev)
        proj[shift:shift + rows * ld] = put(flat, dev)
        caches = [torch.full(s, float("nan"), device=dev, dtype=activation(f32)) for s in ((rows, heads, dim), (kv, ring, dim), (kv, ring, vdim))]
        out = torch.zeros((rows, (heads * vdim + 127) // 128 * 128), device=dev, dtype=activation(f32))
        ml, acc = torch.zeros(rows * heads * 2, device=dev), torch.zeros(rows * heads * vdim, device=dev)
        op = decoder.ChunkAttention(proj=proj.data_ptr() + 4 * shift, frequency=freq.data_ptr(), q_rot=caches[0].data_ptr(), k_cache=caches[1].data_ptr(),
                                    v_cache=caches[2].data_ptr(), out=out.data_ptr(), part=decoder.AttentionPartials(ml.data_ptr(), acc.data_ptr(), heads, vdim, 1, 3),
                                    ld_proj=ld, ld_out=out.shape[1], position=position, rows=rows, heads=heads, kv_heads=kv, dim=dim, vdim=vdim, k_stride=dim,
                                    v_stride=vdim, ring=ring, chunk=3, rot_dims=rot, k_column=k_at, v_column=v_at, scale=dim ** -0.5)
        # (a chunk of three positions: the two behind it in the ring stay as they were)
        assert decoder.lib().qm_chunk_attention_rows(C.byref(op), int(f32), torch.cuda.current_stream().cuda_stream) == 0
        left.append(caches)
    for got, want in zip(*left):
        assert np.array_equal(get(got), get(want), equal_nan=True)     # the same products and sums (a zero behind the turning channels keeps its sign in vectors)


@pytest.mark.parametrize("scale", [0.0, -0.3, 3.0])
def test_chunk_attention_of_other_scales(decoder, dev, scale):
    """Scores that are all equal, whose order the factor turns round, and that run far apart, so that a row's largest rises again and again: against the
    row kernel, which reads the same rounded queries and keys (at a scale of 3 their rounding alone moves a score by up to some 3 x 16 x 16 x 2^-8 = 3)."""
    case = AttentionCase((4, 2, 64, 64, 200, 16), 230, seed=17)
    case.scale = scale
    got, want = case.run(decoder, dev, False, [230]), case.run(decoder, dev, False, [230], rows_only=True)
    assert np.abs(got - want).max() <= 2e-2 * np.abs(want).max()


@pytest.mark.parametrize("exponent", [20, 32, 48])
@pytest.mark.parametrize("heads,kv,dim,vdim", [(4, 2, 64, 64), (2, 1, 192, 128)])
def test_chunk_attention_of_large_scores(decoder, dev, heads, kv, dim, vdim, exponent):
    """Finite scores around 2^exponent, of which an fp32 rounding alone comes to many powers of two: a row is the value of its largest score.  Queries and
    keys are bf16 numbers that do not turn, and two scores of a row nearer to each other than fp32 tells apart do not occur."""
    case = AttentionCase((heads, kv, dim, vdim, 200, 0), 230, seed=19)
    case.proj = cases.bf16(case.proj)
    case.proj[:, :case.v_at] *= 2.0 ** (exponent // 2)
    close(case.run(decoder, dev, False, [230]), case.want(), False)


def test_chunk_attention_of_values_near_the_largest(decoder, dev):
    """A key whose score is 2^6.5 times the others' in powers of two, with a value of 2^123, behind 128 keys that its wave has partly seen: weights are at
    most one on the way, and so no sum leaves the range that the result is in."""
    case = AttentionCase((1, 1, 32, 32, 300, 0), 300)
    case.scale = 1.0
    case.proj[:] = 0.0
    case.proj[:, 0] = 1.0
    case.proj[128, case.k_at] = 4.5
    case.proj[128, case.v_at:case.v_at + 32] = 2.0 ** 123
    close(case.run(decoder, dev, False, [300]), case.want(), False)


def test_chunk_attention_of_more_query_rows_than_a_grid_is_high(decoder, dev):
    """33 312 rows of 63 query heads on one key head are 65 583 blocks of 32 query rows: two layers of a grid, with a block too many."""
    import torch
    rows, heads, dim, chunk = 33312, 63, 8, 32
    gen = torch.Generator(device=dev).manual_seed(23)
    ld = heads * dim + 2 * dim
    proj = torch.randn(rows, ld, device=dev, generator=gen).bfloat16().float()
    k, v, q_rot = [torch.full((n,), float("nan"), device=dev, dtype=torch.bfloat16) for n in (rows * dim, rows * dim, rows * heads * dim)]
    out = torch.full((rows, heads * dim), 7.0, device=dev, dtype=torch.bfloat16)
    ml, acc = torch.empty(rows * heads * 2, device=dev), torch.empty(rows * heads * dim, device=dev)
    op = decoder.ChunkAttention(proj=proj.data_ptr(), q_rot=q_rot.data_ptr(), k_cache=k.data_ptr(), v_cache=v.data_ptr(), out=out.data_ptr(),
                                part=decoder.AttentionPartials(ml.data_ptr(), acc.data_ptr(), heads, dim, 1, chunk), ld_proj=ld, ld_out=heads * dim, rows=rows,
                                heads=heads, kv_heads=1, dim=dim, vdim=dim, k_stride=dim, v_stride=dim, ring=rows, chunk=chunk, k_column=heads * dim,
                                v_column=heads * dim + dim, scale=dim ** -0.5)
    assert decoder.lib().qm_chunk_attention_rows(C.byref(op), 0, torch.cuda.current_stream().cuda_stream) == 0
    parts = proj.double().reshape(rows // chunk, chunk, ld)
    q, keys, values = parts[..., :heads * dim].reshape(-1, chunk, heads, dim), parts[..., heads * dim:heads * dim + dim], parts[..., heads * dim + dim:]
    hidden = torch.ones(chunk, chunk, device=dev, dtype=torch.bool).triu(1)
    for first in range(0, rows // chunk, 205):
        at = slice(first, first + 205)
        s = (q[at].unsqueeze(3) * keys[at].unsqueeze(1).unsqueeze(1)).sum(-1) * dim ** -0.5                # [chunks][row][head][key]
        p = s.permute(0, 2, 1, 3).masked_fill(hidden, -float("inf")).softmax(-1)                           # [chunks][head][row][key]
        want = (p.unsqueeze(-1) * values[at].unsqueeze(1).unsqueeze(1)).sum(-2).permute(0, 2, 1, 3).reshape(-1, heads * dim)
        close(get(out[first * chunk:first * chunk + want.shape[0]]), want.cpu().numpy(), False)


def test_two_attention_kernels_agree(decoder, dev):
    case = AttentionCase((8, 4, 64, 64, 512, 32), 700, seed=9)
    a, b = case.run(decoder, dev, False, [700]), case.run(decoder, dev, False, [700], rows_only=True)
    assert np.abs(a - b).max() <= 2e-2 * np.abs(b).max()


@pytest.mark.parametrize("shape", [(16, 8, 64, 64, 512, 64), (5, 1, 36, 20, 64, 10), (3, 3, 24, 40, 37, 24), (8, 2, 128, 128, 256, 128), (4, 2, 65, 6, 19, 2)])
def test_fp32_attention_of_many_rows_against_the_row_kernel(decoder, dev, shape):
    """Both kernels of fp32 rows stand as close to 64 bits, around the 16 query rows of a block, the 16 keys of a step and
    the end of a chunk; and a row does not know the values of positions that it does not see, whatever they are."""
    worst = {False: [], True: []}
    for rows in (16, 17, 31, 33, 65, 130, 230):
        case = AttentionCase(shape, rows, seed=rows)
        want = case.want()
        for rows_only in (False, True):
            got = case.run(decoder, dev, True, [rows], rows_only=rows_only)
            close(got, want, True, tol32=2e-5)
            worst[rows_only].append(np.sqrt(np.mean((got - want) ** 2)))
    # (over 24 draws of five shapes the ratio was 0.98 to 1.02, and one draw's scatters by 0.07: seven draws' mean by 0.03; five times that)
    assert np.mean(worst[False]) <= 1.15 * np.mean(worst[True])
    whole = AttentionCase(shape, 100, seed=3)
    plain_result = whole.run(decoder, dev, True, [100])
    for at, what in ((99, np.inf), (50, np.nan), (17, -np.inf), (18, np.inf)):
        broken = AttentionCase(shape, 100, seed=3)
        broken.proj[at, broken.v_at:broken.v_at + broken.vdim] = what
        got = broken.run(decoder, dev, True, [100])
        sees = np.array([at <= i < at // whole.chunk * whole.chunk + whole.chunk for i in range(100)])
        assert np.abs(got[~sees] - plain_result[~sees]).max(initial=0.0) <= 4e-6 * np.abs(plain_result).max()
        assert not np.isfinite(got[at]).all()


@pytest.mark.parametrize("shape", [(4, 2, 40, 40, 50, 8), (3, 3, 24, 40, 37, 8), (2, 1, 72, 16, 60, 8), (4, 2, 64, 64, 50, 8)])
def test_fp32_attention_of_many_rows_meets_infinite_keys(decoder, dev, shape):
    """An infinity in a key's last channel decides by the query's sign: a score of -inf is a weight of zero, one of +inf leaves no number."""
    case = AttentionCase(shape, 100, seed=11)
    for at, head in ((3, 0), (61, shape[1] - 1)):
        case.proj[at, case.k_at + head * case.dim + case.dim - 1] = np.inf
    with np.errstate(invalid="ignore"):
        want = case.want()
    got = case.run(decoder, dev, True, [100])
    finite = np.isfinite(want)
    assert not finite.all() and finite[61:case.chunk * 2].any()
    assert np.array_equal(np.isfinite(got), finite)
    close(got[finite], want[finite], True, tol32=2e-5)


@pytest.mark.parametrize("shape,before,splits,here", [
    ((2, 1, 128, 128, 1024, 64), 1000, 1, False), ((4, 1, 64, 64, 2048, 64), 2000, 16, False), ((4, 1, 64, 64, 2048, 64), 2000, 1, True),
    ((16, 8, 64, 64, 512, 64), 200, 1, True), ((16, 8, 64, 64, 512, 64), 200, 4, True)])
def test_long_chunks_of_few_fp32_rows_take_the_row_kernel(decoder, dev, shape, before, splits, here):
    """Where few blocks would walk a long chunk that the caller cut, or one of wide heads, the row kernel ends first and is taken."""
    case = AttentionCase(shape, before + 16, seed=4)
    got, rows_kernel = (case.run(decoder, dev, True, [before, 16], splits=splits, rows_only=only)[before:] for only in (False, True))
    close(got, rows_kernel, True, tol32=2e-5)
    assert np.array_equal(got, rows_kernel) != here


@pytest.mark.parametrize("chunked", [False, True])
@pytest.mark.parametrize("heads,dim,vdim", [(3, 16, 24), (2, 20, 36), (1, 48, 16), (4, 64, 128), (2, 132, 200), (1, 256, 256), (2, 7, 9)])
def test_decay_attention(decoder, dev, chunked, heads, dim, vdim):
    import torch
    rng = np.random.default_rng(dim)
    n = 230
    decay = np.array([0.999, 1.0, 0.3, 0.0][:heads])
    ld = heads * (2 * dim + vdim) + 12
    proj = rng.standard_normal((n, ld)).astype(np.float32)
    k_at, v_at = heads * dim + 4, 2 * heads * dim + 8
    part = lambda at, count, size: plain.silu(proj[:, at:at + count * size].astype(np.float64)).reshape(n, count, size)
    want, state = plain.decayed_linear_attention(part(0, heads, dim), part(k_at, heads, dim), part(v_at, heads, vdim), decay)
    powers = put(np.power(decay[:, None], np.arange(decoder.DECAY_POWERS)[None]).astype(np.float32), dev)
    pd = put(proj, dev)
    for portions in ([n], [100, 2, 28, 1, 17, 64, 16, 2], [1] * 20 + [65, 145]):
        s = torch.zeros((heads, dim, vdim), device=dev)
        got, at = [], 0
        for rows in portions:
            out = torch.full((rows, heads * vdim), 7.0, device=dev)
            floats = decoder.lib().qm_decay_attention_scratch_floats(rows, heads, dim, vdim)
            assert (floats > 0) == (rows >= 16)
            scratch = torch.full((max(1, floats),), float("nan"), device=dev)
            op = decoder.DecayAttention(proj=pd.data_ptr() + 4 * ld * at, powers=powers.data_ptr(), state=s.data_ptr(), out=out.data_ptr(),
                                        scratch=scratch.data_ptr() if chunked else None, ld_proj=ld, scratch_floats=floats, rows=rows, heads=heads, dim=dim,
                                        vdim=vdim, q_column=0, k_column=k_at, v_column=v_at)
            assert decoder.lib().qm_decay_attention_rows(C.byref(op), torch.cuda.current_stream().cuda_stream) == 0
            got.append(get(out))
            at += rows
        close(np.concatenate(got), want.reshape(n, -1), True, tol32=5e-6)
        close(get(s), state, True, tol32=5e-6)


@pytest.mark.parametrize("heads,dim,vdim,rows", [(8, 20, 200, 573), (6, 64, 129, 961), (16, 132, 72, 530), (8, 128, 256, 512), (8, 128, 256, 513),
                                                   (12, 64, 192, 700), (16, 20, 66, 1800)])
def test_decay_attention_in_wide_blocks(decoder, dev, heads, dim, vdim, rows):
    """Passes of around and of more than 256 blocks of 64 value channels, which blocks of 128 take over, and past one round of those."""
    import torch
    rng = np.random.default_rng(rows)
    decay = np.array([0.999, 1.0, 0.3, 0.0, 0.9, 0.99, 0.5, 0.75] * 2)[:heads]
    proj = rng.standard_normal((rows, heads * (2 * dim + vdim))).astype(np.float32)
    part = lambda at, count, size: plain.silu(proj[:, at:at + count * size].astype(np.float64)).reshape(rows, count, size)
    want, state = plain.decayed_linear_attention(part(0, heads, dim), part(heads * dim, heads, dim), part(2 * heads * dim, heads, vdim), decay)
    powers = put(np.power(decay[:, None], np.arange(decoder.DECAY_POWERS)[None]).astype(np.float32), dev)
    pd, s, out = put(proj, dev), torch.zeros((heads, dim, vdim), device=dev), torch.full((rows, heads * vdim), 7.0, device=dev)
    floats = decoder.lib().qm_decay_attention_scratch_floats(rows, heads, dim, vdim)
    scratch = torch.full((floats,), float("nan"), device=dev)
    op = decoder.DecayAttention(proj=pd.data_ptr(), powers=powers.data_ptr(), state=s.data_ptr(), out=out.data_ptr(), scratch=scratch.data_ptr(),
                                ld_proj=proj.shape[1], scratch_floats=floats, rows=rows, heads=heads, dim=dim, vdim=vdim, q_column=0,
                                k_column=heads * dim, v_column=2 * heads * dim)
    assert decoder.lib().qm_decay_attention_rows(C.byref(op), torch.cuda.current_stream().cuda_stream) == 0
    close(get(out), want.reshape(rows, -1), True, tol32=5e-6)          # (as in the smaller passes: the sums are the same)
    close(get(s), state, True, tol32=5e-6)


@pytest.mark.parametrize("chunked", [False, True])
@pytest.mark.parametrize("heads,dim,rank", [(3, 16, 5), (2, 20, 16), (1, 48, 64), (4, 64, 8), (2, 100, 33), (2, 128, 64), (1, 160, 300), (1, 256, 24)])
def test_general_delta(decoder, dev, chunked, heads, dim, rank):
    import torch
    rng = np.random.default_rng(dim + rank)
    n, every = 170, heads * dim
    ld = 4 * every + rank + 8
    proj = rng.standard_normal((n, ld)).astype(np.float32)
    proj[50:60, every:2 * every] = proj[40:50, every:2 * every]          # keys that come back
    columns = dict(r_column=0, k_column=every, v_column=2 * every, a_column=3 * every, z_column=4 * every)
    w2 = (rng.standard_normal((rank, every)) * 2 * rank ** -0.5).astype(np.float32)
    w0, bias = (rng.standard_normal(every) * 3 - 2).astype(np.float32), rng.standard_normal(every).astype(np.float32)
    p = proj.astype(np.float64)
    part = lambda name: p[:, columns[name]:columns[name] + every].reshape(n, heads, dim)
    w = np.exp(-np.exp(-0.5) * plain.sigmoid(np.tanh(p[:, 4 * every:4 * every + rank]) @ w2 + w0)).reshape(n, heads, dim)
    a = plain.sigmoid(part("a_column") + bias.reshape(heads, dim))
    want, state = plain.generalized_delta(part("r_column"), w, part("k_column"), part("v_column"), a)
    d = [put(v, dev) for v in (proj, w2, w0, bias)]
    for portions in ([n], [70, 2, 28, 1, 16, 32, 21], [1] * 12 + [33, 125]):
        s = torch.zeros((heads, dim, dim), device=dev)
        got, at = [], 0
        for rows in portions:
            out = torch.full((rows, every), 7.0, device=dev)
            floats = decoder.lib().qm_general_delta_scratch_floats(rows, heads, dim)
            scratch = torch.full((max(1, floats),), float("nan"), device=dev)
            op = decoder.GeneralDelta(proj=d[0].data_ptr() + 4 * ld * at, w2=d[1].data_ptr(), w0=d[2].data_ptr(), a_bias=d[3].data_ptr(), state=s.data_ptr(),
                                      out=out.data_ptr(), scratch=scratch.data_ptr() if chunked else None, ld_proj=ld, scratch_floats=floats, rows=rows,
                                      heads=heads, dim=dim, rank=rank, unit_eps=1e-6, **columns)
            assert decoder.lib().qm_general_delta_rows(C.byref(op), torch.cuda.current_stream().cuda_stream) == 0
            got.append(get(out))
            at += rows
        close(np.concatenate(got), want.reshape(n, -1), True, tol32=2e-5)
        close(get(s), state, True, tol32=2e-5)


@pytest.mark.parametrize("heads,dim,rank,rows", [(33, 20, 7, 530), (35, 64, 36, 513), (32, 16, 4, 512), (32, 16, 3, 545)])
def test_general_delta_in_many_blocks(decoder, dev, heads, dim, rank, rows):
    """Passes around 512 blocks and more of small heads, which ask for a chunk's rows as they use them."""
    import torch
    rng = np.random.default_rng(rows)
    every = heads * dim
    proj = rng.standard_normal((rows, 4 * every + rank)).astype(np.float32)
    columns = dict(r_column=0, k_column=every, v_column=2 * every, a_column=3 * every, z_column=4 * every)
    w2 = (rng.standard_normal((rank, every)) * 2 * rank ** -0.5).astype(np.float32)
    w0, bias = (rng.standard_normal(every) * 3 - 2).astype(np.float32), rng.standard_normal(every).astype(np.float32)
    p = proj.astype(np.float64)
    part = lambda name: p[:, columns[name]:columns[name] + every].reshape(rows, heads, dim)
    w = np.exp(-np.exp(-0.5) * plain.sigmoid(np.tanh(p[:, 4 * every:]) @ w2 + w0)).reshape(rows, heads, dim)
    a = plain.sigmoid(part("a_column") + bias.reshape(heads, dim))
    want, state = plain.generalized_delta(part("r_column"), w, part("k_column"), part("v_column"), a)
    d = [put(v, dev) for v in (proj, w2, w0, bias)]
    s, out = torch.zeros((heads, dim, dim), device=dev), torch.full((rows, every), 7.0, device=dev)
    floats = decoder.lib().qm_general_delta_scratch_floats(rows, heads, dim)
    scratch = torch.full((floats,), float("nan"), device=dev)
    op = decoder.GeneralDelta(proj=d[0].data_ptr(), w2=d[1].data_ptr(), w0=d[2].data_ptr(), a_bias=d[3].data_ptr(), state=s.data_ptr(), out=out.data_ptr(),
                              scratch=scratch.data_ptr(), ld_proj=proj.shape[1], scratch_floats=floats, rows=rows, heads=heads, dim=dim, rank=rank,
                              unit_eps=1e-6, **columns)
    assert decoder.lib().qm_general_delta_rows(C.byref(op), torch.cuda.current_stream().cuda_stream) == 0
    close(get(out), want.reshape(rows, -1), True, tol32=2e-5)          # (as in the smaller passes)
    close(get(s), state, True, tol32=2e-5)


@pytest.mark.parametrize("chunked", [False, True])
@pytest.mark.parametrize("heads,dim,vdim,rot_dims", [(3, 16, 24, 16), (2, 20, 36, 6), (1, 48, 16, 0), (4, 64, 128, 64), (2, 132, 200, 130), (2, 256, 64, 256)])
def test_retention(decoder, dev, chunked, heads, dim, vdim, rot_dims):
    """The decayed attention with rotated queries and keys, scaled keys and plain values."""
    import torch
    rng = np.random.default_rng(dim)
    n, base = 230, 700.0
    decay = np.array([0.999, 1.0, 0.3, 0.0][:heads])
    ld = heads * (2 * dim + vdim) + 12
    proj = rng.standard_normal((n, ld)).astype(np.float32)
    k_at, v_at = heads * dim + 4, 2 * heads * dim + 8
    proj[3, k_at:k_at + heads * dim] *= 30.0                          # an early key that later queries see through the decay
    part = lambda at, count, size: proj[:, at:at + count * size].astype(np.float64).reshape(n, count, size)
    q, k, v = part(0, heads, dim), part(k_at, heads, dim), part(v_at, heads, vdim)
    want = plain.retention(q, k, v, decay, {"dims": rot_dims, "base": base}).reshape(n, -1)
    powers = put(np.power(decay[:, None], np.arange(decoder.DECAY_POWERS)[None]).astype(np.float32), dev)
    frequency = put(base ** (-2.0 * np.arange(max(1, rot_dims // 2)) / max(1, rot_dims)), dev)
    for portions in ([n], [100, 2, 28, 1, 17, 64, 16, 2], [1] * 20 + [65, 145]):
        pd = put(proj, dev)                                           # (rotated in place)
        s = torch.zeros((heads, dim, vdim), device=dev)
        got, at = [], 0
        for rows in portions:
            out = torch.full((rows, heads * vdim), 7.0, device=dev)
            floats = decoder.lib().qm_decay_attention_scratch_floats(rows, heads, dim, vdim)
            scratch = torch.full((max(1, floats),), float("nan"), device=dev)
            where = torch.tensor([at], dtype=torch.int32, device=dev)
            op = decoder.DecayAttention(proj=pd.data_ptr() + 4 * ld * at, powers=powers.data_ptr(), state=s.data_ptr(), out=out.data_ptr(),
                                        scratch=scratch.data_ptr() if chunked else None, frequency=frequency.data_ptr(), ld_proj=ld, scratch_floats=floats,
                                        rows=rows, heads=heads, dim=dim, vdim=vdim, q_column=0, k_column=k_at, v_column=v_at, options=decoder.DECAY_ROTARY,
                                        rot_dims=rot_dims, position=at, k_scale=dim ** -0.5)
            if rows == 1:
                op.position, op.position_dev = 0, where.data_ptr()
            assert decoder.lib().qm_decay_attention_rows(C.byref(op), torch.cuda.current_stream().cuda_stream) == 0
            got.append(get(out))
            at += rows
        close(np.concatenate(got), want, True, tol32=5e-6)


LATENT = [
    # heads, dim, rot_dim, vdim, kv_rank, scaling
    (3, 16, 8, 24, 40, None), (7, 48, 12, 40, 64, (3.0, 100, 20.0, 1.5)), (5, 20, 6, 28, 100, None), (16, 64, 32, 64, 256, None), (17, 128, 64, 128, 512, None),
    (1, 33, 10, 17, 300, (4.0, 50, 8.0, 0.5)), (2, 40, 64, 72, 128, None), (2, 200, 80, 24, 560, None), (2, 16, 70, 300, 96, None), (40, 8, 2, 8, 24, None),
]


class LatentCase:
    """Projections of a sequence; some latents stand out so that single keys far away, at the edges of passes and tiles, decide."""

    def __init__(self, shape, tokens, seed=0):
        self.heads, self.dim, self.rot, self.vdim, self.rank, scaling = shape
        rng = np.random.default_rng(seed)
        self.n, self.base = tokens, 900.0
        self.scaling = dict(zip(("factor", "original", "fast", "slow"), scaling)) if scaling else None
        self.per_head = self.dim + self.rot
        self.proj = rng.standard_normal((tokens, 20 + self.rank + self.rot + 8)).astype(np.float32)          # 20 columns of a query latent
        self.kv_at = 20 + 4
        self.q = (2.0 * rng.standard_normal((tokens, self.heads * self.per_head + 4))).astype(np.float32)
        self.kv_norm = (1 + 0.2 * rng.standard_normal(self.rank)).astype(np.float32)
        self.q_norm = (1 + 0.2 * rng.standard_normal(20)).astype(np.float32)
        for at in (0, 1, 63, 64, 127, 128, tokens - 40):
            self.proj[at, self.kv_at + self.rank:self.kv_at + self.rank + self.rot] *= 4.0                   # (the latent itself is normed)
        self.up_k = cases.bf16(rng.standard_normal((self.heads * self.dim, self.rank)) * self.rank ** -0.5)
        self.up_v = cases.bf16(rng.standard_normal((self.heads * self.vdim, self.rank)) * self.rank ** -0.5)
        self.scale, self.eps = self.per_head ** -0.5, 0.01
        self.spec = {"heads": self.heads, "dim": self.dim, "rot_dim": self.rot, "vdim": self.vdim, "kv_rank": self.rank, "scale": self.scale,
                     "rot": {"base": self.base, "dims": self.rot, "scaling": self.scaling}}

    def kept(self):
        p = self.proj[:, self.kv_at:self.kv_at + self.rank + self.rot].astype(np.float64)
        return plain.latent_of(p, self.spec, np.eye(self.rank + self.rot), self.kv_norm.astype(np.float64), self.eps)

    def want(self):
        q = self.q[:, :self.heads * self.per_head].astype(np.float64).reshape(self.n, self.heads, self.per_head)
        return plain.latent_attention(q, *self.kept(), self.up_k.astype(np.float64), self.up_v.astype(np.float64), self.spec).reshape(self.n, -1)

    def run(self, decoder, dev, f32, portions, rows_only=False, splits=5):
        import torch
        lib, dtype = decoder.lib(), activation(f32)
        stream = torch.cuda.current_stream().cuda_stream
        up128 = lambda n: (n + 127) // 128 * 128
        ld, key_stride, n_out = up128(self.rank), (self.rot + 7) // 8 * 8, self.heads * self.vdim
        ld_out = up128(n_out)
        v_row = (self.heads * self.dim + 7) // 8 * 8
        up_rows = up128(v_row + n_out)
        up = np.zeros((up_rows, ld), np.float32)
        up[:self.heads * self.dim, :self.rank] = self.up_k
        up[v_row:v_row + n_out, :self.rank] = self.up_v
        up = put(up, dev, torch.bfloat16)
        frequencies, magnitude = plain.yarn(self.rot, self.base, self.scaling)
        freq, proj, q = put(frequencies, dev), put(self.proj, dev), put(self.q, dev)
        kv_norm, q_norm = put(self.kv_norm, dev), put(self.q_norm, dev)
        latent = torch.full((self.n, ld), float("nan"), device=dev, dtype=dtype)
        keys = torch.full((self.n, key_stride), float("nan"), device=dev, dtype=dtype)
        most, stride = max(portions), lib.qm_latent_query_stride(self.rank, self.rot)
        q_scratch = torch.full((most * self.heads * stride,), float("nan"), device=dev, dtype=dtype)
        ml = torch.full((most * self.heads * splits * 2,), float("nan"), device=dev)
        acc = torch.full((most * self.heads * splits * self.rank,), float("nan"), device=dev)
        nbytes = lib.qm_latent_expanded_bytes(self.n, self.heads, self.dim, self.rot, self.vdim, up_rows)
        expanded = torch.full((nbytes // 2,), float("nan"), device=dev, dtype=torch.bfloat16)
        got, norms, at = [], [], 0
        for rows in portions:
            where = torch.tensor([at], dtype=torch.int32, device=dev)
            latent_q = torch.full((rows, 128), 7.0, device=dev, dtype=dtype)
            keep = decoder.LatentRows(proj=proj.data_ptr() + 4 * self.proj.shape[1] * at, q_norm=q_norm.data_ptr(), kv_norm=kv_norm.data_ptr(),
                                      frequency=freq.data_ptr(), q_latent=latent_q.data_ptr(), latent_cache=latent.data_ptr(), key_cache=keys.data_ptr(),
                                      ld_proj=self.proj.shape[1], ld_q=128, ld_latent=ld, position=at, rows=rows, q_rank=20, kv_rank=self.rank,
                                      rot_dim=self.rot, key_stride=key_stride, q_column=0, kv_column=self.kv_at, eps=self.eps, magnitude=magnitude)
            assert lib.qm_latent_rows_norm(C.byref(keep), int(f32), stream) == 0
            norms.append(get(latent_q))
            out = torch.full((rows, ld_out), 7.0, device=dev, dtype=dtype)
            op = decoder.LatentAttention(q=q.data_ptr() + 4 * self.q.shape[1] * at, frequency=freq.data_ptr(), up_k=up.data_ptr(),
                                         up_v=up.data_ptr() + 2 * v_row * ld, latent_cache=latent.data_ptr(), key_cache=keys.data_ptr(), out=out.data_ptr(),
                                         q_scratch=q_scratch.data_ptr(), ml=ml.data_ptr(), acc=acc.data_ptr(), expanded=expanded.data_ptr(),
                                         ld_query=self.q.shape[1], ld_latent=ld, ld_out=ld_out, expanded_bytes=nbytes, position=at, rows=rows,
                                         heads=self.heads, dim=self.dim, rot_dim=self.rot, vdim=self.vdim, kv_rank=self.rank, key_stride=key_stride,
                                         splits=splits, up_rows=up_rows, up_v_row=v_row, options=decoder.ATTENTION_ROWS if rows_only else 0,
                                         scale=self.scale, magnitude=magnitude)
            if rows == 1:
                op.position, op.position_dev = 0, where.data_ptr()
            assert lib.qm_latent_attention_rows(C.byref(op), int(f32), stream) == 0
            out = get(out)
            assert np.all(out[:, n_out:] == 0)
            got.append(out[:, :n_out])
            at += rows
        return np.concatenate(got), np.concatenate(norms), get(latent), get(keys)


@pytest.mark.parametrize("shape", LATENT)
def test_latent_attention(decoder, dev, shape):
    case = LatentCase(shape, 230)
    want, (latent, key_part) = case.want(), case.kept()
    q_latent = plain.rms_norm(case.proj[:, :20].astype(np.float64), case.q_norm, case.eps)
    for portions in ([230], [100, 2, 28, 1, 1, 17, 3, 16, 62], [1] * 8 + [222], [60, 15, 2, 2, 2, 2] + [1] * 60 + [87]):
        got, norms, c, k = case.run(decoder, dev, True, portions)
        close(got, want, True, tol32=2e-5)
        close(norms[:, :20], q_latent, True, tol32=3e-6)
        close(c[:, :case.rank], latent, True, tol32=3e-6)
        close(k[:, :case.rot], key_part, True, tol32=3e-6)
        assert np.all(norms[:, 20:] == 0) and np.all(c[:, case.rank:] == 0) and np.all(k[:, case.rot:] == 0)
        for rows_only in (False, True):
            got, norms, c, k = case.run(decoder, dev, False, portions, rows_only=rows_only)
            close(got, want, False, tol16=3e-2)
            close(c[:, :case.rank], latent, False)


@pytest.mark.parametrize("splits", [1, 2, 32, 64])
def test_latent_attention_splits(decoder, dev, splits):
    case = LatentCase((6, 24, 8, 16, 72, None), 700, seed=2)
    want = case.want()
    portions = [570, 1, 1, 5] + [1] * 70 + [15, 38]
    close(case.run(decoder, dev, True, portions, splits=splits)[0], want, True, tol32=2e-5)
    for rows_only in (False, True):
        close(case.run(decoder, dev, False, portions, splits=splits, rows_only=rows_only)[0], want, False, tol16=3e-2)


def test_many_positions_are_expanded_in_several_linears(decoder, dev):
    case = LatentCase((2, 16, 8, 16, 32, None), 4400, seed=3)
    close(case.run(decoder, dev, False, [2100, 2300])[0], case.want(), False, tol16=3e-2)


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("rows", [1, 2, 5, 16, 40, 300])
@pytest.mark.parametrize("experts,top,width,ff", [(9, 3, 200, 72), (1, 1, 128, 128), (5, 5, 100, 200), (70, 6, 130, 40), (300, 3, 128, 96), (3, 1, 256, 384)])
def test_experts(decoder, dev, f32, rows, experts, top, width, ff):
    import torch
    rng = np.random.default_rng(experts + rows)
    up128 = lambda n: (n + 127) // 128 * 128
    wp, fp = up128(width), up128(ff)
    x = cases.bf16(rng.standard_normal((rows, width)))
    router = rng.standard_normal((experts, width)) * width ** -0.5
    logits = (x @ router.T).astype(np.float32)
    if experts > 1:
        logits[0, 1] = logits[0, 0]                                   # equals: the lower number first
    if rows > 30:
        logits[:, -1] += 4.0                                          # an expert that nearly every row takes
    gate, up, down = (cases.bf16(rng.standard_normal(s) * s[2] ** -0.5) for s in ((experts, ff, width), (experts, ff, width), (experts, width, ff)))

    def padded(a, *shape):
        out = np.zeros(shape, np.float32)
        out[tuple(slice(0, n) for n in a.shape)] = a
        return out

    xd = put(padded(x, rows, wp), dev, activation(f32))
    ld = experts + 5
    ld_logits = put(padded(logits, rows, ld), dev)
    wd = [put(padded(a, experts, *s), dev, torch.bfloat16) for a, s in ((gate, (fp, wp)), (up, (fp, wp)), (down, (wp, fp)))]
    want = np.zeros((rows, width))
    score = plain.sigmoid(logits.astype(np.float64))
    for t in range(rows):
        for e in np.argsort(-logits[t], kind="stable")[:top]:
            want[t] += score[t, e] * plain.gated_mlp(x[t:t + 1].astype(np.float64), *(w[e].astype(np.float64) for w in (gate, up, down)))[0]
    for options in (0, decoder.EXPERTS_ROWS):
        nbytes = decoder.lib().qm_expert_scratch_bytes(rows, experts, top, wp, fp, int(f32))
        scratch = torch.full((nbytes // 4,), float("nan"), device=dev)
        out = torch.full((rows, wp), 7.0, device=dev)
        op = decoder.Experts(x=xd.data_ptr(), logits=ld_logits.data_ptr(), gate=wd[0].data_ptr(), up=wd[1].data_ptr(), down=wd[2].data_ptr(),
                             out32=out.data_ptr(), scratch=scratch.data_ptr(), ld_logits=ld, scratch_bytes=nbytes, rows=rows, experts=experts, top=top,
                             width_p=wp, ff_p=fp, options=options)
        assert decoder.lib().qm_expert_rows(C.byref(op), int(f32), torch.cuda.current_stream().cuda_stream) == 0
        got = get(out)
        close(got[:, :width], want, f32, tol32=5e-6, tol16=2e-2)
        assert np.all(got[:, width:] == 0)


@pytest.mark.parametrize("rows", [287, 288, 464, 465])
def test_experts_whose_rows_are_two_row_tiles(decoder, dev, rows):
    """24 experts of four column tiles with 72 to 116 rows each take one tall row tile, those outside two or three low ones; one expert is crowded."""
    test_experts(decoder, dev, False, rows, 24, 6, 128, 512)
