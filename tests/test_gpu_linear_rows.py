"""GPU parity: linears over token rows (the prompt pass) through the C ABI, against the oracle, which evaluates every
(row, column) as the M = 1 linear does.  Two kernels serve the entry points (QM_OPT_LINEAR_ROWS_KERNEL): the exact chain
(1; also what fewer than 16 rows or shapes off the matrix tiles always run) must be bit-exact; the matrix cores (0,
default) form the same fp32 sum of the same bf16 products in another order, so an output may land on the neighbouring
bf16 value: at most one ulp, and rarely."""
import numpy as np
import pytest

from qm_testlib import to_dev, to_u16, ulp_distance

pytestmark = pytest.mark.gpu

EXACT, MATRIX = 1, 0


@pytest.fixture(autouse=True, params=[EXACT, MATRIX], ids=["exact_chain", "matrix_cores"])
def rows_kernel(request, qm):
    qm.set_option(qm.OPT_LINEAR_ROWS_KERNEL, request.param)
    yield request.param
    qm.set_option(qm.OPT_LINEAR_ROWS_KERNEL, 0)


def _on_matrix_cores(kernel, rows, cols, red):
    return kernel == MATRIX and rows >= 16 and cols % 128 == 0 and red % 128 == 0


def _check(oracle, got, want, matrix, residual=None):
    if not matrix:
        assert np.array_equal(got, want)
        return
    # one bf16 spacing of the sum (which a residual of the opposite sign can leave standing alone in a small result)
    # and, with a residual, the rounding of the second addition on top: two spacings at the larger magnitude
    g, w = oracle.bf16_to_f32(got).astype(np.float64), oracle.bf16_to_f32(want).astype(np.float64)
    scale = np.abs(w) if residual is None else np.maximum(np.abs(w), np.abs(oracle.bf16_to_f32(residual).astype(np.float64)) + np.abs(w))
    bound = np.maximum(1e-2, scale * 2.0 ** (-7 if residual is None else -6))
    assert np.all(np.abs(g - w) <= bound), float(np.max(np.abs(g - w) / bound))
    assert np.count_nonzero(got != want) <= max(2, got.size // 200), (np.count_nonzero(got != want), got.size)


@pytest.mark.parametrize("rows,cols,red,bias,residual", [
    (1, 8, 8, False, False), (7, 20, 40, True, True), (8, 9, 264, True, False), (9, 33, 1000, False, True),
    (100, 2048, 2048, True, True),      # o_proj of a 100-token prompt + residual
    (37, 2048, 6144, False, True),      # down_proj + residual: four columns per block
    (300, 1024, 2048, True, False),     # k_proj
    (16, 128, 128, True, True), (129, 256, 384, False, False), (255, 384, 1024, True, True), (40, 128, 192, True, False),   # edges of the matrix tiles
    (1024, 2048, 2048, True, True),     # o_proj of a 1024-token prompt + residual
])
def test_linear_rows_against_the_oracle(oracle, qm, dev, rows, cols, red, bias, residual, rows_kernel):
    import torch
    seed = 4000 + rows + cols + red
    x = oracle.normal_bf16((rows, red), seed)
    w = oracle.normal_bf16((cols, red), seed + 1, std=0.02)
    b = oracle.normal_bf16((cols,), seed + 2, std=0.1) if bias else None
    r = oracle.normal_bf16((rows, cols), seed + 3) if residual else None
    want = np.zeros((rows, cols), dtype=np.uint16)
    assert oracle.linear_rows(x, w, b, r, want, rows, cols, red, 16) == 0
    out = torch.full((rows, cols), 0x7fc0, dtype=torch.int16, device=dev)
    qm.linear_rows(to_dev(x, dev), to_dev(w, dev), None if b is None else to_dev(b, dev),
                   None if r is None else to_dev(r, dev), out, rows, cols, red)
    torch.cuda.synchronize()
    _check(oracle, to_u16(out), want, _on_matrix_cores(rows_kernel, rows, cols, red), r)


# (a tile of each width and height the rules choose, its last row tile of one row, of all but one and whole)
@pytest.mark.parametrize("rows,cols,red", [(17, 128, 256), (63, 384, 256), (700, 1024, 256), (777, 2048, 128), (1025, 3328, 128), (2048, 2048, 128), (100, 4096, 4096)])
@pytest.mark.parametrize("rows_kernel", [MATRIX], indirect=True)
def test_outputs_and_residuals_that_begin_at_eight_bytes(oracle, qm, dev, rows, cols, red, rows_kernel):
    """Output, residual and bias at eight bytes of a line, the residual added in place, nothing written around the output."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(rows + cols)
    x = torch.randn((rows, red), generator=gen, device=dev).to(torch.bfloat16)
    w = (torch.randn((cols, red), generator=gen, device=dev) * red ** -0.5).to(torch.bfloat16)
    memory = torch.randn(rows * cols + 12 + cols, generator=gen, device=dev).to(torch.bfloat16)
    out, bias, before = memory[4:4 + rows * cols].view(rows, cols), memory[8 + rows * cols:8 + rows * cols + cols], memory.clone()
    v = (x.float() @ w.float().t() + bias.float()).to(torch.bfloat16)
    qm.linear_rows(x, w, bias, out, out, rows, cols, red)
    torch.cuda.synchronize()
    residual = before[4:4 + rows * cols].view(rows, cols)
    want = (residual.float() + v.float()).to(torch.bfloat16)
    _check(oracle, to_u16(out.contiguous().view(torch.int16)), to_u16(want.view(torch.int16)), True, to_u16(residual.contiguous().view(torch.int16)))
    assert torch.equal(memory[:4], before[:4]) and torch.equal(memory[4 + rows * cols:], before[4 + rows * cols:])


def test_a_prompt_row_equals_the_decode_linear_of_that_row(oracle, qm, dev, rows_kernel):
    """(the exact chain; with 64 rows and 128 columns the default kernel is the matrix cores, the other is asked for)"""
    import torch
    rows, cols, red = (12, 96, 2048) if rows_kernel == MATRIX else (64, 128, 2048)
    x = oracle.normal_bf16((rows, red), 1)
    w = oracle.normal_bf16((cols, red), 2, std=0.02)
    b = oracle.normal_bf16((cols,), 3, std=0.1)
    xd, wd, bd = to_dev(x, dev), to_dev(w, dev), to_dev(b, dev)
    out = torch.zeros((rows, cols), dtype=torch.int16, device=dev)
    qm.linear_rows(xd, wd, bd, None, out, rows, cols, red)
    one = torch.zeros(cols, dtype=torch.int16, device=dev)
    for r in (0, 5, rows - 1):
        qm.linear_m1(xd[r], wd, bd, None, one, cols, red)
        torch.cuda.synchronize()
        assert torch.equal(one, out[r])


# (the last three: grids between one and two blocks per CU of 128-column tiles, which take the 192-column tile if the reduction is a
# multiple of 128; 600 rows leave the last row tile ragged)
@pytest.mark.parametrize("rows,hidden,inter", [(1, 8, 1), (9, 200, 33), (64, 2048, 6144), (5, 2048, 512), (200, 1024, 3072),
                                               (640, 256, 6912), (600, 320, 6912), (600, 384, 6912)])
def test_gate_up_swiglu_rows(oracle, qm, dev, rows, hidden, inter, rows_kernel):
    import torch
    seed = 5000 + rows + hidden
    x = oracle.normal_bf16((rows, hidden), seed)
    gw = oracle.normal_bf16((inter, hidden), seed + 1, std=0.03)
    uw = oracle.normal_bf16((inter, hidden), seed + 2, std=0.03)
    want = np.zeros((rows, inter), dtype=np.uint16)
    assert oracle.gate_up_swiglu_rows(x, gw, uw, want, rows, hidden, inter, 16) == 0
    out = torch.full((rows, inter), 0x7fc0, dtype=torch.int16, device=dev)
    qm.gate_up_swiglu_rows(to_dev(x, dev), to_dev(gw, dev), to_dev(uw, dev), out, rows, hidden, inter)
    torch.cuda.synchronize()
    d = ulp_distance(to_u16(out), want)                 # (the device's expf: at most one bf16 ulp, rarely)
    if _on_matrix_cores(rows_kernel, rows, inter, hidden):
        # a gate or up value on the neighbouring bf16 value moves the product by up to two of its spacings; a gate sum
        # that nearly cancels differs by more of ITS spacings, all of them tiny: the bound is absolute + relative
        g, w = oracle.bf16_to_f32(to_u16(out)).astype(np.float64), oracle.bf16_to_f32(want).astype(np.float64)
        assert np.all(np.abs(g - w) <= 1e-3 + np.abs(w) * 2.0 ** -6), float(np.max(np.abs(g - w)))
        assert np.count_nonzero(d) <= rows * inter // 100, np.count_nonzero(d)
    else:
        assert d.max() <= 1 and np.count_nonzero(d) <= max(1, rows * inter // 1000)


def test_linear_rows_argument_errors(qm, dev):
    import torch
    x = torch.zeros((4, 72), dtype=torch.int16, device=dev)
    w = torch.zeros((8, 72), dtype=torch.int16, device=dev)
    o = torch.zeros((4, 8), dtype=torch.int16, device=dev)
    L = qm.lib()
    assert L.qm_linear_rows(None, w.data_ptr(), None, None, o.data_ptr(), 4, 8, 72, None) == -1
    assert L.qm_linear_rows(x.data_ptr(), w.data_ptr(), None, None, o.data_ptr(), 4, 8, 70, None) == -2
    assert L.qm_linear_rows(x.data_ptr(), w.data_ptr(), None, None, o.data_ptr(), -1, 8, 72, None) == -5
    assert L.qm_linear_rows(x.data_ptr() + 2, w.data_ptr(), None, None, o.data_ptr(), 1, 8, 64, None) == -2
    assert L.qm_linear_rows(x.data_ptr(), w.data_ptr(), None, None, o.data_ptr(), 0, 8, 72, None) == 0
    assert L.qm_gate_up_swiglu_rows(x.data_ptr(), w.data_ptr(), None, o.data_ptr(), 4, 72, 8, None) == -1


@pytest.mark.parametrize("rows,cols,red,bias,residual", [
    (128, 2048, 4096, True, True),      # 32 blocks, 64 steps: eight pieces
    (100, 1024, 4096, False, False),    # 16 blocks
    (37, 2048, 6144, False, True),      # down_proj + residual of a short prompt: 96 steps
    (64, 4096, 4096, True, False),      # 32 blocks: eight pieces
    (200, 1024, 4096, False, True),     # 32 blocks: eight pieces
])
def test_linear_rows_with_the_reduction_shared_between_blocks(oracle, qm, dev, rows, cols, red, bias, residual, rows_kernel):
    """qm_linear_rows_split: few token rows leave most CUs without a block; with a workspace the reduction is cut into pieces
    whose fp32 sums a second launch adds in order.  Held to the bounds of the uncut matrix-core call; the same bits on every
    call; on the exact chain the workspace is not used and the result stays bit-exact."""
    import torch
    seed = 4500 + rows + cols + red
    x = oracle.normal_bf16((rows, red), seed)
    w = oracle.normal_bf16((cols, red), seed + 1, std=0.02)
    b = oracle.normal_bf16((cols,), seed + 2, std=0.1) if bias else None
    r = oracle.normal_bf16((rows, cols), seed + 3) if residual else None
    want = np.zeros((rows, cols), dtype=np.uint16)
    assert oracle.linear_rows(x, w, b, r, want, rows, cols, red, 16) == 0
    nbytes = qm.linear_rows_split_workspace_bytes(rows, cols, red)
    assert nbytes > 0
    ws = torch.full((nbytes // 4,), float("nan"), dtype=torch.float32, device=dev)
    xd, wd = to_dev(x, dev), to_dev(w, dev)
    bd, rd = None if b is None else to_dev(b, dev), None if r is None else to_dev(r, dev)
    outs = []
    for _ in range(2):
        out = torch.full((rows, cols), 0x7fc0, dtype=torch.int16, device=dev)
        qm.linear_rows_split(xd, wd, bd, rd, out, rows, cols, red, ws, nbytes)
        torch.cuda.synchronize()
        outs.append(to_u16(out))
    assert np.array_equal(outs[0], outs[1])
    _check(oracle, outs[0], want, rows_kernel == MATRIX, r)
    if rows_kernel == MATRIX:
        assert qm.lib().qm_linear_rows_split(xd.data_ptr(), wd.data_ptr(), None, None, out.data_ptr(), rows, cols, red, ws.data_ptr(),
                                             nbytes - 4, None) == -4
    assert qm.linear_rows_split_workspace_bytes(1024, 2048, 6144) == 0      # enough blocks already
    assert qm.linear_rows_split_workspace_bytes(128, 2048, 2048) == 0       # a reduction of 2048 stays whole


@pytest.mark.parametrize("rows,hidden,inter", [(128, 4096, 3072), (48, 4096, 1536)])
def test_gate_up_swiglu_rows_with_the_reduction_shared_between_blocks(oracle, qm, dev, rows, hidden, inter, rows_kernel):
    import torch
    seed = 5500 + rows + hidden
    x = oracle.normal_bf16((rows, hidden), seed)
    gw = oracle.normal_bf16((inter, hidden), seed + 1, std=0.03)
    uw = oracle.normal_bf16((inter, hidden), seed + 2, std=0.03)
    want = np.zeros((rows, inter), dtype=np.uint16)
    assert oracle.gate_up_swiglu_rows(x, gw, uw, want, rows, hidden, inter, 16) == 0
    nbytes = qm.linear_rows_split_workspace_bytes(rows, inter, hidden, True)
    assert nbytes > 0
    ws = torch.full((nbytes // 4,), float("nan"), dtype=torch.float32, device=dev)
    outs = []
    for _ in range(2):
        out = torch.full((rows, inter), 0x7fc0, dtype=torch.int16, device=dev)
        qm.gate_up_swiglu_rows_split(to_dev(x, dev), to_dev(gw, dev), to_dev(uw, dev), out, rows, hidden, inter, ws, nbytes)
        torch.cuda.synchronize()
        outs.append(to_u16(out))
    assert np.array_equal(outs[0], outs[1])
    d = ulp_distance(outs[0], want)
    if rows_kernel == MATRIX:
        g, w = oracle.bf16_to_f32(outs[0]).astype(np.float64), oracle.bf16_to_f32(want).astype(np.float64)
        assert np.all(np.abs(g - w) <= 1e-3 + np.abs(w) * 2.0 ** -6), float(np.max(np.abs(g - w)))
        assert np.count_nonzero(d) <= rows * inter // 100, np.count_nonzero(d)
    else:
        assert d.max() <= 1 and np.count_nonzero(d) <= max(1, rows * inter // 1000)


@pytest.mark.parametrize("rows,q_cols,kv_cols,red", [(1024, 2048, 1024, 2048), (300, 512, 256, 384), (128, 2048, 1024, 2048), (7, 256, 128, 256)])
def test_qkv_rows_is_three_linear_rows(qm, dev, oracle, rows, q_cols, kv_cols, red):
    """qm_qkv_rows: bit for bit what three qm_linear_rows calls give (one grid on the matrix cores where the shapes are
    served; three calls below sixteen rows)."""
    import torch
    x = to_dev(oracle.normal_bf16((rows, red), 77), dev)
    ws = [to_dev(oracle.normal_bf16((c, red), 78 + i, std=0.03), dev) for i, c in enumerate((q_cols, kv_cols, kv_cols))]
    bs = [to_dev(oracle.normal_bf16((c,), 88 + i, std=0.1), dev) for i, c in enumerate((q_cols, kv_cols, kv_cols))]
    for biases in (bs, [bs[0], None, bs[2]]):
        want = [torch.full((rows, c), 0x7fc0, dtype=torch.int16, device=dev) for c in (q_cols, kv_cols, kv_cols)]
        got = [torch.full((rows, c), 0x7fc0, dtype=torch.int16, device=dev) for c in (q_cols, kv_cols, kv_cols)]
        for w, b, o, c in zip(ws, biases, want, (q_cols, kv_cols, kv_cols)):
            qm.linear_rows(x, w, b, None, o, rows, c, red)
        qm.qkv_rows(x, ws, biases, got, rows, q_cols, kv_cols, red)
        torch.cuda.synchronize()
        for g, w in zip(got, want):
            assert torch.equal(g, w)
    # with a workspace (of whatever size: the one grid never cuts a reduction) the same bits
    wsp = torch.empty(1 << 20, dtype=torch.float32, device=dev)
    got = [torch.full((rows, c), 0x7fc0, dtype=torch.int16, device=dev) for c in (q_cols, kv_cols, kv_cols)]
    qm.qkv_rows(x, ws, bs, got, rows, q_cols, kv_cols, red, wsp, 4 << 20)
    torch.cuda.synchronize()
    for g, w, b, c in zip(got, ws, bs, (q_cols, kv_cols, kv_cols)):
        want = torch.full((rows, c), 0x7fc0, dtype=torch.int16, device=dev)
        qm.linear_rows(x, w, b, None, want, rows, c, red)
        torch.cuda.synchronize()
        assert torch.equal(g, want)


def test_qkv_rows_argument_errors(qm, dev):
    import torch
    x = torch.zeros((16, 128), dtype=torch.int16, device=dev)
    w = torch.zeros((128, 128), dtype=torch.int16, device=dev)
    o = torch.zeros((16, 128), dtype=torch.int16, device=dev)
    f = qm.lib().qm_qkv_rows
    assert f(None, w.data_ptr(), w.data_ptr(), w.data_ptr(), None, None, None, o.data_ptr(), o.data_ptr(), o.data_ptr(), 16, 128, 128, 128, None) == -1
    assert f(x.data_ptr(), w.data_ptr(), w.data_ptr(), w.data_ptr(), None, None, None, o.data_ptr(), o.data_ptr(), None, 16, 128, 128, 128, None) == -1
    assert f(x.data_ptr(), w.data_ptr(), w.data_ptr(), w.data_ptr(), None, None, None, o.data_ptr(), o.data_ptr(), o.data_ptr(), 16, 128, 128, 124, None) == -2
    assert f(x.data_ptr(), w.data_ptr(), w.data_ptr(), w.data_ptr(), None, None, None, o.data_ptr(), o.data_ptr(), o.data_ptr(), -1, 128, 128, 128, None) == -5


def test_qkv_rows_with_an_empty_member(qm, dev, oracle):
    """A linear of no columns among the three leaves the other two as they are alone (the shapes that would share one
    grid: 64 rows, widths in 128s)."""
    import torch
    rows, red = 64, 256
    x = to_dev(oracle.normal_bf16((rows, red), 5), dev)
    for q_cols, kv_cols in ((0, 128), (256, 0)):
        widths = (q_cols, kv_cols, kv_cols)
        ws = [to_dev(oracle.normal_bf16((max(c, 1), red), 6 + i, std=0.03), dev) for i, c in enumerate(widths)]
        got = [torch.full((rows, max(c, 1)), 0x7fc0, dtype=torch.int16, device=dev) for c in widths]
        want = [torch.full((rows, max(c, 1)), 0x7fc0, dtype=torch.int16, device=dev) for c in widths]
        for w, o, c in zip(ws, want, widths):
            qm.linear_rows(x, w, None, None, o, rows, c, red)
        qm.qkv_rows(x, ws, [None, None, None], got, rows, q_cols, kv_cols, red)
        torch.cuda.synchronize()
        for g, w in zip(got, want):
            assert torch.equal(g, w)



@pytest.mark.parametrize("rows,cols,red", [
    # each tile of the matrix-core kernel at a remainder of rows: 64 x 64 (one step, fewer steps than its stages, many), 64 x 128,
    # 64 x 128 with 128 k a step, 128 x 128 with one and several rounds, a pair's 128 x 192 with fewer and with many more steps than its
    # weight lines are asked for ahead
    (17, 128, 128), (65, 256, 256), (190, 2048, 3072), (300, 4096, 256), (129, 16640, 384), (65, 16640, 4096), (1000, 4096, 256), (1030, 8192, 128),
    (600, 6912, 384), (1000, 6144, 2048)])
@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("rows_kernel", [MATRIX], indirect=True)       # (the exact chain is compared bit for bit above)
def test_matrix_core_tiles_against_64_bits(qm, dev, rows, cols, red, pair, rows_kernel):
    """Every output is the rounding of a sum that is within red * 2^-24 * sum |x w| of the exact one; a pair's roundings of gate, SiLU,
    up and product follow, half a spacing (2^-8 at most) of the value each, the gate's through a slope of at most 1.1."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(rows + red)
    x = torch.randn(rows, red, device=dev, generator=gen).bfloat16()
    w, up = ((torch.randn(cols, red, device=dev, generator=gen) * red ** -0.5).bfloat16() for _ in range(2))
    out = torch.full((rows + 1, cols), 7.0, device=dev, dtype=torch.bfloat16)
    if pair:
        qm.gate_up_swiglu_rows(x, w, up, out, rows, red, cols)
    else:
        qm.linear_rows(x, w, None, None, out, rows, cols, red)
    torch.cuda.synchronize()
    assert bool((out[rows:] == 7).all())
    got, unit, half = out[:rows].double(), red * 2.0 ** -24, 2.0 ** -8
    s, most = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    want, bound = s, unit * most + half * s.abs()
    if pair:
        u, u_most = x.double() @ up.double().t(), x.double().abs() @ up.double().abs().t()
        act = torch.nn.functional.silu(s)
        act_bound = 1.1 * bound + half * act.abs()
        u_bound = unit * u_most + half * u.abs()
        want = act * u
        bound = act_bound * u.abs() + u_bound * act.abs() + act_bound * u_bound + half * want.abs()
    assert bool(((got - want).abs() <= bound + 1e-30).all()), float(((got - want).abs() / (bound + 1e-30)).max())


@pytest.mark.parametrize("rows,cols,red", [(600, 3072, 256), (640, 3072, 256), (641, 3072, 256), (1024, 2048, 256), (1025, 2048, 256), (833, 2560, 256), (385, 4992, 256),
                                           (897, 2304, 384), (65, 16384, 4096), (130, 10880, 4096), (130, 11008, 4096)])
@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("rows_kernel", [MATRIX], indirect=True)
def test_grids_of_low_tiles_of_one_round_and_of_more(qm, dev, rows, cols, red, pair, rows_kernel):
    """Tiles of 64 rows come to 240 to 288 blocks: up to 256 they are taken, above tiles of 128 rows are; tolerance as above."""
    test_matrix_core_tiles_against_64_bits(qm, dev, rows, cols, red, pair, rows_kernel)


@pytest.mark.parametrize("rows,cols,red", [(129, 5248, 128), (65, 5376, 256), (300, 5248, 128), (1024, 5888, 128)])
@pytest.mark.parametrize("rows_kernel", [MATRIX], indirect=True)
def test_more_than_forty_column_tiles_that_eight_does_not_divide(qm, dev, rows, cols, red, rows_kernel):
    """The grid's width is rounded up and the blocks beyond the last tile end: every output is written, and nothing behind them."""
    import torch
    gen = torch.Generator(device=dev).manual_seed(rows + cols)
    x = torch.randn(rows, red, device=dev, generator=gen).bfloat16()
    w = torch.randn(cols, red, device=dev, generator=gen).bfloat16()
    out = torch.full((rows + 1, cols), float("nan"), dtype=torch.bfloat16, device=dev)
    qm.linear_rows(x, w, None, None, out, rows, cols, red)
    want = x.double() @ w.double().t()
    # half a bf16 spacing of the sum, and the fp32 sum's own error: red * 2^-24 of the sum of magnitudes
    bound = want.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().t()) * red * 2.0 ** -24
    assert bool(((out[:rows].double() - want).abs() <= bound).all())
    assert bool(out[rows].isnan().all())


@pytest.mark.parametrize("rows_kernel", [MATRIX], indirect=True)
def test_swiglu_of_every_bf16_gate(qm, dev, rows_kernel):
    """Each finite gate value once, through an identity on the matrix cores: the bits of the exact chain's expf and division."""
    import torch
    x = torch.eye(128, device=dev).bfloat16()
    up = torch.ones(128, 128, device=dev).bfloat16()
    for part in range(4):
        bits = (torch.arange(16384, dtype=torch.int32, device=dev) + 16384 * part).to(torch.int16).view(128, 128)
        gate = bits.view(torch.bfloat16)
        gate = torch.where(gate.float().isfinite(), gate, torch.zeros_like(gate)).contiguous()    # (0 times infinity is no gate)
        got = []
        for kernel in (MATRIX, EXACT):
            qm.set_option(qm.OPT_LINEAR_ROWS_KERNEL, kernel)
            out = torch.zeros(128, 128, dtype=torch.int16, device=dev)
            qm.gate_up_swiglu_rows(x, gate, up, out, 128, 128, 128)
            got.append(out)
        torch.cuda.synchronize()
        assert bool((got[0] == got[1]).all()), part


@pytest.mark.parametrize("rows_kernel", [MATRIX], indirect=True)
def test_swiglu_of_gates_that_are_no_numbers(qm, dev, rows_kernel):
    """Through the same identity, a column of infinite and undefined gate weights: the first token's gates are those, every other's 0 times them.  What the
    exact chain makes of them, a NaN being a NaN."""
    import torch
    x, up = torch.eye(128, device=dev).bfloat16(), torch.ones(128, 128, device=dev).bfloat16()
    gate = torch.full((128, 128), 0.5, device=dev).bfloat16()
    gate[0, 0], gate[1, 0], gate[2, 0] = float("inf"), float("-inf"), float("nan")
    got = []
    for kernel in (MATRIX, EXACT):
        qm.set_option(qm.OPT_LINEAR_ROWS_KERNEL, kernel)
        out = torch.zeros(128, 128, dtype=torch.bfloat16, device=dev)
        qm.gate_up_swiglu_rows(x, gate, up, out, 128, 128, 128)
        got.append(out.float())
    torch.cuda.synchronize()
    assert got[1][0, 0] == float("inf") and bool(got[1][0, 1:3].isnan().all()) and bool(got[1][1:, :3].isnan().all())
    assert torch.equal(got[0].isnan(), got[1].isnan())
    assert torch.equal(got[0].nan_to_num(7.0, float("inf"), float("-inf")), got[1].nan_to_num(7.0, float("inf"), float("-inf")))


# rows, columns, reduction: pieces of the reduction with a norm behind (0: whole)
NORM_PIECES = {(16, 2048, 6144): 8, (100, 1024, 4096): 8, (785, 2048, 6144): 2, (1000, 2048, 6144): 2, (1024, 2048, 4224): 0, (1601, 1024, 4096): 0,
               (2048, 1024, 6144): 2, (1025, 2048, 6144): 0, (300, 1536, 4096): 4, (900, 2048, 2048): 0}


@pytest.mark.parametrize("rows,cols,red", list(NORM_PIECES))
@pytest.mark.parametrize("rows_kernel", [MATRIX, EXACT], indirect=True)
@pytest.mark.parametrize("bias", [False, True])
def test_linear_and_norm_of_its_rows(qm, dev, rows, cols, red, rows_kernel, bias):
    """Cut in 128-row tiles, cut in smaller ones, not cut, on the exact chain: the sum with its residual against 64 bits, the norm the bits that
    qm_rmsnorm_rows gives for the output."""
    import torch
    if rows_kernel == EXACT and rows > 100:
        rows = 17
    gen = torch.Generator(device=dev).manual_seed(rows + cols + red)
    x, w, res, gamma = (torch.randn(*shape, device=dev, generator=gen).bfloat16() for shape in ((rows, red), (cols, red), (rows, cols), (cols,)))
    b = torch.randn(cols, device=dev, generator=gen).bfloat16() if bias else None
    need = qm.lib().qm_linear_rows_norm_workspace_bytes(rows, cols, red)
    if rows_kernel == MATRIX:
        assert need == NORM_PIECES[rows, cols, red] * rows * cols * 4
    ws = torch.empty(max(need, 256), dtype=torch.uint8, device=dev)
    out, normed = (torch.full((rows + 1, cols), float("nan"), dtype=torch.bfloat16, device=dev) for _ in range(2))
    call = lambda bytes_: qm.lib().qm_linear_rows_norm(x.data_ptr(), w.data_ptr(), b.data_ptr() if bias else None, res.data_ptr(), out.data_ptr(),
                                                       gamma.data_ptr(), normed.data_ptr(), rows, cols, red, 1e-6, ws.data_ptr(), bytes_, None)
    if need > 0 and rows_kernel == MATRIX:
        assert call(need - 256) < 0
    assert call(need) == 0
    again = torch.empty(rows, cols, dtype=torch.bfloat16, device=dev)
    qm.rmsnorm_rows(out, gamma, again, rows, cols, 1e-6)
    torch.cuda.synchronize()
    assert bool((normed[:rows].view(torch.int16) == again.view(torch.int16)).all())
    assert bool(out[rows].isnan().all() and normed[rows].isnan().all())
    sums = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    want = sums + res.double()
    # two roundings, each half a bf16 spacing at most, and the fp32 sum's own error: red * 2^-24 of the sum of magnitudes
    bound = (sums.abs() + want.abs()) * 2.0 ** -8 + (x.double().abs() @ w.double().abs().t()) * red * 2.0 ** -24
    assert bool(((out[:rows].double() - want).abs() <= bound).all())
