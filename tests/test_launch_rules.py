"""CPU-only checks of rules that choose a launch's shape: small programs over the kernels' own headers, linked with the built library where the rule
lives in it."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "qingming-qwen3-tts_amd", "csrc")
LIB = os.path.join(ROOT, "qingming-qwen3-tts_amd", "lib")


def run(tmp_path, source, *libraries):
    """The output lines of a program of one `main`, which sees no GPU."""
    path = tmp_path / "rule.cpp"
    path.write_text(source)
    link = ["-L" + LIB, "-L/opt/rocm/lib", *("-l" + name for name in libraries), "-Wl,-rpath," + LIB + ":/opt/rocm/lib"] if libraries else []
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, "-I" + os.path.join(ROOT, "include"), "-o",
                    str(tmp_path / "rule"), str(path), *link], check=True)
    hidden = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1")
    return subprocess.run([str(tmp_path / "rule")], check=True, capture_output=True, text=True, env=hidden).stdout.splitlines()


def test_a_rounded_grid_keeps_no_die_much_longer_than_an_even_deal(tmp_path):
    """Row linears: blocks go to the eight dies of 32 CUs in turn, one to a CU.  Where a grid's width is rounded up, no die walks more rounds of blocks than
    all of them do when the tiles are dealt out one by one, or a third more at most (three rounds become four)."""
    lines = run(tmp_path, """
#include <cstdio>
#include "qm_linear_rows_params.h"
int main() {
    for (int columns = 1; columns <= 400; ++columns)
        for (int rows = 1; rows <= 64; ++rows)
            for (int pieces = 1; pieces <= 8; pieces *= 2) std::printf("%d %d %d %d\\n", columns, rows, pieces, qm::rows_grid_columns(columns, rows, pieces));
}""")
    assert len(lines) == 400 * 64 * 4
    rounded = 0
    for line in lines:
        columns, rows, pieces, width = map(int, line.split())
        assert width in (columns, (columns + 7) // 8 * 8)
        tiles = columns * rows * pieces
        if width % 8 == 0:                                   # column c's tiles are all on die c % 8
            busiest = -(-columns // 8) * rows * pieces
        else:                                                # the grid has a tile for every block: dealt out one by one
            assert width == columns
            busiest = -(-tiles // 8)
        if width != columns:
            rounds, even = -(-busiest // 32), -(-(-(-tiles // 8)) // 32)
            assert rounds == even or (even >= 3 and 3 * rounds <= 4 * even), line
            rounded += 1
    assert rounded > 5000
    assert "81 8 1 88" in lines and "81 9 1 88" in lines and "42 6 1 42" in lines and "42 3 2 42" in lines and "42 12 1 42" in lines


ROWS_OF = """
#include <cstdio>
#include <vector>
#include "qm_attn.h"
#include "qm_linear_rows_params.h"
static float planes[1];
static uint16_t weight[1];
static qm::LinearRowsParams of(int rows, std::vector<std::pair<int, int>> linears, int parts = 1, bool norm = false) {
    qm::LinearRowsParams p = {};
    p.rows = rows;
    p.groups = static_cast<int>(linears.size());
    p.reduction_parts = parts;
    if (parts > 1) p.partials = planes;
    if (norm) p.norm_weight = weight;
    p.columns = linears[0].first;
    p.reduction = linears[0].second;
    int columns = p.columns;
    for (int g = 1; g < p.groups; ++g) {
        p.group_first_tile[g - 1] = columns / 128;
        p.group_columns[g - 1] = linears[g].first;
        p.group_reduction[g - 1] = linears[g].second;
        columns += linears[g].first;
    }
    return p;
}
int main() {
"""


# rows; (columns, reduction) each; whether a gate/up pair; pieces; whether a norm adds them
HANGING = [(1024, [(10176, 2048)], 0, 1, 0), (1024, [(10176, 2048)], 1, 1, 0), (16, [(64, 128)], 0, 1, 0), (777, [(2048, 1088)], 0, 1, 0),
           (1024, [(6144, 2080)], 1, 1, 0), (1000, [(2048, 2048), (1088, 2048)], 0, 1, 0), (1000, [(2048, 2048), (1024, 2048), (1024, 2112)], 0, 1, 0),
           (300, [(2048, 4160)], 0, 1, 0), (64, [(2048, 6144)], 0, 5, 0), (64, [(2048, 4224)], 0, 4, 0), (64, [(2048, 6144)], 1, 7, 0),
           (64, [(2048, 6144), (2048, 6144)], 0, 4, 0), (64, [(2048, 6144)], 0, 3, 1), (64, [(4096, 6144)], 0, 2, 1)]


@pytest.mark.parametrize("library", ["qm_attn", "qm_decoder"])
def test_no_tile_of_the_row_linears_hangs_over_a_matrix(tmp_path, library):
    """The launch itself refuses what its tiles and steps do not cover exactly, whoever calls it."""
    calls = "".join("""
    std::printf("%%d\\n", qm::launch_rows_mfma(of(%d, {%s}, %d, %d), %d, nullptr));""" % (rows, ", ".join("{%d, %d}" % l for l in linears), parts, norm, dual)
                    for rows, linears, dual, parts, norm in HANGING)
    calls += """
    qm::LinearRowsParams shifted = of(1024, {{2048, 2048}, {2048, 2048}});
    shifted.group_first_tile[0] = 15;                        // a linear's tiles begin inside the one before
    std::printf("%d\\n", qm::launch_rows_mfma(shifted, false, nullptr));
    qm::LinearRowsParams nowhere = of(64, {{2048, 6144}}, 4);
    nowhere.partials = nullptr;
    std::printf("%d\\n", qm::launch_rows_mfma(nowhere, false, nullptr));
    std::printf("%d\\n", QM_ERR_GEOMETRY);
}"""
    *got, geometry = map(int, run(tmp_path, ROWS_OF + calls, library))
    assert got == [geometry] * (len(HANGING) + 2)


def test_the_row_linears_take_what_their_entry_points_let_through(tmp_path):
    """Whole tiles and steps, for every choice of tile and for the pieces that are chosen."""
    lines = run(tmp_path, ROWS_OF + """
    for (int rows : {16, 100, 520, 777, 1024, 4096})
        for (int columns = 128; columns <= 12288; columns += columns < 2048 ? 128 : 896)
            for (int reduction = 128; reduction <= 16384; reduction += reduction < 1024 ? 128 : 896) {
                bool wide = false;
                const int parts = qm::rows_mfma_reduction_parts(rows, columns, reduction, false), behind = qm::rows_mfma_norm_parts(rows, columns, reduction, &wide);
                bool fits = true;
                for (int tile : {64, 128})
                    fits = fits && qm::rows_are_whole_tiles(of(rows, {{columns, reduction}, {columns, 128}, {128, reduction}}), tile, 128) &&
                           qm::rows_are_whole_tiles(of(rows, {{columns, reduction}}, parts), tile, 64) &&
                           qm::rows_are_whole_tiles(of(rows, {{columns, reduction}}, behind, true), tile, 64);
                std::printf("%d %d %d\\n", fits && qm::rows_are_whole_tiles(of(rows, {{columns, reduction}}), 192, 64) == (columns % 192 == 0), parts, behind);
            }
}""", "qm_attn")
    got = [tuple(map(int, line.split())) for line in lines]
    assert all(fits for fits, _, _ in got) and len(got) > 3000
    assert {1, 2, 4, 8} <= {parts for _, parts, _ in got} and any(behind > parts for _, parts, behind in got)


def test_the_row_linears_take_a_decoders_launches(tmp_path):
    """Linears of several inputs and widths, pairs and the pieces of a reduction get as far as the device, which is not there."""
    shapes = [(list(linears), rows) for linears, rows, _ in CUTS] + [([(11264, 2048)], 1024), ([(128, 128), (3072, 640), (1024, 6144)], 16), ([(128, 128), (-384, 256)], 100)]
    source = OF_SIZES.replace("int main() {", """int main() {
    int devices = 0;
    if (hipGetDeviceCount(&devices) == hipSuccess && devices > 0) return 1;              // (nothing below may be launched: the addresses are made up)
""")
    for linears, rows in shapes:
        source += """
    {
        qm::ReductionCut cut = {reinterpret_cast<float*>(somewhere), int64_t{1} << 40, 0, 0};
        const int rc = qm::launch_decoder_linears(of(%s, %d), 0, nullptr, &cut);
        std::printf("%%d %%d\\n", rc <= QM_ERR_HIP_BASE, cut.planes + 1);
    }""" % (sizes(linears), rows)
    got = [tuple(map(int, line.split())) for line in run(tmp_path, source + "}", "qm_decoder", "amdhip64")]
    assert got[:len(CUTS)] == [(1, pieces) for _, _, pieces in CUTS] and got[len(CUTS):] == [(1, 1)] * 3


# output linears as (columns, reduction) each, the last the one that may be cut; rows; its pieces (the first four are the layers of
# test_gpu_decoder.py's test_down_projection_in_pieces, the last of its test_a_layer_without_feed_forward_is_cut_in_front_of_its_norm)
CUTS = [([(2048, 2048), (2048, 6144)], 1000, 3), ([(2048, 2048), (2048, 2048), (2048, 6144)], 900, 2), ([(1024, 1024), (1024, 3072)], 1601, 3),
        ([(1024, 1024), (1024, 384)], 1601, 1), ([(2048, 2048), (2048, 6144)], 700, 1), ([(2048, 6144)], 1024, 1),
        ([(1024, 256), (1024, 2048)], 1601, 2), ([(1024, 256), (1024, 2048)], 1536, 1)]


def test_pieces_of_a_decoders_reduction_and_their_memory(tmp_path):
    """Into how many pieces the last of several output linears is cut, and that the memory for it holds the pieces of every number of rows."""
    shapes = [linears for linears, _, _ in CUTS] + [[(3072, 3072), (3072, 9216)], [(1280, 640), (1280, 2560), (1280, 5120)]]
    source = """
#include <cstdio>
#include "decoder/qm_decoder_ops.h"
static qm::DecLinearParams of(std::initializer_list<std::pair<int, int>> linears, int rows) {
    qm::DecLinearParams p = {};
    p.rows = rows;
    for (const auto& [n, k] : linears) {
        p.group[p.groups].n = n;
        p.group[p.groups++].k = k;
    }
    return p;
}
int main() {
"""
    for linears in shapes:
        text = "{" + ", ".join("{%d, %d}" % l for l in linears) + "}"
        source += f"""
    for (int rows = 1; rows <= 2300; ++rows)
        std::printf("%d %lld\\n", qm::reduction_pieces(of({text}, rows)), (long long)qm::reduction_cut_floats(of({text}, rows), rows));
"""
    lines = [tuple(map(int, line.split())) for line in run(tmp_path, source + "}", "qm_decoder")]
    assert len(lines) == 2300 * len(shapes)
    for i, linears in enumerate(shapes):
        of_rows = lines[2300 * i:2300 * (i + 1)]
        most = 0
        for rows, (pieces, floats) in enumerate(of_rows, 1):
            assert 1 <= pieces <= 3 and linears[-1][1] % (128 * pieces) == 0
            most = max(most, (pieces - 1) * rows * linears[-1][0])
            assert most <= floats, (linears, rows)                    # enough for as many rows and for fewer
            assert floats <= 2 * (rows + 127) * linears[-1][0] and (floats > 0) == (most > 0), (linears, rows)
    for i, (linears, rows, pieces) in enumerate(CUTS):
        assert lines[2300 * i + rows - 1][0] == pieces, (linears, rows)


# fp32 linears as (columns, reduction), negative columns a pair's channels; rows; whether their inputs are split beforehand, and the last one's pieces (the first
# three are the prompts of test_gpu_decoder.py's test_linears_of_a_long_fp32_prompt and test_norms_that_leave_their_rows_split)
PLANES = [([(1024, 1024), (1024, 3072)], 300, True, 3), ([(1024, 1024), (1024, 1024), (1024, 3072)], 400, True, 2), ([(-3072, 1152)], 200, True, 1),
          ([(-2048, 2176)], 300, True, 1), ([(5120, 1024), (-3072, 1024)], 100, True, 1), ([(4096, 4096)], 300, True, 1),
          # four groups of waves share the reductions, and the shorter ones would lose by planes; then only long ones
          ([(1024, 1024), (1024, 1024), (1024, 3072)], 160, False, 1), ([(1024, 1024), (1024, 1024), (1024, 3072)], 17, False, 1),
          ([(2048, 2048), (2048, 6144)], 100, False, 1), ([(1024, 3072), (1024, 9216)], 100, True, 3),
          # two groups: from 1024 inputs on
          ([(1024, 512), (1024, 4096)], 300, False, 1), ([(1024, 1024), (1024, 4096)], 300, True, 2), ([(-1024, 896), (4096, 896)], 200, False, 1),
          # none: from 512 on
          ([(2048, 512), (2048, 4096)], 600, True, 1), ([(2048, 384), (2048, 4096)], 600, False, 1), ([(4096, 640)], 2000, False, 1),
          # few rows; few outputs
          ([(4096, 4096)], 16, False, 1), ([(16, 1024)], 300, False, 1)]


# fp32 linears of `rows` rows, at one address where only their sizes matter
OF_SIZES = """
#include <cstdio>
#include "decoder/qm_decoder_ops.h"
alignas(16) static char somewhere[16];
static qm::DecLinearParams of(std::initializer_list<std::pair<int, int>> linears, int rows) {
    qm::DecLinearParams p = {};
    p.rows = rows;
    for (const auto& [n, k] : linears) {
        qm::DecLinearGroup& g = p.group[p.groups++];
        g.x = g.out = somewhere;
        g.out32 = reinterpret_cast<float*>(somewhere);
        g.w = reinterpret_cast<const uint16_t*>(somewhere);
        g.w_up = n < 0 ? g.w : nullptr;
        g.ldx = g.k = k;
        g.ldo = g.n = n < 0 ? -n : n;
    }
    return p;
}
static bool goes(const qm::DecLinearParams& p, int f32, int64_t elements) {
    qm::ReductionCut cut = {};
    return qm::goes_through_planes(p, f32, &cut, {reinterpret_cast<uint16_t*>(somewhere), elements});
}
int main() {
"""


def sizes(linears):
    return "{" + ", ".join("{%d, %d}" % l for l in linears) + "}"


def test_which_fp32_inputs_are_split_beforehand(tmp_path):
    source = OF_SIZES
    for linears, rows, _, _ in PLANES:
        source += """
    {
        const qm::DecLinearParams p = of(%s, %d);
        const int64_t all = qm::plane_elements(p);
        std::printf("%%d %%d %%d %%d\\n", goes(p, 1, all), qm::plane_pieces(p), goes(p, 1, all - 1), goes(p, 0, all));
    }""" % (sizes(linears), rows)
    lines = run(tmp_path, source + "}", "qm_decoder")
    assert len(lines) == len(PLANES)
    for line, (linears, rows, takes, pieces) in zip(lines, PLANES):
        got = list(map(int, line.split()))
        assert got[0] == takes and got[2:] == [0, 0], (linears, rows, got)
        assert not takes or got[1] == pieces, (linears, rows, got)


def test_memory_for_fp32_inputs_that_are_split_beforehand(tmp_path):
    """What a prompt of up to so many rows takes of it: as much as the largest that goes that way, and for pieces of a reduction at most a row tile more;
    nothing where none goes."""
    shapes = [linears for linears, _, _, _ in PLANES] + [[(128, 128), (128, 128), (128, 384)], [(2048, 640), (2048, 640), (2048, 640)]]
    most = 700
    source = OF_SIZES
    for linears in shapes:
        text = sizes(linears)
        source += f"""
    for (int rows = 1; rows <= {most}; ++rows) {{
        const qm::DecLinearParams p = of({text}, rows);
        const bool takes = goes(p, 1, int64_t{{1}} << 40);
        std::printf("%lld %lld %lld %lld\\n", takes ? (long long)qm::plane_elements(p) : 0, (long long)qm::plane_elements_up_to(p, rows, true),
                    takes ? (qm::plane_pieces(p) - 1ll) * rows * p.group[p.groups - 1].n : 0, (long long)qm::plane_cut_floats(p, rows));
    }}"""
    lines = [tuple(map(int, line.split())) for line in run(tmp_path, source + "}", "qm_decoder")]
    assert len(lines) == most * len(shapes)
    used = 0
    for i, linears in enumerate(shapes):
        elements = floats = 0
        for rows, (needs, has, cut_needs, cut_has) in enumerate(lines[most * i:most * (i + 1)], 1):
            elements, floats = max(elements, needs), max(floats, cut_needs)
            assert has == elements, (linears, rows)
            assert floats <= cut_has <= 2 * (rows + 63) * abs(linears[-1][0]), (linears, rows)
        used += elements > 0
        assert (cut_has > 0) == (floats > 0), linears
    assert 8 <= used <= len(shapes) - 4 and lines[-1] == (0, 0, 0, 0) and lines[-1 - most] == (0, 0, 0, 0)


def test_a_norm_behind_a_linear_takes_no_cut_away(qm):
    """Whatever the width, a reduction that is cut by itself is cut with the norm behind as well, and the workspace holds its pieces."""
    L, cut, more = qm.lib(), 0, 0
    for cols in (128, 512, 1024, 1536, 2048, 3072, 4096):
        for red in (128, 2048, 4096, 6144, 8192):
            for rows in (1, 15, 16, 64, 100, 200, 300, 520, 768, 769, 900, 1024, 1025, 1600, 2048):
                alone, behind = L.qm_linear_rows_split_workspace_bytes(rows, cols, red, 0), L.qm_linear_rows_norm_workspace_bytes(rows, cols, red)
                assert behind >= alone and behind % (rows * cols * 4) == 0, (rows, cols, red)
                cut += alone > 0
                more += behind > alone
    assert cut > 40 and more > 4, (cut, more)


def test_a_steps_weights_stay_in_flight(tmp_path):
    """A long row's dot products, the first weights asked for at one of several places as in a step's output launch: in the loop over the row nothing waits
    for all loads (vmcnt(0)), a piece's products leave the requests behind it under way."""
    (tmp_path / "loop.hip").write_text("""
#include "decoder/qm_decoder_device.h"
#include "decoder/qm_decoder_dot.h"
using namespace qm;
extern "C" __global__ __launch_bounds__(256) void long_row(DecLinearGroup group, const uint16_t* x, int kind) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    uint16_t* xs = reinterpret_cast<uint16_t*>(smem);
    const auto d = dot_rows<2, false>(group, static_cast<int>(blockIdx.x));
    uint4 piece[kDotAhead][2];
    if (kind == 0) {
        dot_request(d, group.k, piece);
        for (int c = threadIdx.x; c < group.k; c += 256) xs[c] = x[c];
    } else {
        const uint16_t first = x[threadIdx.x];
        dot_request(d, group.k, piece);
        for (int c = threadIdx.x; c < group.k; c += 256) xs[c] = first;
    }
    __syncthreads();
    dot_finish<uint16_t, 1>(group, d, piece, xs, 0, 1);
}
""")
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I" + CSRC, "--cuda-device-only", "-S", str(tmp_path / "loop.hip"), "-o", str(tmp_path / "loop.s")], check=True, capture_output=True)
    text = (tmp_path / "loop.s").read_text()
    body = text[text.index("\nlong_row:"):text.index(".Lfunc_end0")]
    # the loop: the shortest stretch between a label and a branch back to it with products and requests in it
    loops = []
    for m in re.finditer(r"s_cbranch_\w+ (\.LBB\d+_\d+)", body):
        start = body.find("\n" + m.group(1) + ":")
        if 0 <= start < m.start():
            loop = body[start:m.start()]
            if "v_dot2" in loop and "global_load_dwordx4" in loop:
                loops.append(loop)
    assert not re.search(r"s_waitcnt[^\n]*vmcnt\(0\)", min(loops, key=len))
