"""Which form of a kernel a launch takes, by sizes alone: the rules' headers, compiled for the host (no GPU).  For each
size the form that was measured to be the faster one, by more than the runs differ."""
import subprocess

import pytest

from dlcompiler_amd.build import CSRC_DIR

PROGRAM = """
#include <cstdio>
#include <cstring>
#include "moe_rules.h"
#include "prefill_rules.h"
using namespace dlb;
int main() {
  char what[32];
  long long a[9];
  while (scanf("%31s", what) == 1) {
    for (int i = 0; i < 9; ++i) a[i] = 0;
    int n = 0;
    while (n < 9 && scanf("%lld", &a[n]) == 1) ++n;
    if (!strcmp(what, "few")) {  // experts, local, topk, tokens, hidden, inter, cus
      const MoeLaunch up = {true, a[3] * a[2], a[3], a[2], a[0], a[1], a[5], a[4], a[6]};
      const FewRows f = fp8_few_rows(up);
      puts(f == FewRows::kInSteps ? "steps" : f == FewRows::kAhead ? "ahead" : "f32");
    }
    if (!strcmp(what, "shape")) {  // gated, experts, local, slots, columns, row bytes, cus
      const StreamShape f = stream_shape_16bit({a[0] != 0, a[3], a[3], 1, a[1], a[2], a[4], a[5], a[6]});
      printf("%d%d\\n", f.cw, f.nt);
    }
    if (!strcmp(what, "share"))  // paged, head size, heads, sequences, longest, tokens, cus
      puts(heads_share_workgroups(a[0] != 0, (int)a[1], a[3], a[2], a[4], a[5], a[6]) ? "shared" : "single");
    scanf("%*[;\\n ]");
  }
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    folder = tmp_path_factory.mktemp("rules")
    (folder / "rules.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC_DIR}", str(folder / "rules.cpp"), "-o", str(folder / "rules")],
                   check=True)

    def ask(what, *sizes):
        line = " ".join([what, *map(str, sizes)]) + " ;\n"
        return subprocess.run([folder / "rules"], input=line, text=True, capture_output=True, check=True).stdout.strip()

    return ask


# us a layer: in the steps of the main loop, ahead of it, ahead of it with an fp32 intermediate
@pytest.mark.parametrize("E,local,k,T,H,I,us", [
    (128, 128, 8, 10, 1152, 512, (34.3, 34.5, 40.9)), (128, 128, 8, 23, 1152, 512, (48.3, 45.9, 51.8)),
    (256, 128, 8, 7, 1280, 1152, (33.2, 34.0, 39.3)), (128, 64, 8, 16, 1536, 768, (38.8, 39.0, 44.5)),
    (32, 32, 4, 8, 1536, 1280, (34.4, 34.1, 38.1)), (64, 64, 8, 3, 4096, 1024, (56.6, 56.5, 58.6)),
    (64, 64, 6, 8, 3584, 640, (52.9, 53.0, 54.9)), (128, 128, 8, 14, 4096, 256, (55.9, 57.0, 57.4)),
    (64, 64, 8, 6, 4096, 1024, (100.6, 99.3, 88.6)), (128, 128, 8, 8, 2048, 768, (60.4, 57.0, 53.7)),
    (16, 16, 4, 3, 1152, 1664, (20.2, 20.7, 21.9)), (64, 64, 8, 18, 1152, 256, (22.8, 23.1, 25.0)),
    (64, 64, 6, 1, 2048, 1408, (28.6, 27.0, 25.3)), (64, 64, 6, 8, 2048, 1408, (63.5, 60.7, 65.7)),
    (256, 64, 8, 4, 2688, 896, (33.5, 33.3, 25.8)), (8, 8, 2, 1, 4096, 4096, (43.5, 43.0, 32.8)),
])
def test_fp8_few_rows(rule, E, local, k, T, H, I, us):
    chosen = us[("steps", "ahead", "f32").index(rule("few", E, local, k, T, H, I, 256))]
    assert chosen <= 1.02 * min(us)


@pytest.mark.parametrize("E,local,k,T,H,I", [(1, 1, 1, 1, 128, 128), (8, 8, 8, 3, 4224, 128), (4, 1, 4, 100, 4096, 4224),
                                             (256, 256, 8, 10 ** 6, 16384, 128)])
def test_fp8_few_rows_at_the_ends(rule, E, local, k, T, H, I):
    form = rule("few", E, local, k, T, H, I, 256)
    assert form in ("steps", "ahead", "f32") and (H <= 4096 or form == "steps") and (I <= 4096 or form != "f32")


# us a layer with this GEMM's waves side by side and its rows in tiles of 16: 48 44 24 42 22 41 11
SHAPES = ("48", "44", "24", "42", "22", "41", "11")


@pytest.mark.parametrize("gated,E,local,rows,columns,K,us", [
    (0, 8, 8, 43.75, 2432, 2560, (86.1, 88.7, 80.9, 88.3, 91.1, 104.8, 95.4)),
    (0, 16, 16, 67.5, 1792, 1280, (65.5, 73.5, 74.6, 84.2, 78.9, 102.3, 87.9)),
    (0, 16, 16, 106.25, 1408, 3968, (144.7, 134.7, 143.0, 174.9, 165.4, 231.4, 208.8)),
    (1, 16, 16, 77.25, 640, 1536, (50.7, 52.0, 55.0, 50.2, 52.6, 66.2, 65.1)),
    (1, 8, 4, 69.25, 2816, 2816, (78.2, 74.9, 80.5, 71.5, 74.5, 105.9, 97.6)),
    (1, 8, 8, 117.5, 896, 3200, (82.9, 73.5, 57.3, 67.7, 72.5, 107.9, 100.1)),
    (1, 16, 8, 42.5, 1280, 1024, (48.7, 44.5, 41.0, 43.6, 44.7, 45.7, 46.1)),
    (1, 16, 8, 48.5, 1024, 3840, (82.9, 80.7, 62.0, 74.2, 57.3, 80.6, 82.2)),
    (1, 16, 8, 30.0, 1152, 2432, (62.6, 59.8, 48.0, 58.0, 46.8, 59.1, 54.3)),
    (1, 16, 16, 66.0, 640, 3840, (86.9, 84.0, 85.7, 79.8, 86.0, 131.1, 110.2)),
    (0, 16, 16, 36.0, 1280, 1792, (59.3, 63.3, 55.5, 62.0, 60.6, 62.4, 62.3)),
    (0, 8, 8, 48.0, 2048, 3840, (93.1, 104.6, 84.9, 98.9, 81.8, 105.3, 106.0)),
    (0, 16, 8, 61.25, 2688, 2176, (88.6, 89.7, 78.6, 85.4, 87.3, 111.3, 100.1)),
    (0, 16, 8, 89.75, 2944, 896, (82.1, 78.9, 81.2, 85.3, 82.2, 95.9, 91.2)),
    (0, 32, 16, 102.875, 1408, 768, (62.3, 58.3, 61.1, 64.5, 61.6, 74.0, 71.7)),
    (0, 16, 8, 120.0, 2432, 384, (66.8, 64.9, 67.0, 67.0, 65.6, 71.0, 73.5)),
    (1, 16, 16, 273.75, 1664, 1536, (139.1, 164.5, 162.8, 219.1, 208.7, 338.5, 317.8)),
    (1, 8, 8, 26.25, 1152, 1152, (35.8, 36.9, 32.5, 36.1, 31.2, 35.3, 34.3)),
])
def test_16bit_shapes(rule, gated, E, local, rows, columns, K, us):
    chosen = us[SHAPES.index(rule("shape", gated, E, local, int(rows * E), columns, 2 * K, 256))]
    assert chosen <= 1.02 * min(us)


def test_16bit_shapes_have_kernels(rule):
    seen = {rule("shape", g, E, E, int(r * E), c, 2048, 256) for g in (0, 1) for E in (1, 4, 16, 256)
            for r in (0.1, 5, 12, 21, 26, 40, 58, 66, 83, 100, 1000) for c in (64, 704, 2816)}
    assert seen == set(SHAPES)


FIFTEEN = [137, 211, 84, 125, 190, 249, 66, 173, 228, 101, 152, 97, 240, 118, 77]  # short prompts
CHATS = [42, 26, 28, 20, 57, 50, 26, 39, 40, 35, 58, 55, 48, 16, 18]                # short turns


# us with a head per workgroup and with heads that share them
@pytest.mark.parametrize("paged,D,heads,lens,us", [
    (0, 128, 8, [2000, 1500] + FIFTEEN[:14], (35.2, 36.8)), (0, 128, 8, [4000] + FIFTEEN, (63.2, 64.7)),
    (0, 64, 16, [8000] + CHATS, (162.8, 164.9)), (0, 256, 8, [1900, 1500] + CHATS[:14], (58.0, 59.2)),
    (0, 128, 32, [672, 180, 145, 416, 574, 213, 541, 376, 214, 121, 533, 308, 557, 591, 544, 399], (55.5, 51.1)),
    (0, 128, 28, [4000] + FIFTEEN, (133.5, 128.6)), (0, 256, 28, [1024] * 8, (214.7, 201.4)),
    (1, 64, 32, [1000] + CHATS, (78.8, 86.4)), (1, 256, 16, [1000] + CHATS, (215.2, 235.6)),
    (1, 128, 28, [2000] + FIFTEEN, (97.0, 87.0)), (1, 256, 16, [700] * 8, (289.7, 276.0)),
    (1, 128, 32, [430, 483, 571, 314, 538, 427, 326, 380], (185.4, 190.6)), (1, 128, 32, [512] * 8, (222.1, 219.0)),
    (1, 128, 32, [38, 53, 106, 97, 45, 59, 57, 39, 99, 65, 93, 80, 68, 101, 98, 72, 46, 94], (29.0, 30.9)),
])
def test_heads_that_share_workgroups(rule, paged, D, heads, lens, us):
    form = rule("share", paged, D, heads, len(lens), max(lens), sum(lens), 256)
    assert us[("single", "shared").index(form)] == min(us)


def test_unknown_tokens_count_as_part_of_the_longest(rule):
    ask = lambda n, tokens: rule("share", 0, 128, 32, n, 1024, tokens, 256)  # noqa: E731
    assert ask(2, 2 * 1024) == ask(2, 0) == "single" and ask(8, 8 * 1024) == ask(8, 0) == "shared"
