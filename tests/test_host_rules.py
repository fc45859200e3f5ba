"""Rules of the launchers that are host code: what a product refuses before anything is launched, and which form a call takes."""
from helpers import host_program

# tokens of a pass -> shares of k of a 4,096 x 12,288 product whose rows a norm follows
SHARES = {385: 4, 600: 3, 1000: 2, 1153: 3}
# (rows, inputs, tokens) of a bfloat16 product -> 32 and 128 in a tile's tokens and rows, whether k goes in shares: every form there is
FORMS = {(100, 64, 33): (2, 1, False), (1000, 1088, 200): (2, 1, False), (130, 2112, 700): (2, 1, True), (8200, 2112, 400): (2, 2, False),
         (4200, 4160, 129): (2, 2, True), (12300, 2112, 129): (4, 1, False), (8200, 3136, 65): (4, 1, True), (4200, 2112, 1000): (4, 2, False),
         (3000, 6208, 700): (4, 2, True)}

PROGRAM = r"""
#include <stdio.h>

#include "layers.hpp"

int main() {
  // places of 64 KB: none is read or written
  auto place = [](int i) { return (void*)(((uintptr_t)i + 1) << 16); };
  DenseArgs a;
  a.w = place(0);
  a.k = 256;
  a.M = 1;
  a.n_seg = 2;
  for (int i = 0; i < 2; ++i) {
    a.seg[i].x = place(1);
    a.seg[i].ldx = 256;
    a.seg[i].y = place(2 + i);
    a.seg[i].ldy = 256;
    a.seg[i].row0 = 256 * i;
    a.seg[i].rows = 256;
  }
  JoinArgs j;
  j.x = (float*)place(4);
  j.x_out = (float*)place(5);
  j.M = 1;
  j.width = j.ldo = j.ldg = j.ldh = 256;
  j.y = (const float*)place(6);
  j.y_gate = (const float*)place(7);
  j.pairs = (const float*)place(8);
  j.ids = (const int32_t*)place(9);
  j.weights = (const float*)place(10);
  j.top = 2;
  j.experts = 4;
  j.h = place(11);
  j.gate = place(12);
  j.w_post = (const float*)place(13);
  j.out = place(1);
  const void* const reads[] = {j.x, j.y, j.y_gate, j.pairs, j.ids, j.weights, j.h, j.gate};
  for (int f32 = 0; f32 < 2; ++f32) {
    printf("%d\n", launch_dense(a, f32 != 0, nullptr, nullptr, &j));  // nothing shared: the launch alone fails here
    for (const void* r : reads)
      for (int i = 0; i < 2; ++i) {
        DenseArgs b = a;
        b.seg[i].y = const_cast<void*>(r);
        printf("%d\n", launch_dense(b, f32 != 0, nullptr, nullptr, &j));
      }
  }
}
"""


def test_a_product_does_not_write_what_the_sublayers_end_in_it_reads(lib, tmp_path):
    """every workgroup reads the end's operands: one that starts late would read another's outputs"""
    bad_argument, no_device = 1, 3
    assert host_program(tmp_path, PROGRAM) == ([no_device] + 16 * [bad_argument]) * 2


def test_parts_of_a_window_that_their_own_launch_adds_up(lib, tmp_path):
    """few parts of heads with a kv head each; others would be added up one after the other by a single workgroup"""
    shapes = [(8, 8, 1024, 8192), (8, 8, 0, 1024), (8, 8, 64, 8192), (8, 8, 1025, 8192), (8, 8, 0, 8192), (8, 8, 0, 32768),
              (8, 4, 1024, 8192), (8, 1, 128, 8192)]
    calls = "".join('printf("%%d\\n", (int)window_counted_parts(%d, %d, %d, %d));' % s for s in shapes)
    got = host_program(tmp_path, '#include <stdio.h>\n#include "layers.hpp"\nint main() { %s }' % calls)
    assert got == [1, 1, 0, 0, 0, 0, 0, 0]


def test_products_beside_the_attention_of_a_window(lib, tmp_path):
    """behind some thousand workgroups, most of them without keys, a product took up to 18 % longer a token than by itself"""
    calls = [(32, 32, 1024, 131072, 50 << 20), (32, 32, 0, 1024, 50 << 20), (32, 32, 0, 1025, 50 << 20), (32, 32, 0, 32768, 50 << 20),
             (16, 16, 0, 4096, 12 << 20), (16, 16, 0, 4096, 17 << 20), (16, 16, 0, 4097, 12 << 20), (8, 8, 0, 131072, 1 << 20),
             (32, 4, 0, 8192, 50 << 20), (32, 2, 0, 8192, 50 << 20), (12, 3, 0, 8192, 17 << 20)]
    lines = "".join("""{ WindowAttnArgs a; a.heads = %d; a.kv_heads = %d; a.window = %d; a.len_bound = %d; a.kl.row = a.vl.row = 128; a.M = 1;
                         a.parts = (float*)16; printf("%%d\\n", (int)window_takes_product(a, false, %d)); }""" % c for c in calls)
    got = host_program(tmp_path, '#include <stdio.h>\n#include "layers.hpp"\nint main() { %s }' % lines)
    assert got == [1, 1, 0, 0, 1, 0, 0, 0, 1, 1, 1]


def test_few_queries_of_a_window_in_binary32(lib, tmp_path):
    """tiles of sixteen queries took 4 to 15 % longer; heads of 64, other products of heads and queries, more keys and no window are theirs"""
    calls = [(8, 48, 1024, 0, 128), (8, 49, 1024, 0, 128), (8, 4, 1024, 316, 128), (8, 4, 1024, 317, 128), (8, 20, 300, 3000, 128), (8, 22, 300, 3000, 128),
             (8, 4, 0, 0, 128), (8, 4, 1024, 0, 64), (12, 32, 1024, 0, 128), (1, 320, 1024, 0, 128), (1, 321, 1024, 0, 128)]
    lines = "".join("""{ WindowAttnArgs a; a.heads = a.kv_heads = %d; a.M = %d; a.window = %d; a.pos.pos0 = %d; a.kl.row = a.vl.row = %d;
                         printf("%%d\\n", (int)window_few_queries(a)); }""" % c for c in calls)
    got = host_program(tmp_path, '#include <stdio.h>\n#include "layers.hpp"\nint main() { %s }' % lines)
    assert got == [1, 0, 1, 0, 1, 0, 0, 0, 1, 1, 0]


def test_norms_that_are_part_of_their_product(lib, tmp_path):
    """a wavefront per group, a few turns at most: each turn waits for memory behind the one ahead"""
    program = """
#include <stdio.h>
#include "layers.hpp"
int main() {
  for (int groups : {1, 4, 8, 16, 24, 32, 64, 256, 512}) {
    NormConvArgs n;
    n.M = 1;
    n.width = groups == 24 ? 1536 : groups == 1 ? 256 : 2048 < 256 * groups ? 2048 : 256 * groups;
    n.groups = groups;
    n.ld = n.width;
    printf("%d\\n", (int)dense_norm_fused(n, false));
  }
}
"""
    assert host_program(tmp_path, program) == [0, 1, 1, 1, 1, 0, 0, 0, 0]


def test_prompt_positions_that_go_together(lib, tmp_path):
    """the deeper in a sequence, the more of them it takes: a step's attention is cut over workgroups, the pass's is not"""
    calls = "".join('printf("%%d\\n", (int)canon_prompt_from(%d, %d));' % s for s in
                    [(12288, 0), (12288, 1000), (12288, 2000), (4096, 0), (4096, 1500), (4096, 2000), (16384, 0), (16384, 1500)])
    got = host_program(tmp_path, '#include <stdio.h>\n#include "common.hpp"\nint main() { %s }' % calls)
    assert got == [3, 4, 5, 4, 5, 6, 3, 5]


def test_shares_of_the_second_matrix(lib, tmp_path):
    calls = [(4096, 12288, m) for m in list(SHARES) + [256, 1408]] + [(4096, 4096, 1000), (8320, 8192, 385)]
    lines = "".join('printf("%%d\\n", gemm_norm_shares(%d, %d, %d));' % c for c in calls)
    got = host_program(tmp_path, '#include <stdio.h>\n#include "common.hpp"\nint main() { %s }' % lines)
    assert got == list(SHARES.values()) + [0] * 4


def test_products_of_17_to_64_tokens_with_operands_of_a_wavefronts_own(lib, tmp_path):
    """rows per workgroup, 0: another kernel; m, k, tokens, whether there is room for the sums of a cut k"""
    rows = {(4096, 4096): (16, 16, 16, 16, 16), (8192, 4096): (32,) * 5, (12288, 4096): (48,) * 5, (16384, 4096): (64, 64, 64, 64, 0),
            (2048, 4096): (16,) * 5, (1024, 4096): (16, 16, 16, 16, 0), (4096, 2048): (16, 16, 16, 16, 0), (2048, 2048): (16,) * 5,
            (8192, 2048): (32, 32, 32, 32, 0), (10240, 2048): (0, 0, 48, 48, 0), (20480, 2048): (0,) * 5, (4096, 12288): (64, 64, 64, 64, 0),
            (3072, 12288): (48,) * 5, (128, 12288): (16,) * 5, (6144, 12288): (0,) * 5, (4096, 8192): (0,) * 5}
    tokens = (17, 32, 33, 48, 49)
    calls = [(*shape, t, 1) for shape in rows for t in tokens] + [(4096, 4096, 16, 1), (4096, 4096, 65, 1), (4096, 4096, 64, 0), (4096, 12288, 17, 0)]
    lines = "".join('printf("%%d\\n", gemm_panel_rows(%d, %d, %d, %d));' % c for c in calls)
    got = host_program(tmp_path, '#include <stdio.h>\n#include "common.hpp"\nint main() { %s }' % lines)
    assert got == [r for five in rows.values() for r in five] + [0, 0, 16, 0]
    plans = [(4096, 12288, 17, 1), (4096, 12288, 48, 1), (2048, 12288, 64, 1), (4096, 12288, 49, 1), (4096, 12288, 48, 0)]
    assert [lib.awq_gemm_plan(*p) for p in plans] == [9, 9, 9, 1, 1]


def test_shares_of_tiles_of_64_tokens(lib, tmp_path):
    """of Wo and W2 behind prompts of 129 to 512 tokens; the other kernels have the rest"""
    calls = [(4096, k, n) for k in (4096, 12288) for n in (128, 129, 192, 193, 200, 256, 257, 320, 321, 385, 512, 513)]
    lines = "".join('printf("%%d\\n", gemm_norm_shares64(%d, %d, %d));' % c for c in calls)
    got = host_program(tmp_path, '#include <stdio.h>\n#include "common.hpp"\nint main() { %s }' % lines)
    assert got == [0, 4, 4, 4, 4, 4, 0, 0, 2, 2, 2, 0] + [0, 4, 4, 4, 4, 4, 0, 0, 0, 0, 0, 0]


def forms_of(tmp_path, shapes):
    program = """
#include <stdio.h>
#include "layers.hpp"
int main() {
  const int shapes[][3] = {%s};
  for (const auto& s : shapes) {
    DenseArgs a;
    a.k = s[1];
    a.M = s[2];
    a.out = DENSE_F32;
    a.workspace = (float*)16;
    a.workspace_floats = 1 << 25;
    const DenseForm f = dense_form(a, round_up(s[0], kDenseRowAlign));
    printf("%%d %%d %%d\\n", f.tt, f.rb, f.cuts > 1);
  }
}
""" % ", ".join("{%d, %d, %d}" % s for s in shapes)
    got = host_program(tmp_path, program)
    return [tuple(got[i:i + 3]) for i in range(0, len(got), 3)]


def test_forms_of_products_of_many_tokens(lib, tmp_path):
    assert forms_of(tmp_path, FORMS) == list(FORMS.values())
    assert len(set(FORMS.values())) == 8


def test_forms_that_are_near_the_fastest(lib, tmp_path):
    """long rows, and many tokens of short ones: forms that were timed within 6 % of the fastest of all (those that an estimate fitted
    without such shapes took were 13 to 26 % behind them)"""
    near = {(512, 12288, 2048): [(2, 2), (4, 2)], (10752, 15232, 98): [(4, 1), (4, 2)], (6144, 12288, 98): [(4, 1)], (2304, 14720, 512): [(4, 2)],
            (4096, 16384, 278): [(4, 2)], (2304, 14720, 2048): [(4, 2)], (10240, 8320, 160): [(4, 2)], (2816, 512, 1500): [(2, 1)],
            (4096, 512, 1500): [(2, 1)]}
    for shape, form in zip(near, forms_of(tmp_path, near)):
        assert form[:2] in near[shape], shape


def test_shares_of_binary32_products(lib, tmp_path):
    """timed within 5 % of the fastest form, weights of either kind; 8 shares instead of the first three's, or none, were 6 to 13 % behind it"""
    shapes = {(1024, 4096, 33): 16, (1024, 4096, 64): 16, (2048, 4096, 8): 13, (4096, 512, 48): 4, (7168, 512, 32): 4}
    calls = "".join("{ DenseArgs a; a.k = %d; a.M = %d; a.out = DENSE_F32; a.workspace = (float*)16; a.workspace_floats = 1 << 25;"
                    " const DenseForm f = dense_form_f32(a, %d); printf(\"%%d %%d %%d\\n\", f.tt, f.rb, f.cuts); }" % (k, m, r) for r, k, m in shapes)
    got = host_program(tmp_path, "#include <stdio.h>\n#include \"layers.hpp\"\nint main() { %s }" % calls.replace("\n", "\\n"))
    assert got == [v for cuts in shapes.values() for v in (1, 1, cuts)]
