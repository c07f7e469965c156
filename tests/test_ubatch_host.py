"""The host-computable parts of the batched GEMV (csrc/ubatch.hip), compiled
for the CPU: which bytes a weight item's loads depend on, and the split that a
launch takes (no GPU)."""
import os
import re
import subprocess

import pytest

from test_gpu_ubatch import EVERY_SPLIT

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "sinter-qwen36-nomtp-tu102_amd")

SRC = r"""
#include "ubatch.hip"
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
using namespace sinter;

// whether loading item i of n consecutive blocks depends on bytes around them
template <int WT>
static bool reads_outside(uint32_t n, uint32_t i, uint32_t g) {
    typedef WItem<WT> Item;
    alignas(16) unsigned char buf[2][64 + 8 * 210 + 64], item[2][sizeof(Item)];
    for (int p = 0; p < 2; p++) {
        memset(buf[p], p ? 0x5A : 0xA5, sizeof buf[p]);
        for (uint32_t k = 0; k < n * Item::BYTES; k++) buf[p][64 + k] = (unsigned char)(k * 37u + 11u);
        // (the object's representation, padding included)
        memset(item[p], 0, sizeof item[p]);
        Item *w = new (item[p]) Item;
        w->load(buf[p] + 64 + i * Item::BYTES, g);
    }
    return memcmp(item[0], item[1], sizeof(Item)) != 0;
}

template <int WT>
static void split(long rows, long k, long n_tok) {
    UbArgs a = {};
    a.nb = (uint32_t)(k / 256);
    a.n_tok = (uint32_t)n_tok;
    a.n_seg = 1;
    a.rows[0] = (uint32_t)rows;
    const UbSplit p = ub_split<WT>(a);
    const char *kernel = p.kernel == UbSplit::FEW ? "few" : p.kernel == UbSplit::MANY ? "many" : "short";
    printf("%s %u %llu\n", kernel, p.nt, (unsigned long long)p.wgs);
}

int main(int argc, char **argv) {
    if (argc > 1) {   // TYPE ROWS K TOKENS ...
        for (int i = 1; i + 3 < argc; i += 4)
            (atoi(argv[i]) == SINTER_Q4_K ? split<SINTER_Q4_K> : split<SINTER_Q6_K>)(atol(argv[i + 1]), atol(argv[i + 2]),
                                                                                     atol(argv[i + 3]));
        return 0;
    }
    for (uint32_t n = 1; n <= 8; n++)
        for (uint32_t i = 0; i < n; i++)
            for (uint32_t g = 0; g < 4; g++) {
                if (reads_outside<SINTER_Q4_K>(n, i, g)) printf("q4_k %u of %u group %u\n", i, n, g);
                if (reads_outside<SINTER_Q6_K>(n, i, g)) printf("q6_k %u of %u group %u\n", i, n, g);
            }
    return 0;
}
"""


@pytest.fixture(scope="module")
def host_prog(sn, tmp_path_factory):
    import build
    d = tmp_path_factory.mktemp("ubatch_host")
    (d / "t.hip").write_text(SRC)
    exe = d / "t"
    subprocess.run([build.hipcc(), "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
                    "-I", os.path.join(PKG, "csrc"), "-I", os.path.join(ROOT, "include"), str(d / "t.hip"), "-o", str(exe),
                    "-L", PKG, "-lsinter", "-Wl,-rpath," + PKG, "-Wl,--unresolved-symbols=ignore-all"],
                   check=True, capture_output=True)
    return str(exe)


def test_weight_loads_stay_in_the_operand(host_prog):
    """Matrices of 1 to 8 blocks (an odd number of 210-byte Q6_K blocks ends
    between 4-byte boundaries): no loaded register holds a byte outside."""
    assert subprocess.run([host_prog], check=True, capture_output=True, text=True).stdout == ""


def splits(host_prog, cases):
    """[(kernel, token tiles per workgroup, workgroups)] of (type, rows, k, tokens)."""
    args = [str(v) for c in cases for v in c[:4]]
    out = subprocess.run([host_prog, *args], check=True, capture_output=True, text=True).stdout.splitlines()
    return [(f[0], int(f[1]), int(f[2])) for f in map(str.split, out)]


def test_every_split_case_takes_the_split_it_names(host_prog):
    """The GPU test of every compiled split reaches each of them, whatever the
    prices that choose are fitted to next."""
    got = splits(host_prog, EVERY_SPLIT)
    assert [g[:2] for g in got] == [c[4:] for c in EVERY_SPLIT]
    src = open(os.path.join(PKG, "csrc", "ubatch.hip")).read()
    launch = src[src.index("hipError_t launch_ubatch("):src.index("hipError_t launch_gemv_ubatch(")]
    compiled = {(k, int(nt)) for f, k in (("launch_gemv<WT, {}>", "few"), ("launch_gemm<WT, {}>", "many"),
                                          ("launch_gemm<WT, {}, true>", "short"))
                for nt in re.findall(f.format(r"(\d+)"), launch)}
    assert compiled == {c[4:] for c in EVERY_SPLIT}


@pytest.mark.parametrize("t", [12, 14])
def test_split_fits_a_launch_wherever_64_row_tiles_do(host_prog, t):
    """A launch holds fewer than 2^32 threads (256 per workgroup): a matrix
    that fits one with 64 rows and 64 tokens per workgroup is never split finer
    than that allows, up to what 288 GB of weights hold."""
    cases = [(t, rows, k, n) for k in (256, 512, 768, 1024, 5120) for n in (1, 2, 4, 5, 16, 17, 33, 64, 65, 129)
             for rows in (2**22, 2**27, 2**28, 2**28 + 1, 300_000_000, 450_000_000, 2**30 - 64)
             if rows * (k // 256) * (144 if t == 12 else 210) < 288e9 and -(-rows // 64) * -(-n // 64) * 256 < 2**32]
    assert len(cases) > 100
    for c, g in zip(cases, splits(host_prog, cases)):
        assert g[2] * 256 < 2**32, (c, g)
