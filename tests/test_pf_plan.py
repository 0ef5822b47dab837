"""The cut of a prefill pass and its scratch (qwengine_amd/csrc/pf_plan.hpp), on the CPU, for the built tile shape and for
the others that the build options QWA_PF_WAVES / QWA_PF_RT name: no pass takes more token-splits than its workspace
holds, a workspace for a longer pass covers every shorter one, and the exchange of partial states through LDS is used
only where every wave's area lies inside the ring."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r'''
#include <stdio.h>
#include "pf_plan.hpp"
using namespace qwa;
#define CHECK(c, ...) do { if (!(c)) { fprintf(stderr, __VA_ARGS__); return 1; } } while (0)
int main() {
    const int ends[] = {1, 32, 33, 200, 257, 1000, 2049, 20088, 81920, 81921, MAX_POS};
    for (int nb = 1; nb <= PF_MAXB; nb++) {
        CHECK(nb == 1 || pf_token_splits(nb) >= pf_token_splits(nb - 1), "size decreases at %d tokens\n", nb);
        for (int npos : ends) {
            if (npos < nb) continue;
            const int ns = pf_splits(nb, npos), tiles = (npos - 1) / PF_TILE + 1;
            CHECK(ns >= 1 && (pf_row_blocks(nb) > PF_FEW || ns <= tiles), "%d splits of %d tiles\n", ns, tiles);
            CHECK(pf_row_blocks(nb) > PF_FEW || pf_row_blocks(nb) * NKV * ns <= 256, "%d tokens: over one round\n", nb);
            CHECK(ns <= 64, "%d splits: more than the lanes of the combine\n", ns);
            CHECK(ns * nb <= pf_token_splits(nb), "%d tokens at %d: %d splits in %d token-splits\n", nb, npos, ns,
                  pf_token_splits(nb));
        }
    }
    // the last wave's last 8-byte unit of the exchange
    const long last = (PF_WAVES - 1) * (long)PF_XCH_BYTES + 8 * (64 * 15 + 63) + 8;
    CHECK(!PF_XCH_FITS || last <= (long)PF_IMG_NBUF * PF_IMG_BYTES, "exchange past the ring\n");
    CHECK(QWA_PF_WAVES != 8 || PF_XCH_FITS, "the built shape lost the exchange\n");
    return 0;
}
'''


@pytest.mark.parametrize("waves,rt", [(8, None), (8, 1), (8, 4), (4, None), (12, None), (16, None), (16, 2)])
def test_workspace_holds_every_pass(tmp_path, waves, rt):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(SRC)
    cmd = ["g++", "-std=c++17", "-Wall", "-Werror", f"-DQWA_PF_WAVES={waves}"] + ([f"-DQWA_PF_RT={rt}"] if rt else [])
    subprocess.run([*cmd, "-I", os.path.join(ROOT, "qwengine_amd", "csrc"), "-I", os.path.join(ROOT, "include"), str(src),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def test_longer_passes_take_the_instantiated_split_counts(tmp_path):
    """Past 12 row blocks: 6, 7 or 8 splits, each of them by some pass (the combine is built for these)."""
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text('#include <stdio.h>\n#include "pf_plan.hpp"\nint main() { for (int nb = 513; nb <= 1024; nb++) '
                   'printf("%d ", qwa::pf_splits(nb, 262144)); }')
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "qwengine_amd", "csrc"), "-I",
                    os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
    counts = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    assert set(counts) == {"6", "7", "8"}
