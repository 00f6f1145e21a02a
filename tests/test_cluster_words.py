"""The geometry of a clustered launch in two words (cluster_words.h): for every number of strips, sequences and members that a launch can
have, each workgroup finds its strip, its sequence and its place in the cluster.  The header is compiled for the host."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ane_amd", "csrc")

PROGRAM = r"""
#include "cluster_words.h"
#include <stdio.h>
int main() {
    long launches = 0;
    for (int members = 2; members <= 8; members *= 2)
        for (int strips = 1; strips * members <= 2048; strips++)
            for (int batch = 1; strips * batch * members <= 2048; batch++, launches++) {
                const int nblk = strips * batch * members, rows = 1 + (strips * 37 + batch) % 512;
                const unsigned a = cluster_word_a(nblk, members, rows), b = cluster_word_b(strips);
                if (cluster_nblk(a) != nblk) return 1;
                for (int blk = 0; blk < nblk; blk++) {
                    const ClusterGeo g = cluster_of(a, b, blk);
                    if (g.blk != blk || g.csplit != members || g.rows_pm != rows || g.member != blk % members || g.first != blk - blk % members ||
                        g.strip != blk / members % strips || g.slab != blk / members / strips) {
                        printf("members %d strips %d batch %d workgroup %d\n", members, strips, batch, blk);
                        return 1;
                    }
                }
            }
    printf("%ld\n", launches);
    return 0;
}
"""


def test_every_workgroup_of_every_launch(tmp_path):
    src, exe = tmp_path / "words.cpp", tmp_path / "words"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and int(out.stdout) > 10000, out.stdout
