"""The LDS Jacobi's block addresses, from the header that the kernel is compiled
from, on the host: over the orbital counts of a molecule that takes it, every
address of every round lies inside the ring storage, and the blocks of a round
are the elements between its pairs, each once."""

import subprocess

import pytest

from dxtb_amd.build import PKG, ROOT, hipcc

SOURCE = r"""
#include <cstdio>
#include <vector>
#include "wg.h"
using namespace xtb;

static int check(int n, int W) {
    const int K = ring_pairs(n), m = 2 * K - 1, nblk = K * (K - 1) / 2, size = ring_doubles(n, W);
    for (int r = 0; r < m; ++r) {
        std::vector<int> hits(size, 0);
        for (int e = 0; e < (nblk > 0 ? nblk : 1); ++e) {
            const RingBlock x = ring_block(K, W, e / K, e % K);
            if (x.P < 0 || x.R < 0 || x.P >= K || x.R >= K) return 1;
            for (int u = 0; u < 4; ++u) {
                if (u < 2 && x.P == 0 && n % 2) continue;  // the dummy index of an odd n
                const int at = x.row[u] + (x.col[u] + r) % m;
                if (x.col[u] < 0 || x.col[u] >= m || at < 0 || at >= size) return 2;
                if (nblk > 0 && ++hits[at] > 1) return 3;
            }
        }
        // every element is in one block, on the diagonal or a pivot
        int own = 0;
        for (int h : hits) own += h;
        if (own != n * (n + 1) / 2 - n - n / 2) return 4;
    }
    return 0;
}

int main() {
    for (int n = 2; n <= 202; ++n)
        for (int pad = 0; pad < 4; ++pad) {
            const int W = 2 * ring_pairs(n) - 1 + pad;
            if (const int e = check(n, W)) {
                printf("n = %d, pitch %d: fault %d\n", n, W, e);
                return 1;
            }
        }
    printf("ok\n");
    return 0;
}
"""


def test_block_addresses_stay_in_the_ring(tmp_path):
    try:
        cc = hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    src, exe = tmp_path / "ring.hip", tmp_path / "ring"
    src.write_text(SOURCE)
    subprocess.run([cc, "-O1", "-std=c++17", "--offload-arch=gfx950", "--offload-host-only", f"-I{PKG / 'csrc'}",
                    f"-I{ROOT / 'include'}", str(src), "-o", str(exe)], check=True, capture_output=True, timeout=300)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout
