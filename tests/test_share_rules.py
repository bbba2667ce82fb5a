"""The rules by which a head's keys are shared out over workgroups (csrc/attn_decode_rules.h), walked over all sizes on the CPU: the second of
two launches adds up what the first has written, so there have to be at least two shares of which none is empty, and room for them."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton_amd", "csrc")
WALK = r"""
#include <cstdio>
#include "attn_decode_rules.h"
using namespace trn;
static long bad = 0, split = 0;
static void look(int bh, int kv, int keys, int d) {
    const int room = decode_splits(bh, keys), ns = few_query_shares(bh, kv, keys, d), blocks = (keys + 31) / 32;
    const int per = (blocks + ns - 1) / ns;
    split += ns > 1;
    // a workspace of trn_attn_workspace_bytes: shares, and no more than it holds; every share begins inside the keys; never more than one a CU
    if (ns < 1 || (room > 1 && (ns < 2 || ns > room)) || (ns - 1) * per >= blocks || ns * bh > 256) {
        if (bad++ < 5) std::printf("%d heads on %d, %d keys, head_dim %d: room for %d shares, %d taken\n", bh, kv, keys, d, room, ns);
    }
}
int main() {
    for (int d = 64; d <= 128; d += 64)
        for (int bh = 1; bh <= 130; ++bh)
            for (int kv = 1; kv <= bh; ++kv) {
                if (bh % kv) continue;
                for (int keys = 1; keys <= 20000; keys += 31) look(bh, kv, keys, d);
                for (int at : {2000, 2048, 4096, 8192, 2600 + 74 * kv, 3300 + 24 * kv, 2500 + 27 * kv})
                    for (int keys = at - 2; keys <= at + 2; ++keys) look(bh, kv, keys, d);
                for (int keys = 32768; keys <= 1 << 20; keys += 32749) look(bh, kv, keys, d);
            }
    std::printf("%ld shared out, %ld wrong\n", split, bad);
    return bad != 0;
}
"""


def test_two_launches_have_two_shares(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(WALK)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and int(r.stdout.split()[0]) > 100000, r.stdout
