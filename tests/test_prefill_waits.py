"""The waits that the prefill kernel counts by hand (frag_younger): for every tile the order of a wave's LDS operations is played through
and each slot's wait held against it.  Host code only."""
import os
import subprocess

import pytest

from bitween_amd.csrc import build

PROGRAM = r"""
#include "bw_qgemm_kernel.h"
#include <cstdio>
#include <vector>

struct Op { int kind, of; };                   // 0: fragment read of a slot, 1: words of region `of % NT` of MFMA step `of / NT`

template <int MT, int NT, int PW>
int tile(const char* name) {
    constexpr int RING = 8, MF = 4, SLOTS = MT * MF;
    std::vector<Op> done;
    int bad = 0;
    for (int s = 0; s < RING; s++) done.push_back({0, s});
    for (int g = 0; g < SLOTS * NT; g++) {
        const int S = g / NT, j = g % NT, t = S / MT, in_step = g - t * MT * NT, r = in_step / MT, k = in_step % MT;
        if (j == 0) {
            const int allowed = frag_younger<RING, SLOTS, MT, NT, PW>(S);
            // a 4-bit counter: 15 is no wait at all
            if (allowed < 0 || allowed > 14) { printf("%s slot %d: a wait for %d\n", name, S, allowed); bad++; }
            // the slot's fragment, and the words that unpacks beginning in this slot or before it take (handed over one MFMA step earlier); the
            // last gap of a slot is the read's and unpacks nothing
            const int last_region = (in_step + NT - 2) / MT;
            for (int i = 0; i < (int)done.size(); i++) {
                const bool needed = done[i].kind == 0 ? done[i].of == S : done[i].of <= (t - 1) * NT + last_region;
                const int younger = (int)done.size() - 1 - i;
                if (needed && younger < allowed) { printf("%s slot %d: %d younger operations, waits for %d\n", name, S, younger, allowed); bad++; }
            }
        }
        if (PW && k >= hand_gap(NT) && k < hand_gap(NT) + PW) done.push_back({1, t * NT + r});
        if (j == NT - 1 && S + RING < SLOTS) done.push_back({0, S + RING});
    }
    return bad;
}

int main() {
    int bad = 0;
    bad += tile<4, 4, 0>("64 x 256") + tile<8, 4, 0>("128 x 256") + tile<16, 4, 0>("256 x 256") + tile<8, 3, 0>("128 x 192") + tile<16, 3, 0>("256 x 192");
    bad += tile<4, 4, 2>("64 x 256, 8 bits") + tile<8, 4, 2>("128 x 256, 8 bits") + tile<8, 3, 2>("128 x 192, 8 bits");
    return bad != 0;
}
"""


def test_every_slot_waits_for_what_it_uses(tmp_path):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "waits.hip", tmp_path / "waits"
    src.write_text(PROGRAM)
    subprocess.run([hipcc, "--offload-arch=gfx950", "-std=c++17", "-O1", "--cuda-host-only", "-I" + build.HERE, "-o", str(exe), str(src)],
                   check=True, capture_output=True, text=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
