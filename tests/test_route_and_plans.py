"""Host side of bw_qlinear_ws, without a GPU: the memory of searched plans."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bitween_amd", "csrc")

PLAN_CACHE_PROGRAM = r"""
#include "bw_plan_cache.h"
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
int main() {
    // four decoder models' layers (q/k/v/o, fused q/k/v, gate, fused gate + up, down) in two formats each, at one row count
    static BwPlanCache<long long> cache;
    const long long hidden[] = {2048, 4096, 5120, 8192}, inter[] = {5632, 11008, 13824, 28672};
    int most = 0;
    for (long long m : {17, 40, 64, 128, 512, 2048})
        for (int model = 0; model < 4; model++)
            for (int key : {(4 * 2 + 1) * 256 + 128, (8 * 2 + 1) * 256 + 32}) {
                const long long h = hidden[model], f = inter[model];
                const long long shapes[5][2] = {{h, h}, {3 * h, h}, {f, h}, {2 * f, h}, {h, f}};
                int searched = 0;
                for (int pass = 0; pass < 3; pass++)
                    for (auto& s : shapes) {
                        const long long want = m * 1000003 + s[0] * 31 + s[1] * 7 + key;
                        if (cache.get(m, s[0], s[1], key, [&] { searched++; return want; }) != want) return 1;
                    }
                most = searched > most ? searched : most;
            }
    std::printf("%d\n", most);
    // a set of three shapes: the older one goes, values stay those of their shapes
    for (int i = 0; i < 100000; i++) {
        const long long m = 1 + std::rand() % 9, n = 32 * (1 + std::rand() % 9), k = 128 * (1 + std::rand() % 9);
        if (cache.get(m, n, k, 7, [&] { return m * n + k; }) != m * n + k) return 2;
    }
    return 0;
}
"""


def test_layers_of_a_model_keep_their_plans(tmp_path):
    """The five layer shapes of a model, called in turn, are searched once each: sizes that are all multiples of 32 (or 128) do not meet
    in one place of the cache."""
    source, binary = tmp_path / "cache.cpp", tmp_path / "cache"
    source.write_text(PLAN_CACHE_PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", str(binary), str(source)], check=True)
    out = subprocess.run([str(binary)], capture_output=True, text=True)
    assert out.returncode == 0, out.returncode
    assert int(out.stdout) == 5
