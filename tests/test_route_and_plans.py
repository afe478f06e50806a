"""Host side of bw_qlinear_ws and bw_qdgrad, without a GPU: the memory of searched plans, the choice between the batch and the prefill kernel,
slices of the input gradient."""
import os
import subprocess

import pytest
import torch

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


# (K, N, rows, bits, group, us of the batch kernel, us of the prefill kernel) on an MI355X, float16 x unless marked: calls on which the two
# differ by 8 % and more.  Beside each the prefill kernel's tile height, or what sets its time.  (All but the last seven
# were timed with two sets of x in flight; with one most of them take less, and the call of 770 rows, 70.0 then, changed sides.)
MEASURED = [
    (4096, 14336, 80, 4, 128, 24.0, 27.4), (2048, 2048, 333, 4, 128, 10.8, 20.4), (4096, 4096, 316, 4, 128, 21.1, 25.9),
    (13824, 5120, 140, 4, 32, 40.3, 47.0), (8192, 8192, 334, 4, 128, 76.2, 61.2), (6912, 8048, 218, 4, 128, 46.9, 42.0),
    (11008, 4096, 434, 4, 64, 67.0, 55.8), (13824, 5120, 1539, 2, 128, 290.8, 230.9), (5120, 13824, 656, 4, 128, 132.7, 103.5),   # (the last two: 256)
    (4096, 11008, 310, 4, 128, 53.4, 46.1), (4096, 14336, 269, 4, 128, 53.2, 46.6), (4608, 10864, 321, 4, 128, 58.6, 51.9),      # one round, just over half full
    (4096, 4096, 1042, 2, 128, 55.0, 49.2), (5888, 8512, 396, 4, 128, 79.5, 69.1), (2304, 4432, 813, 4, 128, 37.0, 32.1),
    (14336, 4096, 107, 8, 32, 33.6, 37.5), (14336, 4096, 99, 8, 64, 34.8, 39.9),                                                # 64 (the second: bfloat16)
    (512, 6149, 299, 4, 128, 12.5, 18.6), (896, 6299, 399, 2, 128, 18.6, 24.1), (640, 4945, 389, 2, 128, 17.1, 24.7),            # rows of y off 8 bytes
    (11968, 3760, 359, 2, 64, 49.0, 57.8), (8768, 3520, 242, 2, 32, 33.3, 40.5),                                                # K % 128 != 0
    (3840, 5224, 770, 8, 32, 55.3, 62.6), (7040, 2944, 449, 8, 128, 35.3, 41.3),
    (576, 2704, 1065, 2, 64, 15.3, 19.9), (10624, 4883, 802, 8, 64, 126.1, 181.7), (704, 2976, 1117, 2, 32, 17.4, 21.1),         # beyond 512 rows, close by the models
    (1600, 5059, 1987, 2, 32, 67.5, 84.0), (12928, 6592, 649, 8, 128, 155.7, 212.5),
]


@pytest.mark.skipif(torch.cuda.is_available(), reason="the choice for 256 compute units, what the library assumes without a GPU")
@pytest.mark.parametrize("k,n,m,bits,g,batch,prefill", MEASURED)
def test_route_takes_the_faster_kernel(k, n, m, bits, g, batch, prefill):
    """bw_qlinear_workspace_bytes asks for room to cast a bfloat16 x only where the prefill kernel runs: that tells the route."""
    from bitween_amd.kernels import hip_loader
    need = hip_loader.load().bw_qlinear_workspace_bytes
    takes_prefill = need(m, n, k, bits, g, hip_loader.BW_BF16) > need(m, n, k, bits, g, hip_loader.BW_F16)
    assert takes_prefill == (prefill < batch)


@pytest.mark.skipif(torch.cuda.is_available(), reason="the route for 256 compute units, what the library assumes without a GPU")
@pytest.mark.parametrize("bits,g,n,k,m", [(4, 128, 512, 6400, 9), (4, 128, 2048, 8192, 16), (4, 128, 1024, 9216, 12), (2, 64, 512, 7168, 9), (2, 128, 2048, 8192, 16),
                                          (2, 64, 1024, 12288, 5), (4, 64, 512, 11264, 5), (4, 32, 512, 9216, 5), (8, 32, 768, 6400, 9)])
def test_short_narrow_calls_are_one_launch(bits, g, n, k, m):
    """Narrow layers whose decode kernel is done in less than an eager call of two launches and a workspace takes the host (8.1 us): K is not
    cut (1.08 ... 1.33 of the time in a loop of eager calls)."""
    from bitween_amd.kernels import hip_loader
    assert hip_loader.load().bw_qlinear_workspace_bytes(m, n, k, bits, g, hip_loader.BW_F16) == 0


@pytest.mark.skipif(torch.cuda.is_available(), reason="the plan for 256 compute units, what the library assumes without a GPU")
@pytest.mark.parametrize("m,n,k,slices", [
    (21, 5120, 1024, 20), (10, 4096, 1536, 16), (19, 2304, 2816, 9), (30, 1024, 4288, 6), (48, 1216, 5376, 5), (39, 2048, 2048, 11)])
def test_input_gradient_slices_are_whole_passes(m, n, k, slices):
    """The stepping kernel takes its steps of 32 rows of N in twos, so slices of an odd number of steps are not worth their number: 23 of 7
    instead of 20 of 8 steps cost 11 %."""
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    assert lib.bw_qdgrad_tile_rows(m, n, k, 4, 64) == 128
    need = lib.bw_qdgrad_workspace_bytes(m, n, k, 4, 64)
    assert need == -(-k // 128) * slices * m * 128 * 4                        # a partial tile is the call's m rows
    assert -(-(-(-n // 32)) // slices) % 2 == 0


@pytest.mark.skipif(torch.cuda.is_available(), reason="the plan for 256 compute units, what the library assumes without a GPU")
@pytest.mark.parametrize("m,n,k,bits,g,dtype,taken", [
    (16, 1024, 4096, 4, 128, 0, True), (16, 960, 4096, 4, 128, 0, False), (16, 1472, 4096, 2, 32, 1, True), (16, 1024, 4096, 4, 128, 1, False),
    (32, 1472, 4096, 8, 64, 0, True), (17, 1024, 4096, 4, 128, 0, False), (17, 7424, 4096, 8, 32, 1, True), (32, 6400, 4096, 4, 128, 1, False),
    (48, 7424, 4096, 4, 128, 0, True), (33, 6400, 4096, 4, 128, 0, False), (33, 11008, 4096, 4, 128, 1, False), (49, 11008, 4096, 4, 128, 0, False),
    (40, 8192, 4096, 8, 32, 0, False), (48, 9792, 4096, 8, 32, 0, True), (40, 8192, 4096, 2, 32, 0, True),
    (9, 6252, 4096, 4, 128, 0, False), (9, 4096, 4224, 4, 128, 0, False)])                 # n off eights, an odd number of groups
def test_input_gradients_of_few_rows_that_have_their_own_kernel(m, n, k, bits, g, dtype, taken):
    from bitween_amd.kernels import hip_loader
    assert (hip_loader.load().bw_qdgrad_rows_slices(m, n, k, bits, g, dtype) > 0) == taken


@pytest.mark.skipif(torch.cuda.is_available(), reason="the tiles for 256 compute units, what the library assumes without a GPU")
@pytest.mark.parametrize("m,n,k,bits,g,rows,cols", [
    (961, 12544, 384, 4, 128, 256, 256), (1406, 9200, 512, 4, 64, 256, 256), (961, 12548, 384, 4, 128, 128, 192), (961, 12544, 256, 4, 128, 128, 192),
    (300, 8192, 384, 4, 64, 128, 192)])
def test_prefill_tiles_of_few_k_steps(m, n, k, bits, g, rows, cols):
    """With three and four K steps a round of 256 x 256 tiles is not given up for 128 x 192 tiles that need a second one (1.06 of its time, up to 1.14)."""
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    assert (lib.bw_qgemm_tile_rows(m, n, k, bits, g), lib.bw_qgemm_tile_cols(m, n, k, bits, g)) == (rows, cols)
