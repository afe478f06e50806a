// The batch kernel's plan, its reduction, and bw_qlinear, which sends a call to the decode, the batch or the prefill kernel.
#include "bw_plan_cache.h"
#include "bw_qbatch_kernel.h"

#include <stddef.h>

bool bw_fast_shape(int64_t M, int64_t N, int64_t K, int64_t ldx, int bits, int group);
float bw_qgemm_expected_us(int64_t M, int64_t N, int64_t K, int bits, int group);
bool bw_qgemm_small_workspace_serves(int64_t M, int64_t N, int64_t K, int bits, int group, size_t workspace_bytes);

namespace {

// y = sum over the splits of the partial sums, plus bias, rounded once.  A thread owns four columns of one row.
__global__ __launch_bounds__(256) void qbatch_reduce_kernel(const float* __restrict__ ws, const _Float16* __restrict__ bias, _Float16* __restrict__ y,
                                                            int M, int N, int npad, int ldy, int splits) {
    const int quads = npad >> 2, idx = (int)blockIdx.x * 256 + threadIdx.x;
    if (idx >= M * quads) return;
    const int m = idx / quads, n = (idx - m * quads) * 4;
    const float* p = ws + (int64_t)m * npad + n;
    const int64_t step = (int64_t)M * npad;
    f4 v = {0.f, 0.f, 0.f, 0.f};
    int s = 0;
    for (; s + 4 <= splits; s += 4) {
        f4 t[4];
#pragma unroll
        for (int i = 0; i < 4; i++) t[i] = *reinterpret_cast<const f4*>(p + (s + i) * step);
#pragma unroll
        for (int i = 0; i < 4; i++) v += t[i];
    }
    for (; s < splits; s++) v += *reinterpret_cast<const f4*>(p + s * step);
    _Float16 h[4];
#pragma unroll
    for (int e = 0; e < 4; e++) h[e] = (_Float16)(v[e] + (bias && n + e < N ? (float)bias[n + e] : 0.f));
    _Float16* dst = y + (int64_t)m * ldy + n;
    if (n + 3 < N && ldy % 4 == 0 && ((uintptr_t)y & 7) == 0) {
        *reinterpret_cast<u2*>(dst) = u2{as_u32(h2{h[0], h[1]}), as_u32(h2{h[2], h[3]})};
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (n + e < N) dst[e] = h[e];
    }
}

// ---- plan ----
struct BatchPlan { int mt, ntw, splits; };

inline int batch_mt(int64_t M) { const int t = (int)((M + 15) / 16); return t <= 4 ? t : t <= 6 ? 6 : 8; }

// Rows of 16 per tile, column tiles per wave and cuts of K for a call, from a model of the launch fitted to 270000 timings of 45000 calls
// (17 ... 640 rows, K 512 ... 14336, N 512 ... 22016, 2 / 4 / 8 bits, both activation types; rms error 6 %, its choice within 0.7 % of the
// best on average).  A round costs 0.20 MT + (0.39 + 0.16 at 8 bits) NTW us, of 256 values (MT > 4) 0.13 MT + (0.29 - 0.01 MT + 0.05 at 8 bits)
// NTW; every wave of workgroups (0.01 + 0.25 NTW) MT or (0.04 + 0.19 NTW) MT more, a launch 2.5 ... 3, a cut of K the reduction: 2 us and
// 1.5 us per million partial sums.  Four column tiles a wave halve the LDS traffic of 8 x 2 tiles for the same outputs: W4 g128 us, 128 rows of 4096
// -> 14336 float16 27.7 -> 25.6, bfloat16 30.2 -> 26.0; 14336 -> 4096 32.0 -> 28.5.  Not built at 8 bits: in
// 64-row tiles their weights spill 59 ... 135 registers; lower ones spill none (48 rows in groups of 32: 10 ... 13) and have not been timed.  Of the tiles
// that are, W4 g32 4 x 4 spills 12, W4 g64 4, W8 6 x 3 8 ... 12; the fit has their timings.
//
// Lower tiles than the call has rows read the weights (out of L2) once per tile, but fill the chip without a cut of K and its
// reduction: W4 g128 us, one tile of rows against the plan, 2048 x 2048 at 64 rows 8.5 -> 5.3, at 128 rows 11.4 -> 6.3; 4096 x 4096 at
// 64 rows 12.4 -> 8.8, at 128 rows 18.1 -> 12.2; 4096 -> 11008 at 128 rows 28.6 -> 23.8 (with two sets of x in flight).
struct BatchCost { BatchPlan plan; float us; bool ahead; };   // ahead: this kernel takes a call of 17 rows and more

// Calls that scale a group's sum in float32: the rows that are, or by bw_qlinear_decode_rows would be, the decode kernels'.
inline bool batch_sums(int64_t M, int64_t N, int64_t K, int bits, int group) {
    return bw_qbatch_sums(bits, group, 1, 1) && M <= bw_qlinear_decode_rows(N, K, bits);
}

BatchCost batch_search(int64_t M, int64_t N, int64_t K, int bits, int group, bool may_split) {
    const int nchunks = (int)((K + 127) / 128), cus = bw_device_cus(), whole = batch_mt(M);
    BatchCost best{{whole, 1, 1}, 1e30f, true};
    const bool sums = batch_sums(M, N, K, bits, group);
    for (const int mt : {1, 2, 3, 4, 6, 8}) {
        const int64_t mtiles = (M + 16 * mt - 1) / (16 * mt);
        if (mt > whole || (mt < 4 && mtiles > 4)) continue;   // (more tiles of few rows: not measured)
        const bool large = mt > 4;
        for (int ntw = 1; ntw <= (mt <= 4 ? bits == 8 ? 3 : 4 : mt == 6 ? 3 : 2); ntw++) {
            if (sums && !bw_qbatch_sums(bits, group, mt, ntw)) continue;
            const int64_t tiles = mtiles * ((N + 32 * ntw - 1) / (32 * ntw));
            const float b8 = bits == 8 ? 1.f : 0.f;
            float round = large ? 0.128f * mt + (0.291f - 0.009f * mt + (0.086f - 0.006f * mt) * b8) * ntw - 0.185f
                                : 0.196f * mt + (0.386f + 0.004f * mt + (0.155f - 0.005f * mt) * b8) * ntw - 0.081f;
            if (bits == 4 && group == 32 && ntw == 4) round *= 1.04f;   // (12 registers spill)
            const float wave = large ? (0.04f + 0.19f * ntw) * mt + 0.78f : (0.01f + 0.254f * ntw) * mt + 0.18f;
            for (int s = 1; s <= 16 && (s == 1 || (may_split && 2 * s <= nchunks)); s++) {
                const int cps = (nchunks + s - 1) / s, used = (nchunks + cps - 1) / cps, rounds = large ? (cps + 1) / 2 : (cps + 3) / 4;
                if (used != s || (s > 1 && M * N * s > ((int64_t)32 << 20))) continue;   // (128 MiB of partial sums)
                const float waves = (float)((tiles * s + cus - 1) / cus);
                const float us = (large ? 2.5f : 2.95f) + waves * (rounds * round + wave) + (s > 1 ? (large ? 1.7f : 2.3f) + 0.08f * s + 1.5e-6f * (float)M * (float)N * s : 0.f);
                if (us < best.us) best = {{mt, ntw, s}, us, true};
            }
        }
    }
    // what a format costs more or less than that; the plan stays
    best.us *= bits == 2 ? 0.965f : bits == 8 ? group == 32 ? 1.015f : 0.98f : group == 32 ? 1.03f : group == 64 ? 1.01f : 1.f;
    if (N % 4) best.us *= 1.02f;                              // rows of y off an 8-byte boundary
    // the chosen plan on a chip that others of the fit left idle: 2 % more, 9 % at 1 PFLOP/s (the clock comes down)
    best.us *= 1.02f + 0.14e-9f * (float)M * (float)N * (float)K / best.us;
    return best;
}

// 17 ... 64 rows: this kernel; on 1493 layers, formats and row counts there it takes 0.15 ... 0.94 of the time of the prefill kernel and of
// the decode kernels in launches of 16 rows (W4 g128 at 64 rows, us, prefill kernel against this one: 4096 x 4096 17.8 -> 8.8, 4096 ->
// 11008 20.9 -> 17.2, 11008 -> 4096 24.8 -> 18.9; 2048 x 2048 13.3 -> 5.3).  Beyond, whichever is expected to be done first: the prefill
// kernel's 128 x 256 tiles leave the chip idle on most layers of a few hundred rows, or have to be cut along K (W4 g128, us, prefill
// against this: 2048 x 2048 at 333 rows 20.4 -> 10.8, at 768 rows 26.7 -> 14.5; 4096 x 4096 at 256 rows 28.6 -> 17.6, at 512
// rows 32.4 -> 30.0, but at 768 rows 39.8 against 47.9; 4096 -> 14336 at 128 rows 31.3 -> 27.4, at 160 rows 41.5 against 42.9, at 269
// 46.5 against 53.2; 4096 -> 11008 at 310 rows 46.1 against 53.4; 512 -> 13056 at 200 rows 11.3 against 15.2).  The models
// are of float16 x; bfloat16 costs this kernel 4 % and the prefill kernel a cast (3.2 us and 0.5 us per million values).  Both types take
// one route, so that a bfloat16 x and its float16 rounding give the same bits: half of both is added.  A doubtful call of up
// to 128 rows stays here (1.06: in eager code the prefill kernel's cast is one launch more, and an MLP that takes 92 us here takes 95 ...
// 98 there).  No allowance beyond: near the line both models are 2 ... 10 % high, this one more, and 760 calls of 513 ... 2048 rows that a
// factor of 0.95 sends to the prefill kernel take 0.955 (float16) and 0.887 (bfloat16) of its time here (weights out of HBM); with 1.04 as
// many calls would lose as gain with float16 x.  Against the lines of two sets of x and three column tiles: 7978 calls within 15 % of the
// line, 74 with float16 and 78 with bfloat16 x 5 % and more longer (0.95 beyond 512 rows: 132 and 270).
bool batch_ahead(int64_t M, int64_t N, int64_t K, int bits, int group, float us) {
    if (M <= 64) return true;
    const float half_cast = 1.6f + 0.25e-6f * (float)M * (float)K, prefill = bw_qgemm_expected_us(M, N, K, bits, group) + half_cast;
    return 1.035f * us < (M <= 128 ? 1.06f : 1.f) * prefill;
}

BatchCost batch_cost(int64_t M, int64_t N, int64_t K, int bits, int group, bool may_split) {
    static thread_local BwPlanCache<BatchCost> cache = {};   // the search takes 1 ... 3 us of a call's host time, the prefill kernel's model as much again; a look here 10 ns
    return cache.get(M, N, K, (bits * 2 + may_split) * 256 + group, [&] {
        BatchCost found = batch_search(M, N, K, bits, group, may_split);
        found.ahead = batch_ahead(M, N, K, bits, group, found.us);
        return found;
    });
}

BatchPlan batch_plan(int64_t M, int64_t N, int64_t K, int bits, int group, bool may_split) { return batch_cost(M, N, K, bits, group, may_split).plan; }

inline size_t batch_ws_bytes(int64_t M, int64_t N, const BatchPlan& p) { return p.splits > 1 ? (size_t)p.splits * M * ((N + 3) & ~(int64_t)3) * 4 : 0; }

// ---- which kernel ----
enum Route { kDecode, kBatch, kPrefill };

// Up to 16 rows the decode kernels keep the call except where they stage x several times over: rows longer than one round of theirs
// (K > 4096), or more column tiles than their resident workgroups hold; and except on narrow layers with long rows, where this kernel cuts
// K and they have a few workgroups that walk all of it.  From 49000 timings (5 ... 16 rows, nine formats, K 512 ... 14336, N 512 ...
// 22016; this kernel's time over theirs at 9 ... 16 rows, and at 5 ... 8): K > 4096 with tiles > CUs 0.40 ... 0.89 (0.55 ... 0.98);
// tiles > 3 CUs at 8 bits, groups of 32 or an odd number of them 0.73 ... 0.97, else 0.94 ... 1.03 at K <= 2048 (g64: 3072) and 1.0 ... 1.06 up
// to K = 4096; tiles <= CUs / 2 at K > 11008 0.51 ... 0.83 (0.72 ... 1.04), at K <= 4096 1.0 ... 1.2; between CUs / 2 and CUs, where
// every CU has one decode workgroup, 0.85 ... 1.1 at K > 8192 and 1.0 ... 1.5 below, of that up to 3/4 CUs at 2 bits 0.72 ... 1.06 (W4 g64 at K
// > 11008 0.84 ... 1.05), beyond 0.95 ... 1.07 (1.02 ... 1.15) until the rows are long: W2 g64 12800 0.94 ... 1.0, 14336 0.80 ... 0.87, W4 g64
// 14336 0.83 ... 1.01; at 8 bits CUs ... 2 CUs tiles 0.67 ... 0.97 for K > 3072, 5 ... 8 rows 0.9 ... 1.1.  Layers of 8 bits in groups of
// 64 with up to 3 CUs tiles keep the line they had, as their decode kernels scale a group's sum in float32 and this kernel rounds every
// weight; beyond 3 CUs, where all of their calls of 5 rows and more were this kernel's, the wide line gave some back.
// The timings above are graphs.  In eager code the cut costs the host an allocation and a second launch, 8.1 us a call against 6 ... 7, so a
// narrow layer's line lies where the decode kernels take that long (this kernel's time over theirs in a loop of eager calls, and in a
// graph, tiles <= CUs / 2): W2 9 ... 16 rows K = 8192 1.16 ... 1.28 (0.85 ... 0.99), 9216 0.90 ... 0.98 (0.69 ... 0.82); W4 g128 9216 1.05 ...
// 1.17 (0.83 ... 0.98), 11264 0.85 ... 1.04 (0.77 ... 0.90); W8 g32 6400 0.86 ... 1.12 (0.82 ... 0.94), 7168 0.81 ... 1.06 (0.79 ... 0.90); 5 ... 8
// rows W2 g64 12288 1.12 ... 1.20 (0.84 ... 1.04), 12800 0.95 ... 1.02 (0.76 ... 0.95); W4 g64 11264 0.99 ... 1.17 (0.88 ... 1.0), 12288 0.88 ... 1.05
// (0.75 ... 0.89); W4 g32 9216 0.97 ... 1.10 (0.78 ... 0.93), 10240 0.90 ... 1.06 (0.79 ... 0.89).
inline bool batch_takes_decode_rows(int64_t M, int64_t N, int64_t K, int bits, int group) {
    const int64_t tiles = (N + 15) / 16, cus = bw_device_cus();
    const bool many = M > 8, narrow = tiles <= cus / 2;
    if (M < 5) return false;
    if (bits == 8) {
        if (tiles > 3 * cus) return many ? K > 1024 : K > 3072 && (tiles <= 4 * cus || group == 32);
        if (group == 64) return many && K >= 8192;
        if (tiles > 2 * cus) return many && K > 6144;
        if (tiles > cus) return many && K > 3072;
        if (narrow) return K > (many ? group == 32 ? 6400 : 8191 : group == 32 ? 8192 : 11008);
        return many && K > (group == 32 ? 8192 : 11008);
    }
    if (K > 4096 ? tiles > cus : K >= 3072 && tiles > 4 * cus) return true;
    if (many && tiles > 3 * cus && (group == 32 || K / group % 2 || K <= (group == 64 ? 3072 : 2048))) return true;
    if (many && group == 32) return K > 4096 || (tiles > cus && tiles <= 2 * cus);
    if (K <= 4096) return false;
    if (narrow && many) return K > (bits == 2 ? 8192 : group == 128 ? 10240 : 6144);
    if (narrow) return group != 128 && K > (bits == 2 ? 12288 : group == 32 ? 9216 : 11264);
    const bool full = 4 * tiles > 3 * cus && K / group % 2 == 0;
    return many && (bits == 2 ? K > (!full ? 8192 : group == 64 ? 12288 : 13312) : group == 64 && K > (full ? 13312 : 11008));
}

Route route(int64_t M, int64_t N, int64_t K, int bits, int group) {
    if (M <= 16) return batch_takes_decode_rows(M, N, K, bits, group) ? kBatch : kDecode;
    return M <= 2048 && batch_cost(M, N, K, bits, group, true).ahead ? kBatch : kPrefill;
}

// What the batch kernel asks of a call beyond bw_fast_shape: whole float16 values of scales, offsets of x in 31 bits.
inline bool batch_takes(const void* x, int64_t M, int64_t N, int64_t K, int64_t ldx, const void* qweight, const void* scale16, const void* zp16, int bits, int group) {
    return bw_fast_shape(M, N, K, ldx, bits, group) && bw_aligned(x, 16) && (ldx * 2) % 16 == 0 && bw_aligned(qweight, 16) && bw_aligned(scale16, 2) &&
           bw_aligned(zp16, 2) && M * ldx * 2 < (int64_t)kBatchMaxBytes;
}

int launch_batch(const void* x, int act_dtype, int64_t M, int64_t K, int64_t ldx, const int32_t* qweight, const void* scale16, const void* zp16,
                 const void* bias, int64_t N, int bits, int group, void* y, int64_t ldy, void* workspace, const BatchPlan& plan, hipStream_t st) {
    BatchArgs a;
    a.x = x; a.qweight = qweight; a.scale = scale16; a.zp = zp16; a.bias = (const _Float16*)bias; a.y = (_Float16*)y;
    a.ws = (float*)workspace;
    a.M = (int)M; a.N = (int)N; a.K = (int)K; a.ldx = (int)ldx; a.ldy = (int)ldy; a.npad = (int)((N + 3) & ~(int64_t)3);
    a.groups = (int)(K / group);
    a.row_bytes = (int)(K * bits / 8);
    a.nchunks = (int)((K + 127) / 128);
    a.x_bytes = (uint32_t)(((M - 1) * ldx + K) * 2);
    a.w_bytes = (uint32_t)(N * a.row_bytes);
    a.meta_bytes = (uint32_t)(N * a.groups * 2);
    a.splits = plan.splits;
    a.chunks_per_split = (a.nchunks + plan.splits - 1) / plan.splits;
    a.x_bf16 = act_dtype == BW_BF16;
    a.sums = batch_sums(M, N, K, bits, group);
    const int r = bits == 4   ? bw_launch_qbatch_w4(group, plan.mt, plan.ntw, a, st)
                  : bits == 8 ? bw_launch_qbatch_w8(group, plan.mt, plan.ntw, a, st)
                              : bw_launch_qbatch_w2(group, plan.mt, plan.ntw, a, st);
    if (r != BW_OK || a.splits == 1) return r;
    const int64_t items = M * (a.npad / 4);
    hipLaunchKernelGGL(qbatch_reduce_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, st, a.ws, a.bias, a.y, a.M, a.N, a.npad, a.ldy, a.splits);
    return hipGetLastError() == hipSuccess ? BW_OK : BW_ELAUNCH;
}

inline size_t cast_bytes(int64_t M, int64_t K) { return ((size_t)M * K * 2 + 255) & ~(size_t)255; }

}  // namespace

// Rows up to which bw_qlinear takes bfloat16 x and, without a workspace, stays off the prefill kernel.  (Set when more than
// 16 rows ran as several decode launches; kept as part of the interface.)
extern "C" int bw_qlinear_decode_rows(int64_t N, int64_t K, int bits) {
    if (N < 1 || K < 1 || !bw_bits_ok(bits)) return 0;
    const int64_t bytes = N * (K * bits / 8);
    return bytes < ((int64_t)10 << 20) ? 48 : bytes < ((int64_t)40 << 20) ? 32 : 16;
}

extern "C" size_t bw_qlinear_workspace_bytes(int64_t M, int64_t N, int64_t K, int bits, int group, int act_dtype) {
    if (!bw_shape_ok(N, K, bits, group) || M < 1 || M >= ((int64_t)1 << 31)) return 0;
    const bool fast = bw_fast_shape(M, N, K, K, bits, group);
    const Route r = fast ? route(M, N, K, bits, group) : M <= 16 ? kDecode : kPrefill;
    size_t split = r == kPrefill && M > 16 ? bw_qgemm_workspace_bytes(M, N, K, bits, group) : 0;
    if (r == kBatch) split = batch_ws_bytes(M, N, batch_plan(M, N, K, bits, group, true));
    const bool cast = act_dtype == BW_BF16 && (r == kPrefill || !fast);
    return split + (cast ? cast_bytes(M, K) : 0);
}

extern "C" int bw_qlinear_ws(const void* x, int act_dtype, int64_t M, int64_t K, int64_t ldx, const int32_t* qweight, const void* scale16,
                             const void* zp16, const void* bias, int64_t N, int bits, int group, void* y, int64_t ldy, void* workspace,
                             size_t workspace_bytes, void* stream) {
    if (!x || !qweight || !scale16 || !zp16 || !y) return BW_EINVAL;
    if (!bw_shape_ok(N, K, bits, group) || M < 1 || M >= ((int64_t)1 << 31) || ldx < K || ldy < N) return BW_EINVAL;
    if (act_dtype != BW_F16 && act_dtype != BW_BF16) return BW_EUNSUPPORTED;
    if (workspace && !bw_aligned(workspace, 16)) return BW_EALIGN;
    if (!workspace) workspace_bytes = 0;
    bw_note_kernel("");
    const bool fast = bw_fast_shape(M, N, K, ldx, bits, group);
    Route r = fast ? route(M, N, K, bits, group) : M <= 16 ? kDecode : kPrefill;
    // Without room for the prefill kernel's cast of a bfloat16 x this kernel takes the call, which reads x as it is (and cuts K only if
    // there is room for that).
    if (fast && r == kPrefill && M <= 2048 && act_dtype == BW_BF16 && workspace_bytes < cast_bytes(M, K)) r = kBatch;
    const bool cut = r != kBatch || batch_ws_bytes(M, N, batch_plan(M, N, K, bits, group, true)) <= workspace_bytes;   // room for the plan's cut of K
    // Up to 16 rows a narrow layer comes here for that cut: without room for it the decode kernels are ahead (9 rows, us: W4 g128
    // 14336 -> 512 uncut 15.1, theirs 10.6; W8 g32 14336 -> 4096 23.6 and 19.9; 83 calls with tiles <= CUs 0.6 ... 1.01).
    if (!cut && M <= 16 && (N + 15) / 16 <= bw_device_cus()) r = kDecode;
    if (r == kBatch && batch_takes(x, M, N, K, ldx, qweight, scale16, zp16, bits, group)) {
        const BatchPlan plan = batch_plan(M, N, K, bits, group, cut);
        return launch_batch(x, act_dtype, M, K, ldx, qweight, scale16, zp16, bias, N, bits, group, y, ldy, workspace, plan, (hipStream_t)stream);
    }
    if (M <= 16) {
        const int st = bw_qgemv(x, act_dtype, M, K, ldx, qweight, scale16, zp16, bias, N, bits, group, y, ldy, stream);
        if (st != BW_EUNSUPPORTED || act_dtype != BW_BF16) return st;      // bfloat16 on a shape that only the generic kernel takes
    }
    if (act_dtype == BW_BF16) {                                            // the prefill kernel wants float16 in memory
        const size_t need = cast_bytes(M, K);
        if (workspace_bytes < need) return BW_EWORKSPACE;
        const int st = bw_cast_bf16_f16(x, M, K, ldx, workspace, K, stream);
        if (st != BW_OK) return st;
        x = workspace;
        ldx = K;
        workspace_bytes -= need;
        workspace = workspace_bytes ? (char*)workspace + need : nullptr;
    }
    // A workspace too small for the plan that bw_qgemm_workspace_bytes asks for may still serve the cut of the 256-column tiles: 1455 calls of 65 ... 2048 rows with
    // what that needs take 0.911 of the time of always cutting (11 over 2 % longer, at most 1.08) and 0.944 of never cutting (2, at most 1.03).
    const size_t need = bw_qgemm_workspace_bytes(M, N, K, bits, group);
    const bool split = need && (workspace_bytes >= need || bw_qgemm_small_workspace_serves(M, N, K, bits, group, workspace_bytes));
    return bw_qgemm_ws(x, BW_F16, M, K, ldx, qweight, scale16, zp16, bias, N, bits, group, y, ldy, split ? workspace : nullptr, split ? workspace_bytes : 0, stream);
}

extern "C" int bw_qlinear(const void* x, int act_dtype, int64_t M, int64_t K, int64_t ldx, const int32_t* qweight,
                          const void* scale16, const void* zp16, const void* bias, int64_t N, int bits, int group,
                          void* y, int64_t ldy, void* stream) {
    bw_note_kernel("");
    if (M >= 1 && M <= bw_qlinear_decode_rows(N, K, bits) && (act_dtype == BW_F16 || act_dtype == BW_BF16)) {
        // the batch kernel where it is what bw_qlinear_ws runs too and K needs no cut for want of workgroups
        if (x && qweight && scale16 && zp16 && y && bw_shape_ok(N, K, bits, group) && ldx >= K && ldy >= N &&
            batch_takes(x, M, N, K, ldx, qweight, scale16, zp16, bits, group) && route(M, N, K, bits, group) == kBatch &&
            batch_plan(M, N, K, bits, group, true).splits == 1)
            return launch_batch(x, act_dtype, M, K, ldx, qweight, scale16, zp16, bias, N, bits, group, y, ldy, nullptr,
                                batch_plan(M, N, K, bits, group, true), (hipStream_t)stream);
        for (int64_t m0 = 0; m0 < M; m0 += 16) {
            const int st = bw_qgemv((const _Float16*)x + m0 * ldx, act_dtype, M - m0 < 16 ? M - m0 : 16, K, ldx, qweight, scale16,
                                    zp16, bias, N, bits, group, (_Float16*)y + m0 * ldy, ldy, stream);
            if (st != BW_OK) return st;
        }
        return BW_OK;
    }
    return bw_qgemm(x, act_dtype, M, K, ldx, qweight, scale16, zp16, bias, N, bits, group, y, ldy, stream);
}
