// Prefill path: y[M][N] = x[M][K] @ W16[N][K]^T (+ bias) for any M, built for
// M >= 128 where the matrix cores are the bound.
//
// A workgroup of 4 waves owns a 128 (M) x 256 (N) output tile; each wave owns
// 128 x 64 of it (8 x 4 MFMA 16x16 tiles, 128 accumulator registers).  Per K
// step of one chunk (64 packed bytes per weight row):
//   * weights go global -> registers with one 128-bit load per lane per 16
//     rows, already in MFMA operand layout, and are unpacked in registers
//     to the float16 values the reference's dequantize kernel would store
//     (bitween/modules.py:55-58).  No wave unpacks a weight another wave of
//     the workgroup also unpacks; each weight is unpacked M/128 times overall.
//   * activations go global -> LDS once per workgroup, double buffered, and
//     every fragment read from LDS feeds 4 MFMAs.
// Two schedules of that loop.  Natural order (K a multiple of 128: step16 below):
// the activations go memory -> LDS without passing through registers (buffer
// loads with LDS destination), the weights are unpacked to natural k order, and
// the side work of an MFMA step is dealt out one instruction per MFMA.  Register
// staged (any other K: step8): the activations pass through registers and are
// permuted into the k order a cheaper unpack emits.
// Grids that fill the device run the natural-order schedule with 256 x 256
// tiles (a wave owns 256 x 64: all 256 accumulation registers): every weight
// is unpacked once for twice the rows.  Which tile height a call gets is
// gemm_tile(); a short last round of tiles is cut along K (gemm_plan()),
// and the tiles are numbered so that the workgroups an XCD runs together share
// operand tiles in its L2 (GemmArgs::panel).  Both heights also come 192 columns
// wide (a wave owns 48): finer tiles for the grids that 256 columns would fill badly.
// Also holds the shape-generic fallback used when the fast layouts do not
// apply (odd K or group size): correct for everything the reference accepts.
#include "bw_plan_cache.h"
#include "bw_qgemm_kernel.h"

#include <atomic>

bool bw_fast_shape(int64_t M, int64_t N, int64_t K, int64_t ldx, int bits, int group);

namespace {

// The natural-order schedule (activations memory -> LDS by buffer loads with LDS destination, step16) takes whole K
// steps of 128 values and offsets of rows past M that still fit 32 bits; other shapes run the register-staged kernel.
inline bool gemm_nat(int64_t M, int64_t K, int64_t ldx) {
#ifdef BW_TUNE   // measurement builds only (-DBW_TUNE, never the library build.py makes): kernel choices from the environment, for A/B runs
    if (const char* e = getenv("BW_GEMM_NAT")) if (atoi(e) == 0) return false;
#endif
    return K % 128 == 0 && (M + 256) * ldx * 2 < ((int64_t)1 << 32);
}

struct GemmTile { int rows, cols; };

constexpr size_t kScratchBytes = (size_t)32 << 20;       // bw_qgemm_static's device array: 256 partial tiles of 128 x 256 floats, one full round

// Tile of 256 columns for this call.  Calls of at most 64 rows take 64-row tiles: half the MFMAs and half the activation
// traffic of a 128-row tile that would be at least half padding (17 ... 64 rows on the five Llama MLP / attention shapes at
// 4 bits: 0.84-0.95 of the 128-row time, same bits).  A 256-row tile unpacks every weight once for twice the rows and keeps the matrix pipe
// busier: a full round of 256-row tiles takes about 1.65 x the time of a full round of 128-row tiles for twice the
// work.  Which grid finishes first then depends on how each fills its rounds (one workgroup per CU): whole rounds,
// plus a last round that costs a full one when more than half full and about three quarters of one when its tiles are
// split along K (a workspace is on offer).  That model reproduces a sweep of both heights over K, N in {4096, 11008,
// 14336} and M = 512 ... 2048 (4 bits; e.g. 4096 -> 14336 at 2048 rows: 3.75 against 3.3 rounds, measured 207 against
// 184 us; 4096 x 4096 at 2048 rows: 1.0 against 1.24, measured 60 against 75 us); the 256-row grid is taken when it is
// ahead by 5 % or more.  Only with the natural-order schedule, and only while the split-K blocks of its plan fit the
// workspace on offer.
inline GemmTile gemm_tile_wide(int64_t M, int64_t N, int64_t K, int64_t ldx, int bits, bool have_workspace, size_t workspace_bytes) {
    constexpr int wide = tile_cols(4);
    if (!gemm_nat(M, K, ldx)) return {128, wide};
    const int nchunks = gemm_chunks(K, bits, true);
#ifdef BW_TUNE
    if (const char* e = getenv("BW_GEMM_BM")) return {atoi(e) == 256 ? 256 : atoi(e) == 64 ? 64 : 128, wide};
#endif
    // (up to 128 rows as two 64-row tiles where N is at most 16 tiles wide: 4096 x 4096, 11008 -> 4096 and 14336 -> 4096 at
    // 80 ... 128 rows 0.88-0.95 of the 128-row time - half the partial-tile traffic of the K split -, but 1.06-1.11 at
    // N = 11008 and 14336, where every weight would be unpacked twice for nothing)
    if (M <= 64) return {64, wide};
    auto fits = [&](int rows, int cols) { return !have_workspace || gemm_plan(M, N, nchunks, true, rows, cols).ws_bytes <= workspace_bytes; };
    if (M <= 128 && (N + wide - 1) / wide <= 16 && fits(64, wide)) return {64, wide};
    const int64_t cus = bw_device_cus();
    auto rounds = [&](int64_t tiles) {
        const int64_t full = tiles / cus, rest = tiles % cus;
        const bool split = have_workspace && nchunks >= 8 && rest <= cus / 2;
        return (double)full + (rest == 0 ? 0.0 : split ? 0.75 : 1.0);
    };
    const int64_t tiles_n = (N + wide - 1) / wide;
    const double t128 = rounds(tiles_n * ((M + 127) / 128)), t256 = 1.65 * rounds(tiles_n * ((M + 255) / 256));
    return {t256 > 0.95 * t128 || !fits(256, wide) ? 128 : 256, wide};
}

// What a call takes, us, with 128- or 256-row tiles of the natural-order schedule (float16 x, weights out of HBM): a base; per 128 values of K
// of every round of tiles `step` on an empty chip and `fill` more on a full one; where the tiles of a short round are cut along K, `cut`, `part`
// per million partial sums, and the same two for their slices; more per step at 8 bits and in groups of 32; rows of y that start off an 8-byte
// boundary cost a round of tiles `odd`, their stores going out as 2-byte pieces.  Fitted to 11796 calls of 129 ... 2048 rows, each timed with
// the four tiles (all formats, K 512 ... 14336, N 512 ... 22016; rms error 6 ... 7 % each).
inline float gemm_us(int64_t M, int64_t N, int64_t K, int bits, int group, GemmTile tile, bool have_workspace) {
    struct Cost { float base, step, fill, cut, part, cut_step, cut_fill, b8, g32, odd; };
    static constexpr Cost k128 = {8.1f, 0.864f, 0.924f, 4.1f, 0.85f, 1.11f, 0.41f, 0.16f, 0.09f, 7.2f},
                          k256 = {12.1f, 1.468f, 1.507f, 7.0f, 0.42f, 1.37f, 1.32f, 0.31f, 0.07f, 13.6f},
                          n128 = {7.1f, 0.745f, 0.564f, 2.8f, 1.32f, 0.97f, 0.12f, 0.17f, 0.08f, 5.1f},
                          n256 = {10.9f, 1.077f, 1.266f, 4.3f, 0.57f, 1.21f, 0.83f, 0.26f, 0.06f, 8.9f};
    const Cost& c = tile.cols == tile_cols(4) ? tile.rows == 128 ? k128 : k256 : tile.rows == 128 ? n128 : n256;
    const int nchunks = gemm_chunks(K, bits, true), cus = bw_device_cus();
    const GemmPlan p = gemm_plan(M, N, nchunks, have_workspace, tile.rows, tile.cols);
    const int rest = p.tiles - p.full_tiles, rounds = (p.full_tiles + cus - 1) / cus;
    const float extra = (bits == 8 ? c.b8 : 0.f) + (group == 32 ? c.g32 : 0.f);
    float us = c.base + nchunks * ((c.step + extra) * rounds + c.fill * p.full_tiles / cus) + (N % 4 ? c.odd * rounds : 0.f);
    if (rest)
        us += c.cut + c.part * 1e-6f * rest * p.splits * (tile.rows * tile.cols) + p.chunks_per_split * (c.cut_step + extra + c.cut_fill * rest * p.splits / cus);
    return us;
}

// rounds of a grid of tiles t, `per_cu` workgroups at once on every CU
inline int64_t tile_rounds(int64_t M, int64_t N, GemmTile t, int per_cu) {
    const int64_t tiles = ((M + t.rows - 1) / t.rows) * ((N + t.cols - 1) / t.cols), places = (int64_t)per_cu * bw_device_cus();
    return (tiles + places - 1) / places;
}

// Tile for this call: 192 columns where the model above is ahead of the 256-column tile's by 5 % (10 % of a 256-row tile on less than eight
// K steps, which it has too slow).  Finer tiles leave fewer CUs idle in a short round (4096 -> 11008 at 509 rows: 172 tiles of 128 x 256 on 256
// CUs, 232 of 128 x 192; W4 g128 52.2 -> 46.7 us), their base is smaller, and a K step takes 0.86 of the time where CUs are idle and 0.73 on
// a full chip, for 0.75 of the work.  8489 of the 11796 calls take 192 columns; all together they take 0.917 of the time, 16 of them over 5 %
// more (K below 1024), and the best of the four tiles each time would save another 1 %.  Beyond the rows that the model is fitted to, half of the calls of
// 2049 ... 8192 rows and a third of those up to 32768 take 192 columns: 13553 of them timed against the 256-column rule, 0.866 on average (0.872 up to 4096 rows,
// 0.863 to 8192, 0.864 beyond), 24 over 5 % more, at most 1.17 (26142 rows of 11520 -> 672).
inline GemmTile gemm_tile(int64_t M, int64_t N, int64_t K, int64_t ldx, int bits, int group, bool have_workspace, size_t workspace_bytes) {
    const GemmTile wide = gemm_tile_wide(M, N, K, ldx, bits, have_workspace, workspace_bytes);
    if (wide.rows == 64 || !gemm_nat(M, K, ldx)) return wide;
    const int nchunks = gemm_chunks(K, bits, true);
    if (have_workspace && gemm_plan(M, N, nchunks, true, wide.rows, wide.cols).ws_bytes > workspace_bytes) return wide;   // refused, whatever a narrow plan needs
#ifdef BW_TUNE
    if (const char* e = getenv("BW_GEMM_BN")) return {wide.rows, atoi(e) == tile_cols(3) && wide.rows != 64 ? tile_cols(3) : tile_cols(4)};
    if (getenv("BW_GEMM_BM")) return wide;
#endif
    static thread_local BwPlanCache<GemmTile> cache = {};    // the four models take 0.2 us
    const GemmTile best = cache.get(M, N, K, (bits * 4 + 2 * have_workspace + (wide.rows == 256)) * 256 + group, [&] {
        GemmTile b = wide;
        float us = gemm_us(M, N, K, bits, group, wide, have_workspace) * (wide.rows == 256 && nchunks < 8 ? 0.9f : 0.95f);
        for (const int rows : {128, 256}) {
            const GemmTile narrow = {rows, tile_cols(3)};
            // (no plan that bw_qgemm_static could not run: its results are bw_qgemm_ws's bit for bit)
            if (have_workspace && gemm_plan(M, N, nchunks, true, rows, narrow.cols).ws_bytes > kScratchBytes) continue;
            // Three and four K steps: the model has one round of 256 x 256 tiles too slow beside 128 x 192 tiles that need a second one of two workgroups a CU (10257
            // calls of 129 ... 2048 rows with K = 128 ... 640, each with the four tiles: at K = 384 42 of 46 such calls took longer, 1.06 on average, up to 1.14; rows of y
            // off 16 bytes make 256 columns the slower ones all the same).  One and two steps are left: 46 of 4355 calls over 2 % longer than with 256 columns, up
            // to 1.17, 0.871 of the time on average; this line would help 17 of them and cost 24 others as much.
            if ((nchunks == 3 || nchunks == 4) && rows == 128 && wide.rows == 256 && N % 8 == 0 && tile_rounds(M, N, wide, 1) == 1 && tile_rounds(M, N, narrow, 2) > 1) continue;
            const float t = gemm_us(M, N, K, bits, group, narrow, have_workspace);
            if (t < us) { b = narrow; us = t; }
        }
        return b;
    });
    if (best.cols != wide.cols && have_workspace && gemm_plan(M, N, nchunks, true, best.rows, best.cols).ws_bytes > workspace_bytes) return wide;
    return best;
}

// Shape-generic fallback: one thread per output element, any group size and
// any K the reference accepts.  Same arithmetic: W16 = fp16(s * (q - z)) from
// the float32 product, float32 accumulation, one rounding of the result.
__global__ void qgemm_generic_kernel(const _Float16* __restrict__ x, int M, int K, int64_t ldx,
                                     const uint32_t* __restrict__ qweight, const _Float16* __restrict__ scale,
                                     const _Float16* __restrict__ zp, const _Float16* __restrict__ bias, int N, int bits,
                                     int group, _Float16* __restrict__ y, int64_t ldy) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)M * N) return;
    const int n = (int)(idx % N), m = (int)(idx / N);
    const int vpi = 32 / bits, words = K / vpi, groups = K / group;
    const uint32_t mask = (1u << bits) - 1;
    float acc = 0.f;
    for (int wi = 0; wi < words; wi++) {
        const uint32_t w = qweight[(int64_t)n * words + wi];
        for (int i = 0; i < vpi; i++) {
            const int k = wi * vpi + i;
            const float q = (float)((w >> (i * bits)) & mask);
            const float s = (float)scale[(int64_t)n * groups + k / group], z = (float)zp[(int64_t)n * groups + k / group];
            const _Float16 w16 = (_Float16)(s * (q - z));
            acc = __builtin_fmaf((float)x[(int64_t)m * ldx + k], (float)w16, acc);
        }
    }
    if (bias) acc += (float)bias[n];
    y[(int64_t)m * ldy + n] = (_Float16)acc;
}

// bfloat16 -> float16 of a row-major matrix, 8 values (16 bytes) per unit; a thread converts the units
// idx, idx + T, idx + 2T, idx + 3T (T = all threads) with every load issued before the first store.
__global__ __launch_bounds__(256) void cast_bf16_f16_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ y,
                                                            int64_t units, int upr, int64_t ldx, int64_t ldy) {
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    u4 v[4];
    int64_t dst[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t u = t0 + i * stride;
        dst[i] = -1;
        if (u < units) {
            const int64_t r = u / upr, c = (u - r * upr) * 8;
            v[i] = *reinterpret_cast<const u4*>(x + r * ldx + c);
            dst[i] = r * ldy + c;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (dst[i] < 0) continue;
        u4 o;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float lo = __builtin_bit_cast(float, v[i][j] << 16), hi = __builtin_bit_cast(float, v[i][j] & 0xFFFF0000u);
            o[j] = as_u32(h2{(_Float16)lo, (_Float16)hi});
        }
        *reinterpret_cast<u4*>(y + dst[i]) = o;
    }
}

}  // namespace

// What a call of 65 ... 2048 rows takes, us, with the 256-column tiles it would run (gemm_tile_wide, a workspace on offer), float16 x.  Fitted to 1773
// timings of 65 ... 2048 rows where this kernel and the batch kernel are within a factor of two (all formats, K and N 512 ...
// 22016; rms error 6 %; 14 % with 128-row tiles assumed throughout and no look at format and N): a base; per 128 values of K of every
// round of tiles `step` on an empty chip and `fill` more on a full one; the same for the slices of a short round that is cut along K,
// 7.3 and 0.38 us per million partial sums for the cut; more per step at 8 bits, groups of 32 and K % 128 != 0; rows of y that start
// off an 8-byte boundary cost a round of uncut tiles `odd`, their stores going out as 2-byte pieces.  (192-column tiles have not moved the line between the
// kernels: by gemm_us of the chosen tile 955 of 22338 calls more would come here and take 0.906 of the batch kernel's time, 28 of them over 8 % longer.)
float bw_qgemm_expected_us(int64_t M, int64_t N, int64_t K, int bits, int group) {
    struct Cost { float base, step, fill, cut_step, cut_fill, b8, odd; };
    static constexpr Cost k64 = {5.8f, 0.61f, 0.68f, 0.66f, 0.38f, 0.39f, 0.f}, k128 = {7.4f, 0.96f, 0.68f, 0.77f, 0.87f, 0.27f, 7.4f},
                          k256 = {12.1f, 1.34f, 1.41f, 0.77f, 0.87f, 0.34f, 16.6f};
    const bool nat = gemm_nat(M, K, K);
    const int rows = gemm_tile_wide(M, N, K, K, bits, true, ~(size_t)0).rows, nchunks = gemm_chunks(K, bits, nat), cus = bw_device_cus();
    const Cost& c = rows == 64 ? k64 : rows == 128 ? k128 : k256;
    const GemmPlan p = gemm_plan(M, N, nchunks, true, rows);
    const float steps = bits == 2 && !nat ? 2.f : 1.f;       // of 128 values in a chunk
    const int rest = p.tiles - p.full_tiles, rounds = (p.full_tiles + cus - 1) / cus;
    const float extra = (bits == 8 ? c.b8 : bits == 2 ? -0.04f : 0.f) + (nat ? 0.f : 0.37f) + (group == 32 ? bits == 8 ? 0.18f : 0.12f : 0.f);
    float us = c.base + steps * nchunks * ((c.step + extra) * rounds + c.fill * p.full_tiles / cus) + (N % 4 ? c.odd * rounds : 0.f);
    if (rest)
        us += 7.3f + 0.38e-6f * rest * p.splits * (rows * tile_cols(4)) + steps * p.chunks_per_split * (c.cut_step + extra + c.cut_fill * rest * p.splits / cus);
    return us;
}

extern "C" int bw_cast_bf16_f16(const void* x, int64_t rows, int64_t cols, int64_t ldx, void* y, int64_t ldy, void* stream) {
    if (!x || !y || rows < 1 || cols < 1 || ldx < cols || ldy < cols) return BW_EINVAL;
    if (cols % 8 || ldx % 8 || ldy % 8 || cols / 8 >= ((int64_t)1 << 31)) return BW_EUNSUPPORTED;
    if (!bw_aligned(x, 16) || !bw_aligned(y, 16)) return BW_EALIGN;
    const int64_t units = rows * (cols / 8), blocks = (units + 4 * 256 - 1) / (4 * 256);
    if (blocks >= ((int64_t)1 << 31)) return BW_EUNSUPPORTED;
    hipLaunchKernelGGL(cast_bf16_f16_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (const uint16_t*)x,
                       (uint16_t*)y, units, (int)(cols / 8), ldx, ldy);
    return hipGetLastError() == hipSuccess ? BW_OK : BW_ELAUNCH;
}

int bw_qgemm_generic(const void* x, int act_dtype, int64_t M, int64_t K, int64_t ldx, const int32_t* qweight,
                     const void* scale16, const void* zp16, const void* bias, int64_t N, int bits, int group, void* y,
                     int64_t ldy, void* stream) {
    if (act_dtype != BW_F16) return BW_EUNSUPPORTED;
    const int64_t total = M * N;
    hipLaunchKernelGGL(qgemm_generic_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const _Float16*)x, (int)M, (int)K, ldx, (const uint32_t*)qweight, (const _Float16*)scale16,
                       (const _Float16*)zp16, (const _Float16*)bias, (int)N, bits, group, (_Float16*)y, ldy);
    return hipGetLastError() == hipSuccess ? BW_OK : BW_ELAUNCH;
}

#ifdef BW_TUNE
static unsigned long long* g_tune_clk = nullptr;
extern "C" void bw_tune_clock_buffer(void* p) { g_tune_clk = (unsigned long long*)p; }   // 4096 bytes of device memory, or null
#endif

// Workspace of the plans with 256-column tiles: the call's own ldx and workspace decide which of them runs.
static size_t gemm_wide_ws_bytes(int64_t M, int64_t N, int64_t K, int bits) {
    size_t need = gemm_plan(M, N, gemm_chunks(K, bits, false), true, 128).ws_bytes;
    if (gemm_nat(M, K, K)) {
        const size_t nat128 = gemm_plan(M, N, gemm_chunks(K, bits, true), true, 128).ws_bytes;
        if (nat128 > need) need = nat128;
        const int rows = gemm_tile_wide(M, N, K, K, bits, true, ~(size_t)0).rows;
        if (rows != 128) {
            const size_t other = gemm_plan(M, N, gemm_chunks(K, bits, true), true, rows).ws_bytes;
            if (other > need) need = other;
        }
    }
    return need;
}

extern "C" size_t bw_qgemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int bits, int group) {
    if (!bw_shape_ok(N, K, bits, group) || M < 1 || M >= ((int64_t)1 << 31) || !bw_fast_shape(M, N, K, K, bits, group)) return 0;
    const size_t need = gemm_wide_ws_bytes(M, N, K, bits);
    if (!gemm_nat(M, K, K)) return need;
    const GemmTile tile = gemm_tile(M, N, K, K, bits, group, true, ~(size_t)0);
    const size_t chosen = gemm_plan(M, N, gemm_chunks(K, bits, true), true, tile.rows, tile.cols).ws_bytes;
    return chosen > need ? chosen : need;
}

// Whether a workspace smaller than bw_qgemm_workspace_bytes asks for is worth passing on: it has room for the plan of the 256-column tiles, which
// bw_qgemm_ws then runs, and that is expected to be done before the best of the uncut plans is.
bool bw_qgemm_small_workspace_serves(int64_t M, int64_t N, int64_t K, int bits, int group, size_t workspace_bytes) {
    if (!bw_shape_ok(N, K, bits, group) || M < 1 || M >= ((int64_t)1 << 31) || !bw_fast_shape(M, N, K, K, bits, group)) return false;
    const size_t least = gemm_wide_ws_bytes(M, N, K, bits);
    if (!least || workspace_bytes < least) return false;
    if (!gemm_nat(M, K, K)) return true;
    const GemmTile cut = gemm_tile_wide(M, N, K, K, bits, true, workspace_bytes), uncut = gemm_tile(M, N, K, K, bits, group, false, 0);
    if (cut.rows == 64 || uncut.rows == 64) return true;
    return gemm_us(M, N, K, bits, group, cut, true) <= gemm_us(M, N, K, bits, group, uncut, false);
}

extern "C" int bw_qgemm_tile_rows(int64_t M, int64_t N, int64_t K, int bits, int group) {
    if (!bw_shape_ok(N, K, bits, group) || M < 1 || M >= ((int64_t)1 << 31) || !bw_fast_shape(M, N, K, K, bits, group)) return 0;
    return gemm_tile(M, N, K, K, bits, group, true, ~(size_t)0).rows;
}

extern "C" int bw_qgemm_tile_cols(int64_t M, int64_t N, int64_t K, int bits, int group) {
    if (!bw_shape_ok(N, K, bits, group) || M < 1 || M >= ((int64_t)1 << 31) || !bw_fast_shape(M, N, K, K, bits, group)) return 0;
    return gemm_tile(M, N, K, K, bits, group, true, ~(size_t)0).cols;
}

extern "C" int bw_qgemm_ws(const void* x, int act_dtype, int64_t M, int64_t K, int64_t ldx, const int32_t* qweight,
                           const void* scale16, const void* zp16, const void* bias, int64_t N, int bits, int group,
                           void* y, int64_t ldy, void* workspace, size_t workspace_bytes, void* stream) {
    if (!x || !qweight || !scale16 || !zp16 || !y) return BW_EINVAL;
    if (!bw_shape_ok(N, K, bits, group) || M < 1 || M >= ((int64_t)1 << 31) || ldx < K || ldy < N) return BW_EINVAL;
    if (act_dtype != BW_F16) return BW_EUNSUPPORTED;
    if (!bw_fast_shape(M, N, K, ldx, bits, group) || !bw_aligned(x, 16) || (ldx * 2) % 16 || !bw_aligned(qweight, 16))
        return bw_qgemm_generic(x, act_dtype, M, K, ldx, qweight, scale16, zp16, bias, N, bits, group, y, ldy, stream);
    if (workspace && !bw_aligned(workspace, 16)) return BW_EALIGN;
    GemmArgs a;
    a.x = x; a.qweight = qweight; a.scale = (const _Float16*)scale16; a.zp = (const _Float16*)zp16;
    a.bias = (const _Float16*)bias; a.y = (_Float16*)y;
    a.M = (int)M; a.N = (int)N; a.K = (int)K; a.ldx = (int)ldx; a.ldy = (int)ldy;
    a.groups = (int)(K / group);
    a.row_bytes = (int)(K * bits / 8);
    const bool nat = gemm_nat(M, K, ldx);
    a.nchunks = gemm_chunks(K, bits, nat);
    a.x_bytes = (uint32_t)(((M - 1) * ldx + K) * 2);
    a.w_bytes = (uint32_t)(N * a.row_bytes);
    a.meta_bytes = (uint32_t)(N * a.groups * 2);
    a.ws = nullptr;
    a.tiles_n = a.full_tiles = 0;
    a.tiles_m = a.panel = 1;
    a.xcd_tiles = 0;
#ifdef BW_TUNE
    a.clk = g_tune_clk;
#endif
    a.splits = 1;
    a.chunks_per_split = a.nchunks;
    hipStream_t st = (hipStream_t)stream;
    const GemmTile tile = gemm_tile(M, N, K, ldx, bits, group, workspace != nullptr, workspace_bytes);
    if (tile.cols != tile_cols(4)) return bw_launch_gemm_cols192(bits, group, tile.rows, a, workspace, workspace_bytes, st);
    if (tile.rows != 128) return bw_launch_gemm_rows(bits, group, tile.rows, a, workspace, workspace_bytes, st);
#define BW_CASE(B, G)                                                                               \
    if (bits == B && group == G)                                                                     \
        return nat ? launch_gemm<B, G, 8, true>(a, workspace, workspace_bytes, st)                   \
                   : launch_gemm<B, G, 8, false>(a, workspace, workspace_bytes, st);
    BW_CASE(4, 128) BW_CASE(4, 64) BW_CASE(4, 32)
    BW_CASE(8, 128) BW_CASE(8, 64) BW_CASE(8, 32)
    BW_CASE(2, 128) BW_CASE(2, 64) BW_CASE(2, 32)
#undef BW_CASE
    return BW_EUNSUPPORTED;
}

// ---- the same without a caller's workspace: the split-K partial tiles go to a device array of the library ----
// For callers that cannot allocate (code under graph capture, serving loops, harnesses that forbid it).  The array
// is one per GPU, shared by every call on that GPU and kept for the life of the process.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
constexpr int kMaxDevices = 64;
static std::atomic<void*> g_scratch_ptr[kMaxDevices];    // device address of `scratch` on each GPU, looked up once

extern "C" int bw_qgemm_static(const void* x, int act_dtype, int64_t M, int64_t K, int64_t ldx, const int32_t* qweight,
                               const void* scale16, const void* zp16, const void* bias, int64_t N, int bits, int group,
                               void* y, int64_t ldy, void* stream) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return BW_ELAUNCH;
    void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        // `scratch` names the array in host code only as a handle: its memory on the current device is at the
        // address this returns (each GPU holds its own copy at its own address)
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return BW_ELAUNCH;
        g_scratch_ptr[dev].store(ptr, std::memory_order_release);
    }
    // (plans of 192-column tiles always fit)
    const bool fast = bw_shape_ok(N, K, bits, group) && M >= 1 && M < ((int64_t)1 << 31) && bw_fast_shape(M, N, K, K, bits, group);
    if (fast && gemm_wide_ws_bytes(M, N, K, bits) > kScratchBytes) return BW_EWORKSPACE;
    return bw_qgemm_ws(x, act_dtype, M, K, ldx, qweight, scale16, zp16, bias, N, bits, group, y, ldy, ptr, kScratchBytes, stream);
}

extern "C" int bw_qgemm(const void* x, int act_dtype, int64_t M, int64_t K, int64_t ldx, const int32_t* qweight,
                        const void* scale16, const void* zp16, const void* bias, int64_t N, int bits, int group,
                        void* y, int64_t ldy, void* stream) {
    return bw_qgemm_ws(x, act_dtype, M, K, ldx, qweight, scale16, zp16, bias, N, bits, group, y, ldy, nullptr, 0, stream);
}
