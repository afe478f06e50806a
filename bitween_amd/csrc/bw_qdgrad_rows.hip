// bw_qdgrad_rows.hip - the input gradient of a few rows: grad_x[M][K] = grad_y[M][N] @ W16[N][K] for M <= 48.
//
// The kernels of bw_qdgrad.hip dequantise a weight tile into LDS to read it back transposed, in tiles of 128 rows of m and more; with a few
// rows of grad_y that fill is all they do (16 rows of 4096 <- 11008, W4 g128: 1.6 us a step of 64 n for 0.5 us of MFMAs, seven
// eighths of them padding).  Here no weight crosses LDS.  A lane holds the same 16 consecutive k of 8 consecutive rows n, so the 8 values of one
// k that an MFMA operand wants are in its registers, one in each of 8 words: two byte permutes make pairs (n, n + 1) of the words, and
// the masks that unpack neighbouring k elsewhere here unpack neighbouring n, each with its own scale and zero point.  One MFMA multiplies 32 n x 16
// columns that are 16 apart; which columns lie together is the business of the stores only.
//   * A workgroup owns 256 columns (16 lanes x 16) and a slice of N; its waves take steps of 32 n in turn, weights and scales of the next one
//     requested ahead, 16 lanes to the 128 bytes (4 bits) of a row.  Scales and zero points of a step - two, four or eight groups of 32
//     rows - come in 32 lanes to an array and are turned to [group][n] in the wave's own LDS.
//   * What bounds it now: the unpack (28 vector instructions for 16 weights, pairs included) and the sums of the waves, 64 KB a workgroup for 16
//     rows; 16 rows of 4096 <- 11008 take 12.0 us here and 3.8 in the reduction (kernel trace; 14.2 as a graph), of which the weights' way out of HBM is 3.5.
//   * The waves' sums meet in LDS, sixteen rows of m at a time; slices of N go through the caller's workspace and qdgrad_rows_reduce_kernel.
#include "bw_qdgrad_rows.h"

namespace {

typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));

// two float32 -> two 16-bit values of the gradient's type, round to nearest even, as one dword
template <int DT>
BW_DEV uint32_t round2(float a, float b) {
    if constexpr (DT == BW_F16) return as_u32(h2{(_Float16)a, (_Float16)b});
    else return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, bf2));
}

BW_DEV __amdgpu_buffer_rsrc_t rows_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// Columns of a workgroup, n of a step, waves.  Eight waves write twice the sums into LDS and read them back: 16 rows of 4096 <- 4096 11.3 us, with four
// waves 10.4; 4096 <- 11008 15.5 and 14.2; 32 rows 14.4 and 13.2, 19.3 and 17.8 (W4 g128).
constexpr int RK = 256, RN = 32, RW = 4;

// Waves a SIMD that the registers leave room for (a grid has one workgroup a CU at most: what counts is how the compiler lays them out).  Two, as long as
// nothing spills: a spilled register comes back through the counter of the loads and waits for all that is requested ahead.  8 bits, bfloat16, two
// row tiles in groups of 32 and 64 do not fit (4 and 2 spilled, with two waves 1.03 ... 1.04 and 0.93 ... 0.97 of the other kernels' time on 2981 calls, with one
// 0.79 ... 0.85 and 0.73 ... 0.81); in groups of 128 two are ahead (0.69 ... 0.77 against 0.72 ... 0.80), as at 4 and 2 bits (one takes 1.03 ... 1.07 of their time).
template <int BITS, int GROUP, int DT, int MT>
constexpr int rows_waves = MT > 2 || (MT == 2 && BITS == 8 && GROUP < 128 && DT == BW_BF16) ? 1 : 2;

template <int BITS, int GROUP, int DT, int MT>
__global__ __launch_bounds__(64 * RW, (rows_waves<BITS, GROUP, DT, MT>)) void qdgrad_rows_kernel(const DgradRowsArgs a) {
    constexpr int W = RW, GS = RK / GROUP, LANE_BYTES = 2 * BITS, WORDS = LANE_BYTES / 4;
    constexpr uint32_t kOob = 0x80000000u;
    constexpr int META = 2 * GS * RN * 2;                              // a wave's scales and zero points of a step, [array][group][n]
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 15, kq = lane >> 4;
    const int strip = (int)blockIdx.x / a.splits, slice = (int)blockIdx.x - strip * a.splits;
    const int k0 = strip * RK + nl * 16;                               // the lane's 16 columns
    const int s_begin = slice * a.steps_per_split, s_end = min(s_begin + a.steps_per_split, (a.N + RN - 1) / RN);
    const int mine = (s_end - s_begin - wave + W - 1) / W;             // steps of this wave: s_begin + wave, + W, ...
    char* const meta = smem + wave * META;
    const __amdgpu_buffer_rsrc_t rw = rows_rsrc(a.qweight, a.w_bytes), rs = rows_rsrc(a.scale, a.meta_bytes), rz = rows_rsrc(a.zp, a.meta_bytes),
                                 rg = rows_rsrc(a.go, a.go_bytes);

    struct Step {
        uint32_t w[8][WORDS];
        uint32_t s[GS / 2], z[GS / 2];
        u4 g[MT];
    };
    Step step[2];
    const uint32_t w_lane = k0 < a.K ? (uint32_t)(8 * kq) * a.row_bytes + (uint32_t)k0 * BITS / 8 : kOob;
    const uint32_t m_lane = lane < 32 ? ((uint32_t)lane * a.groups + strip * GS) * 2 : kOob;
    auto issue = [&](Step& t, int r) {
        const int n = (s_begin + wave + W * r) * RN;                   // (rows past N lie past every buffer: zeros)
        const bool live = r < mine;
        const uint32_t wo = __builtin_amdgcn_readfirstlane(live ? (uint32_t)n * a.row_bytes : kOob), mo = __builtin_amdgcn_readfirstlane(live ? (uint32_t)n * a.groups * 2 : kOob);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t off = w_lane + wo + (uint32_t)i * a.row_bytes;
            if constexpr (WORDS == 1) t.w[i][0] = __builtin_amdgcn_raw_buffer_load_b32(rw, off, 0, 0);
            else if constexpr (WORDS == 2) {
                const u2 v = __builtin_amdgcn_raw_buffer_load_b64(rw, off, 0, 0);
                t.w[i][0] = v[0]; t.w[i][1] = v[1];
            } else {
                const u4 v = __builtin_amdgcn_raw_buffer_load_b128(rw, off, 0, 0);
                t.w[i][0] = v[0]; t.w[i][1] = v[1]; t.w[i][2] = v[2]; t.w[i][3] = v[3];
            }
        }
        auto load_meta = [&](const __amdgpu_buffer_rsrc_t& rsrc, uint32_t* m) {
            if constexpr (GS == 2) m[0] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, m_lane + mo, 0, 0);
            else if constexpr (GS == 4) {
                const u2 v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, m_lane + mo, 0, 0);
                m[0] = v[0]; m[1] = v[1];
            } else {
                const u4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, m_lane + mo, 0, 0);
                m[0] = v[0]; m[1] = v[1]; m[2] = v[2]; m[3] = v[3];
            }
        };
        load_meta(rs, t.s);
        load_meta(rz, t.z);
        const int c = n + 8 * kq;                                      // (N is a multiple of 8)
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const uint32_t off = (uint32_t)((16 * i + nl) * a.ldg + c) * 2;
            t.g[i] = __builtin_amdgcn_raw_buffer_load_b128(rg, live && c < a.N && 16 * i + nl < a.M ? off : kOob, 0, 0);
        }
    };

    f4 acc[MT][16];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < 16; t++) acc[i][t] = f4{0.f, 0.f, 0.f, 0.f};
    const char* const my_meta = meta + (nl * 16 / GROUP) * (RN * 2) + kq * 16;   // the lane's group, its 8 rows
    auto body = [&](Step& t, int r) {
        // scales and zero points -> [array][group][n]
        if (lane < 32) {
#pragma unroll
            for (int g = 0; g < GS; g++) {
                *reinterpret_cast<uint16_t*>(meta + (g * RN + lane) * 2) = (uint16_t)(t.s[g / 2] >> (16 * (g & 1)));
                *reinterpret_cast<uint16_t*>(meta + ((GS + g) * RN + lane) * 2) = (uint16_t)(t.z[g / 2] >> (16 * (g & 1)));
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const u4 sv = *reinterpret_cast<const u4*>(my_meta), zv = *reinterpret_cast<const u4*>(my_meta + GS * RN * 2);
        __builtin_amdgcn_wave_barrier();
        h2 s[4], z0[4], z1[4], z2[4], z3[4];                           // of rows 2 p, 2 p + 1 of the lane's eight: -(1024 + z), -(64 + z); 2 bits: -(256 + z), -(64 + z), -(16 + z)
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const uint32_t sw = sv[p], zw = zv[p];
            s[p] = as_h2(sw);
            z0[p] = splat((_Float16)(-1024.0f)) - as_h2(zw);
            z1[p] = splat((_Float16)(BITS == 2 ? -256.0f : -64.0f)) - as_h2(zw);
            z2[p] = splat((_Float16)(-64.0f)) - as_h2(zw);
            z3[p] = splat((_Float16)(-16.0f)) - as_h2(zw);
        }
        const h2 k4 = splat((_Float16)0.25f), k16 = splat((_Float16)0.0625f), k64 = splat((_Float16)0.015625f);
#pragma unroll
        for (int b = 0; b < 4; b++) {                                  // columns 4 b .. + 3 of the lane's sixteen
            __builtin_amdgcn_sched_barrier(0);                         // (four blocks unpacked ahead spill 30 ... 180 registers)
            h2 o[4][4];                                                // [column][pair of rows]: q - z, exact
#pragma unroll
            for (int p = 0; p < 4; p++) {
                if constexpr (BITS == 8) {
                    const uint32_t lo = t.w[2 * p][b], hi = t.w[2 * p + 1][b];
                    o[0][p] = as_h2(__builtin_amdgcn_perm(hi, lo, 0x0C040C00u) | kMagic) + z0[p];
                    o[1][p] = as_h2(__builtin_amdgcn_perm(hi, lo, 0x0C050C01u) | kMagic) + z0[p];
                    o[2][p] = as_h2(__builtin_amdgcn_perm(hi, lo, 0x0C060C02u) | kMagic) + z0[p];
                    o[3][p] = as_h2(__builtin_amdgcn_perm(hi, lo, 0x0C070C03u) | kMagic) + z0[p];
                } else {
                    constexpr uint32_t low = 0x05040100u, high = 0x07060302u;
                    const int word = BITS == 4 ? b / 2 : 0;
                    const uint32_t pair = __builtin_amdgcn_perm(t.w[2 * p + 1][word], t.w[2 * p][word], (BITS == 4 ? b % 2 : b / 2) ? high : low);
                    if constexpr (BITS == 4) {
                        const uint32_t up = pair >> 8;
                        o[0][p] = as_h2(and_or(pair, 0x000F000Fu, kMagic)) + z0[p];
                        o[1][p] = __builtin_elementwise_fma(as_h2(and_or(pair, 0x00F000F0u, kMagic)), k16, z1[p]);
                        o[2][p] = as_h2(and_or(up, 0x000F000Fu, kMagic)) + z0[p];
                        o[3][p] = __builtin_elementwise_fma(as_h2(and_or(up, 0x00F000F0u, kMagic)), k16, z1[p]);
                    } else {
                        const uint32_t x = b % 2 ? pair >> 8 : pair;
                        o[0][p] = as_h2(and_or(x, 0x00030003u, kMagic)) + z0[p];
                        o[1][p] = __builtin_elementwise_fma(as_h2(and_or(x, 0x000C000Cu, kMagic)), k4, z1[p]);
                        o[2][p] = __builtin_elementwise_fma(as_h2(and_or(x, 0x00300030u, kMagic)), k16, z2[p]);
                        o[3][p] = __builtin_elementwise_fma(as_h2(and_or(x, 0x00C000C0u, kMagic)), k64, z3[p]);
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                u4 f;
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    if constexpr (DT == BW_F16) f[p] = as_u32(o[j][p] * s[p]);
                    else f[p] = round2<DT>((float)o[j][p][0] * (float)s[p][0], (float)o[j][p][1] * (float)s[p][1]);
                }
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const u4 g = t.g[i];
                    if constexpr (DT == BW_F16) acc[i][4 * b + j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, g), __builtin_bit_cast(h8, f), acc[i][4 * b + j], 0, 0, 0);
                    else acc[i][4 * b + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, g), __builtin_bit_cast(bf8, f), acc[i][4 * b + j], 0, 0, 0);
                }
            }
        }
        issue(t, r + 2);
    };
    issue(step[0], 0);
    issue(step[1], 1);
    int r = 0;
    for (; r + 2 <= mine; r += 2) {
        body(step[0], r);
        body(step[1], r + 1);
    }
    if (r < mine) body(step[0], r);

    // acc[i][t][e] of a lane: row 16 i + 4 kq + e, column k0 + t.  A wave's 16 rows in LDS: rows of 64 pieces of four columns and one of
    // padding, piece 4 nl + q at q ^ (nl >> 2 & 3), so that the sixteen lanes of a row spread over the banks.
    constexpr int PIECES = RK / 4 + 1;
    f4* const red = reinterpret_cast<f4*>(smem);
#pragma unroll
    for (int i = 0; i < MT; i++) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                red[(wave * 16 + 4 * kq + e) * PIECES + 4 * nl + (q ^ (nl >> 2 & 3))] = f4{acc[i][4 * q][e], acc[i][4 * q + 1][e], acc[i][4 * q + 2][e], acc[i][4 * q + 3][e]};
        __syncthreads();
        for (int it = tid; it < 16 * (RK / 4); it += 64 * W) {
            const int row = it / (RK / 4), piece = it % (RK / 4), m = 16 * i + row, k = strip * RK + 4 * piece;
            if (m >= a.M || k >= a.K) continue;
            const int at = row * PIECES + ((piece & ~3) | ((piece & 3) ^ (piece >> 4 & 3)));
            f4 v = red[at];
#pragma unroll
            for (int w = 1; w < W; w++) v += red[w * 16 * PIECES + at];
            *reinterpret_cast<f4*>(a.ws + ((int64_t)slice * a.M + m) * a.K + k) = v;
        }
    }
}

// grad_x = sum over the slices, rounded once.  A thread owns four columns of one row.
template <int DT>
__global__ __launch_bounds__(256) void qdgrad_rows_reduce_kernel(const float* __restrict__ ws, _Float16* __restrict__ gx, int M, int K, int ldx, int splits) {
    const int quads = K >> 2, idx = (int)blockIdx.x * 256 + threadIdx.x;
    if (idx >= M * quads) return;
    const int m = idx / quads, k = (idx - m * quads) * 4;
    const float* p = ws + (int64_t)m * K + k;
    const int64_t part = (int64_t)M * K;
    f4 v = {0.f, 0.f, 0.f, 0.f};
    int z = 0;
    for (; z + 4 <= splits; z += 4) {
        f4 t[4];
#pragma unroll
        for (int e = 0; e < 4; e++) t[e] = *reinterpret_cast<const f4*>(p + (z + e) * part);
#pragma unroll
        for (int e = 0; e < 4; e++) v += t[e];
    }
    for (; z < splits; z++) v += *reinterpret_cast<const f4*>(p + z * part);
    *reinterpret_cast<u2*>(gx + (int64_t)m * ldx + k) = u2{round2<DT>(v[0], v[1]), round2<DT>(v[2], v[3])};
}

template <int BITS, int GROUP, int DT, int MT>
int launch_rows(const DgradRowsArgs& a, hipStream_t stream) {
    constexpr int LDS = RW * 16 * (RK / 4 + 1) * 16;
    static_assert(LDS <= 160 * 1024 && 2 * (RK / GROUP) * RN * 2 <= 16 * (RK / 4 + 1) * 16, "a wave's scales lie where its sums go later");
    auto kern = qdgrad_rows_kernel<BITS, GROUP, DT, MT>;
    static uint64_t big_lds_devices = 0;                   // per instantiation
    if (LDS > 64 * 1024 && !bw_allow_big_lds(reinterpret_cast<const void*>(kern), big_lds_devices)) return BW_ELAUNCH;
    hipLaunchKernelGGL(kern, dim3((unsigned)((a.K + RK - 1) / RK * a.splits)), dim3(64 * RW), LDS, stream, a);
    if (hipGetLastError() != hipSuccess) return BW_ELAUNCH;
    hipLaunchKernelGGL(qdgrad_rows_reduce_kernel<DT>, dim3((unsigned)(((int64_t)a.M * (a.K / 4) + 255) / 256)), dim3(256), 0, stream, a.ws, a.gx, a.M, a.K, a.ldx, a.splits);
    return hipGetLastError() == hipSuccess ? BW_OK : BW_ELAUNCH;
}

template <int BITS, int GROUP>
int launch_rows_group(const DgradRowsArgs& a, int dtype, hipStream_t stream) {
#define BW_MT(T, DT) \
    if (a.M <= 16 * T && dtype == DT) return launch_rows<BITS, GROUP, DT, T>(a, stream);
    BW_MT(1, BW_F16) BW_MT(1, BW_BF16) BW_MT(2, BW_F16) BW_MT(2, BW_BF16) BW_MT(3, BW_F16)
#undef BW_MT
    return BW_EUNSUPPORTED;
}

}  // namespace

int bw_launch_dgrad_rows(const DgradRowsArgs& a, int bits, int group, int dtype, hipStream_t stream) {
#define BW_CASE(B, G) if (bits == B && group == G) return launch_rows_group<B, G>(a, dtype, stream);
    BW_CASE(4, 128) BW_CASE(4, 64) BW_CASE(4, 32)
    BW_CASE(8, 128) BW_CASE(8, 64) BW_CASE(8, 32)
    BW_CASE(2, 128) BW_CASE(2, 64) BW_CASE(2, 32)
#undef BW_CASE
    return BW_EUNSUPPORTED;
}
