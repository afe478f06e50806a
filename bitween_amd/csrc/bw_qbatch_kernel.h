// bw_qbatch_kernel.h - the batch kernel: y[M][N] = x[M][K] @ W16[N][K]^T (+ bias) for M of a serving batch, shared by the
// translation units that instantiate it per weight width (bw_qbatch.hip and bw_qbatch_w*.hip, compiled in parallel).
//
// Between the decode kernels (16 rows a launch) and the prefill kernel (tiles of 64 x 256 outputs and more) a call is
// bound by how many bytes a compute unit has to take in: every workgroup needs its slice of x, so x crosses from L2 to
// the CUs N / BN times, next to the weights once from HBM.  A workgroup of 8 waves owns all M rows (128 of them beyond that) x
// BN = 32 NTW output columns and a slice of K:
//   * K is walked in rounds of 512 values (256 beyond 64 rows); of a round's four chunks each wave takes one (kw) and NTW of the
//     2 NTW column tiles (wn), so that the grid has enough workgroups for narrow layers and a fragment of x read from LDS
//     feeds NTW MFMAs;
//   * x goes global -> registers -> LDS (double buffered, one round ahead), converted from bfloat16 straight into the order the unpack
//     emits, or permuted to it, on the way; scales and zero points of a round come in with it, whole rows at a time.  One set of
//     registers, asked for a round before it is staged: x comes out of L2, a round is long enough for that, and the first multiplication
//     waits for one request fewer (two sets: 40 rows of 4096 -> 12288, W4 g64, bfloat16 16.3 us, one 15.4; 128 rows of 4096 -> 14336, g128, 26.6 and
//     25.9; permuting after the conversion instead of converting into the order 16.7 and 27.2);
//   * weights go global -> registers two rounds ahead, four lanes to the 64 bytes of a row, are permuted between the lanes
//     to operand layout (ds_bpermute) and unpacked to the reference's W16 in registers.  Asking for them in operand layout
//     right away (neighbouring lanes on neighbouring rows) costs the address unit 60 cycles an instruction instead of 16:
//     37 bytes/ns per CU out of L2 instead of 109;
//   * what bounds it (128 rows of 4096 -> 14336, MT = NTW = 4, float16, 25.6 us): without a loop 10.8 (launch 2.4, the first requests 6,
//     the sums of the four waves 2.2), without unpack and MFMAs 19.2, without memory 21.2 - LDS (x in once, out twice: 1.5 MB a
//     workgroup), the vector unit and the matrix pipe each need 8 ... 10 us and two waves a SIMD in step overlap them in part;
//   * the four waves that share columns add up through LDS at the end.  Where N / BN leaves CUs idle K is also cut
//     across workgroups: float32 partial sums in the caller's workspace, added by qbatch_reduce_kernel.
#pragma once
#include "bw_common.h"

struct BatchArgs {
    const void* x;
    const void* qweight;
    const void* scale;
    const void* zp;
    const _Float16* bias;
    _Float16* y;
    float* ws;                        // splits > 1: [splits][M][npad] partial sums
    uint32_t x_bytes, w_bytes, meta_bytes;
    int M, N, K, ldx, ldy, npad;
    int groups, row_bytes, nchunks;   // chunks of 128 values of K
    int splits, chunks_per_split, mtiles, ntiles;
    int x_bf16, sums;
};

// rows of 16 (mt) and column tiles per wave (ntw) of the launch; BW_EUNSUPPORTED for a combination that is not built
int bw_launch_qbatch_w2(int group, int mt, int ntw, const BatchArgs& a, hipStream_t stream);
int bw_launch_qbatch_w4(int group, int mt, int ntw, const BatchArgs& a, hipStream_t stream);
int bw_launch_qbatch_w8(int group, int mt, int ntw, const BatchArgs& a, hipStream_t stream);

// Tiles of which there is a kernel that multiplies sums of a group by its scale, and not every weight.
constexpr bool bw_qbatch_sums(int bits, int group, int mt, int ntw) {
    return group == 128 && bits != 2 && mt <= 3 && mt * ntw <= (bits == 4 ? 6 : 4);
}

namespace {

constexpr uint32_t kBatchMaxBytes = 0x7FFF0000u;                      // extent of x a launch takes

BW_DEV __amdgpu_buffer_rsrc_t batch_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// Shape of a workgroup of 8 waves: KR values of K per round, cut over WK = 4 waves of CK values (VPL of them in a lane); WN = 2
// waves side by side over the columns.  Up to 64 rows a round is 512 values; beyond, x of a round would not fit LDS twice.
// (Beyond 64 rows as 2 waves of 128 values x 4 side by side, every fragment of x crossed LDS four times instead of twice, and
// LDS was what the loop waited for.)
template <int MT, int NTW>
struct BatchCfg {
    static constexpr int KR = MT <= 4 ? 512 : 256, WK = 4, CK = KR / WK, VPL = CK / 4, WN = 2, BN = 16 * WN * NTW;
    static constexpr int PITCH = (KR + 8) * 2;                        // bytes of an LDS row of x
    static constexpr int X_BYTES = 16 * MT * PITCH;
    static constexpr int RPW = 512 / KR, PASSES = 2 * MT / RPW;       // rows a wave stages per pass, passes per round
    template <int GROUP> static constexpr int lds() {
        const int two = 2 * (X_BYTES + 2 * BN * (KR / GROUP) * 2), red = WK * 16 * MT * (BN / 4 + 1) * 16;
        return two > red ? two : red;
    }
};

template <int BITS, int GROUP, int MT, int NTW, bool BF16, bool SUMS>
__global__ __launch_bounds__(512, 2) void qbatch_kernel(const BatchArgs a) {
    constexpr uint32_t kOob = 0x80000000u, kOobRow = kBatchMaxBytes;   // beyond every buffer, also added to one another
    using C = BatchCfg<MT, NTW>;
    constexpr int KR = C::KR, WK = C::WK, CK = C::CK, VPL = C::VPL, BN = C::BN, PITCH = C::PITCH, PASSES = C::PASSES, X_BYTES = C::X_BYTES;
    constexpr int LANE_BYTES = VPL * BITS / 8, STEPS = VPL / 8;       // packed bytes, and MFMA steps, of a lane's weights of a round
    constexpr int WL = LANE_BYTES > 16 ? LANE_BYTES / 16 : 1, WW = LANE_BYTES > 16 ? 4 : LANE_BYTES / 4;   // requests, words of each
    constexpr int CHUNK_BYTES = CK * BITS / 8, GR = KR / GROUP;       // groups per round
    constexpr int ML = (BN * GR / 2 + 255) / 256;                     // words of scales (zero points) a thread brings in
    constexpr int BUF = X_BYTES + 2 * BN * GR * 2;
    // SUMS: a wave's chunk is one group; its partial dot product of the exact q - z is multiplied by the scale in float32, as the decode
    // kernels do it, so that calls of a few rows keep their rounding: 2.07e-4 against scale * (q - z) in 64 bits, 2.76e-4 with
    // every weight rounded to float16 - the reference's W16, against which the errors are the other way round.  Only tiles
    // whose registers hold both sums (3 x 3 at 4 bits, 3 x 2 at 8 spill: 20 -> 50 us); as fast as W16.
    static_assert(!SUMS || GROUP == CK);
    constexpr int XF = MT * NTW >= 12 ? 1 : 2;                        // sets of x fragments: the next step's are read early where registers allow
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 15, kq = lane >> 4, kw = wave % WK, wn = wave / WK;
    // Which tile.  Workgroups go to the 8 XCDs round-robin.  Where x is more than an XCD's L2 takes beside the weights (2 MB) each XCD works
    // through one contiguous eighth of the tiles, slice by slice of K, in panels of four tiles of rows, columns last, instead of
    // reading all of x: W4 g128 us, 999 x 8192 -> 544 29.8 -> 23.1, 300 x 4096 -> 4096 20.7 -> 19.4; W2 1146 x 10240 -> 529 38.4 -> 28.2.
    // Elsewhere the slices of a tile, then its columns, lie side by side: 128 x 14336 -> 4096 in four slices 28.0, the other way 28.7.
    // (Divisions only where there is something to divide: the five of the first order cost 0.15 us a launch.)
    int slice = 0, ntile, mtile = 0;
    if (a.mtiles >= 4 && a.x_bytes > (2u << 20)) {
        const int xcd = (int)blockIdx.x & 7, share = (int)gridDim.x >> 3, extra = (int)gridDim.x & 7, tiles = a.mtiles * a.ntiles;
        int tile = xcd * share + min(xcd, extra) + ((int)blockIdx.x >> 3);
        slice = tile / tiles;
        tile -= slice * tiles;
        const int panel = tile / (4 * a.ntiles), rows = min(4, a.mtiles - 4 * panel);
        tile -= panel * 4 * a.ntiles;
        ntile = tile / rows;
        mtile = 4 * panel + tile - ntile * rows;
    } else {
        ntile = (int)blockIdx.x;
        if (a.splits > 1) {
            ntile /= a.splits;
            slice = (int)blockIdx.x - ntile * a.splits;
        }
        if (a.mtiles > 1) {
            mtile = ntile / a.ntiles;
            ntile -= mtile * a.ntiles;
        }
    }
    const int n_base = ntile * BN, m_base = mtile * 16 * MT;
    const int M = min(a.M - m_base, 16 * MT);                         // rows of this tile
    // chunks of CK values (the slices are counted in 128s)
    const int c_begin = slice * a.chunks_per_split * (128 / CK), c_end = min(a.nchunks, (slice + 1) * a.chunks_per_split) * (128 / CK);
    const int rounds = (c_end - c_begin + WK - 1) / WK;
    const int k_end = min(a.K, c_end * CK);
    const __amdgpu_buffer_rsrc_t rw = batch_rsrc(a.qweight, a.w_bytes),
                                 rx = batch_rsrc((const char*)a.x + (int64_t)m_base * a.ldx * 2, a.x_bytes - (uint32_t)m_base * a.ldx * 2);

    uint32_t w_off[NTW];
#pragma unroll
    for (int j = 0; j < NTW; j++) {
        const int row = min(n_base + (wn * NTW + j) * 16 + (lane >> 2), a.N - 1);   // columns past N repeat the last one and are not stored
        w_off[j] = (uint32_t)row * a.row_bytes + (lane & 3) * LANE_BYTES + kw * CHUNK_BYTES;
    }
    struct WSet { u4 w[NTW][WL]; };
    WSet wset[2];
    auto w_scalar = [&](int r) {
        // one VGPR per tile plus a scalar (opaque, or the compiler makes branches with full waits of the selection); past the
        // slice the scalar lies beyond every buffer and the hardware's range check returns zeros
        const int c = c_begin + WK * r;
        return (uint32_t)__builtin_amdgcn_readfirstlane(c + kw < c_end ? (uint32_t)c * CHUNK_BYTES : kOob);
    };
    auto issue_w = [&](WSet& s, int j, int l, uint32_t so) {
        const uint32_t off = w_off[j] + so;
        if constexpr (WW == 1) {
            s.w[j][0][0] = __builtin_amdgcn_raw_buffer_load_b32(rw, off, 0, 0);
        } else if constexpr (WW == 2) {
            const u2 v = __builtin_amdgcn_raw_buffer_load_b64(rw, off, 0, 0);
            s.w[j][0][0] = v[0];
            s.w[j][0][1] = v[1];
        } else {
            s.w[j][l] = __builtin_amdgcn_raw_buffer_load_b128(rw, off + 16 * l, 0, 0);
        }
    };
    // x: pass p of a wave stages RPW rows of the round, 8 values a lane.  All workgroups of a slice ask for the same rows at about
    // the same time, which L2 serves better than requests that start at different rows (16.4 against 17.0 us at 40 rows of
    // 4096 -> 14336).
    struct XSet { u4 x[PASSES]; u2 m[ML]; };                  // a thread's share of a round: x, and scales or zero points
    XSet xset;
    auto x_row = [&](int p) { return (p * 8 + wave) * C::RPW; };
    const int sub = C::RPW == 1 ? 0 : lane / (KR / 8), col = (C::RPW == 1 ? lane : lane % (KR / 8)) * 8;   // of the lane in its wave's pass
    uint32_t row_off[PASSES];                                 // scalars
#pragma unroll
    for (int p = 0; p < PASSES; p++) {
        const int row = x_row(p);                             // (row + 1 = M of an odd M lies past the buffer's end)
        row_off[p] = __builtin_amdgcn_readfirstlane(row < M ? (uint32_t)row * a.ldx * 2 : kOobRow);
    }
    auto x_offset = [&](int r) {
        const int k = (c_begin + WK * r) * CK + col;
        return k < k_end ? (uint32_t)(k + sub * a.ldx) * 2 : kOob;
    };
    auto issue_x = [&](XSet& xs, int p, uint32_t ko) { xs.x[p] = __builtin_amdgcn_raw_buffer_load_b128(rx, ko + row_off[p], 0, 0); };
    // scales (waves 0 - 3) and zero points (waves 4 - 7) of a round: GR / 2 words for each of the BN columns, neighbouring
    // threads on neighbouring words; 8 bytes from the 4-byte boundary below, of which the row's parity (and the array's, where it starts
    // off a 4-byte boundary, as a row slice of an odd number of groups may) picks two halves
    uint32_t meta_off[ML], meta_shift[ML];
    // (of the pointer itself: two more kernel arguments cost every launch 0.2 ... 0.35 us; the two bytes ahead of such an array belong to
    // the word it starts in)
    const char* const marr = (const char*)(wave < 4 ? a.scale : a.zp);
    const uint32_t skew = (uint32_t)(uintptr_t)marr & 2u;
#pragma unroll
    for (int i = 0; i < ML; i++) {
        const int item = (tid & 255) + 256 * i, n = item / (GR / 2), w = item - n * (GR / 2);
        const uint32_t off = (uint32_t)(min(n_base + n, a.N - 1) * a.groups + c_begin * CK / GROUP) * 2 + 4 * w + skew;
        meta_off[i] = n < BN ? off & ~3u : kOob;
        meta_shift[i] = (off & 2) * 8;
    }
    const __amdgpu_buffer_rsrc_t rm = batch_rsrc(marr - skew, (a.meta_bytes + skew + 3) & ~3u);
    auto issue_meta = [&](XSet& xs, int i, int r) { xs.m[i] = __builtin_amdgcn_raw_buffer_load_b64(rm, meta_off[i] + (uint32_t)r * (GR * 2), 0, 0); };
    auto stage_x = [&](const XSet& xs, int p, char* buf) {
        const u4 in = xs.x[p];
        u4 o;                                                 // pairs (k, k + 4) at 4 bits: the order dequant_word4 emits
        if constexpr (BF16) {
            float lo[4], hi[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                lo[j] = __builtin_bit_cast(float, in[j] << 16);
                hi[j] = __builtin_bit_cast(float, in[j] & 0xFFFF0000u);
            }
            if constexpr (BITS == 4) {
                o[0] = as_u32(h2{(_Float16)lo[0], (_Float16)lo[2]});
                o[1] = as_u32(h2{(_Float16)hi[0], (_Float16)hi[2]});
                o[2] = as_u32(h2{(_Float16)lo[1], (_Float16)lo[3]});
                o[3] = as_u32(h2{(_Float16)hi[1], (_Float16)hi[3]});
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) o[j] = as_u32(h2{(_Float16)lo[j], (_Float16)hi[j]});
            }
        } else if constexpr (BITS == 4) {
            o[0] = __builtin_amdgcn_perm(in[2], in[0], 0x05040100u);
            o[1] = __builtin_amdgcn_perm(in[2], in[0], 0x07060302u);
            o[2] = __builtin_amdgcn_perm(in[3], in[1], 0x05040100u);
            o[3] = __builtin_amdgcn_perm(in[3], in[1], 0x07060302u);
        } else o = in;
        *reinterpret_cast<u4*>(buf + (x_row(p) + sub) * PITCH + col * 2) = o;
    };
    auto stage_meta = [&](const XSet& xs, int i, char* buf) {
        const int item = (tid & 255) + 256 * i;
        if (item < BN * GR / 2) reinterpret_cast<uint32_t*>(buf + X_BYTES)[(wave >> 2) * (BN * GR / 2) + item] = __builtin_amdgcn_alignbit(xs.m[i][1], xs.m[i][0], meta_shift[i]);
    };

    f4 acc[MT][NTW];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NTW; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    using GC = std::conditional_t<BITS == 4, GroupConst<4>, GroupConstNat<BITS>>;
    // the lane that asked for a piece -> the lane that multiplies it
    const int from = ((nl << 2) | kq) << 2;
    auto permute_w = [&](WSet& s, const WSet& q, int j, int l) {
#pragma unroll
        for (int e = 0; e < WW; e++) s.w[j][l][e] = __builtin_amdgcn_ds_bpermute(from, (int)q.w[j][l][e]);
    };
    // One round: multiply what lies in `cur` and `s`; and, dealt out over the column tiles' MFMA groups so that neither the
    // address unit nor LDS sees a burst while the matrix pipe idles (12288 x 4096 at 40 rows 18.2 -> 15.9 us),
    // put round r + 1 into `nxt` and `sn` from the registers it was requested into, and request x of round r + 2 and weights
    // of round r + 3 there.
    constexpr int TASKS = PASSES + ML + NTW * WL, SLOTS = STEPS * NTW;
    auto round = [&](auto more, const char* cur, char* nxt, XSet& xs, WSet& wq, const WSet& s, WSet& sn, int r) {
        constexpr bool MORE = decltype(more)::value;
        // the lane's group of the round, kept inside the row
        const int g = min((kw * CK + kq * VPL) / GROUP, a.groups - 1 - (c_begin + WK * r) * CK / GROUP);
        const uint32_t ko = x_offset(r + 2), so = w_scalar(r + 3);
        GC gc[NTW];
#pragma unroll
        for (int j = 0; j < NTW; j++) {
            const _Float16* m = reinterpret_cast<const _Float16*>(cur + X_BYTES) + ((wn * NTW + j) * 16 + nl) * GR + g;
            // values past K (of the last round only) meet zeros of x; what is unpacked there must be finite
            const bool past = !MORE && (c_begin + WK * r + kw) * CK + kq * VPL >= a.K;
            gc[j].set(past ? (_Float16)0.f : m[0], past ? (_Float16)0.f : m[BN * GR]);
        }
        f4 sc[SUMS ? NTW : 1];                                // of the columns a lane accumulates
        if constexpr (SUMS) {
#pragma unroll
            for (int j = 0; j < NTW; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) sc[j][e] = (float)reinterpret_cast<const _Float16*>(cur + X_BYTES)[((wn * NTW + j) * 16 + 4 * kq + e) * GR + g];
        }
        f4 part[SUMS ? MT : 1][SUMS ? NTW : 1];
        const char* xp = cur + nl * PITCH + (kw * CK + kq * VPL) * 2;
        h8 xf[XF][MT];
        auto read_x = [&](int t) {
#pragma unroll
            for (int i = 0; i < MT; i++) xf[t % XF][i] = *reinterpret_cast<const h8*>(xp + i * (16 * PITCH) + t * 16);
        };
        if constexpr (XF == 2) read_x(0);
        static_for<0, STEPS>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
            static_for<0, NTW>([&](auto jc) {
                constexpr int j = decltype(jc)::value, slot = t * NTW + j;
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (j == 0 && XF == 1) read_x(t);
                if constexpr (j == 0 && XF == 2 && t + 1 < STEPS) read_x(t + 1);
                h2 o[4];
                if constexpr (BITS == 4) dequant_word4<!SUMS>(s.w[j][0][t], gc[j], o);
                else if constexpr (BITS == 2) dequant_halfword2_nat(s.w[j][0][t / 2], t % 2, gc[j], o);
                else {
                    dequant_word8_nat<!SUMS>(s.w[j][t / 2][2 * (t % 2)], gc[j], o);
                    dequant_word8_nat<!SUMS>(s.w[j][t / 2][2 * (t % 2) + 1], gc[j], o + 2);
                }
                const h8 wf = pack_h8(o);
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    if constexpr (!SUMS) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, xf[t % XF][i], acc[i][j], 0, 0, 0);
                    else part[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, xf[t % XF][i], t == 0 ? f4{0.f, 0.f, 0.f, 0.f} : part[i][j], 0, 0, 0);
                }
                if constexpr (MORE) {
                    static_for<0, TASKS>([&](auto kc) {
                        constexpr int k = decltype(kc)::value;
                        if constexpr (k * SLOTS / TASKS == slot) {
                            if constexpr (k < PASSES) {
                                stage_x(xs, k, nxt);
                                issue_x(xs, k, ko);
                            } else if constexpr (k < PASSES + ML) {
                                stage_meta(xs, k - PASSES, nxt);
                                issue_meta(xs, k - PASSES, r + 2);
                            } else {
                                constexpr int jl = k - PASSES - ML;
                                permute_w(sn, wq, jl / WL, jl % WL);
                                issue_w(wq, jl / WL, jl % WL, so);
                            }
                        }
                    });
                }
            });
        });
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SUMS) {
#pragma unroll
            for (int j = 0; j < NTW; j++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[i][j][e] = __builtin_fmaf(part[i][j][e], sc[j][e], acc[i][j][e]);
        }
        if constexpr (MORE) __syncthreads();
    };
    auto request_x = [&](int r) {
        const uint32_t ko = x_offset(r);
#pragma unroll
        for (int p = 0; p < PASSES; p++) issue_x(xset, p, ko);
#pragma unroll
        for (int i = 0; i < ML; i++) issue_meta(xset, i, r);
    };
    auto request_w = [&](WSet& ws, int r) {
        const uint32_t so = w_scalar(r);
#pragma unroll
        for (int j = 0; j < NTW; j++)
#pragma unroll
            for (int l = 0; l < WL; l++) issue_w(ws, j, l, so);
    };
    WSet s0, s1;                                              // weights in operand layout: this round's, the next one's
    request_x(0);
    request_w(wset[0], 0);
    __builtin_amdgcn_sched_barrier(0);                        // the loop's wait counts assume this order of the requests
    request_w(wset[1], 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < PASSES; p++) stage_x(xset, p, smem);
#pragma unroll
    for (int i = 0; i < ML; i++) stage_meta(xset, i, smem);
    __builtin_amdgcn_sched_barrier(0);
    request_x(1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NTW; j++)
#pragma unroll
        for (int l = 0; l < WL; l++) permute_w(s0, wset[0], j, l);
    __builtin_amdgcn_sched_barrier(0);
    request_w(wset[0], 2);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    auto last = [&](const char* buf, const WSet& s, int r) {  // only the last round of a slice can have chunks past its end
        if (c_begin + WK * r + kw < c_end) round(std::false_type{}, buf, nullptr, xset, wset[0], s, s1, r);
    };
    // (whole pairs of rounds in a loop without a way out in the middle: another path to the loop's head, with fewer requests
    // behind it, would make every wait of the first half as strict as that path needs)
    int r = 0;
    for (; r + 2 < rounds; r += 2) {
        round(std::true_type{}, smem, smem + BUF, xset, wset[1], s0, s1, r);
        round(std::true_type{}, smem + BUF, smem, xset, wset[0], s1, s0, r + 1);
    }
    if (r + 1 < rounds) {
        round(std::true_type{}, smem, smem + BUF, xset, wset[1], s0, s1, r);
        last(smem + BUF, s1, r + 1);
    } else {
        last(smem, s0, r);
    }
    __syncthreads();

    // acc[i][j] of a lane: row 16 i + nl, columns 16 (wn NTW + j) + 4 kq .. + 3.  The waves' sums meet in LDS row-major (rows of
    // BN / 4 pieces of four columns, one piece of padding), so that neighbouring threads then add and store neighbouring
    // columns: whole 128-byte lines of y instead of 32 bytes in each of 16 rows per instruction.
    constexpr int QUADS = BN / 4;
    f4* red = reinterpret_cast<f4*>(smem);
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NTW; j++) red[(kw * 16 * MT + 16 * i + nl) * (QUADS + 1) + 4 * (wn * NTW + j) + kq] = acc[i][j];
    __syncthreads();
    const bool wide = a.ldy % 4 == 0 && ((uintptr_t)a.y & 7) == 0;
    const int items = M * QUADS;
    for (int t = tid; t < items; t += 512) {
        const int m = t / QUADS, q = t - m * QUADS, n = n_base + 4 * q;
        if (n >= a.N) continue;
        f4 v = red[m * (QUADS + 1) + q];
#pragma unroll
        for (int w = 1; w < WK; w++) v += red[(w * 16 * MT + m) * (QUADS + 1) + q];
        if (a.splits > 1) {
            *reinterpret_cast<f4*>(a.ws + ((int64_t)slice * a.M + m_base + m) * a.npad + n) = v;
            continue;
        }
        _Float16 h[4];
#pragma unroll
        for (int e = 0; e < 4; e++) h[e] = (_Float16)(v[e] + (a.bias && n + e < a.N ? (float)a.bias[n + e] : 0.f));
        _Float16* dst = a.y + (int64_t)(m_base + m) * a.ldy + n;
        if (wide && n + 3 < a.N) {
            *reinterpret_cast<u2*>(dst) = u2{as_u32(h2{h[0], h[1]}), as_u32(h2{h[2], h[3]})};
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < a.N) dst[e] = h[e];
        }
    }
}

template <int BITS, int GROUP, int MT, int NTW, bool BF16, bool SUMS>
int launch_qbatch(BatchArgs a, hipStream_t stream) {
    constexpr int LDS = BatchCfg<MT, NTW>::template lds<GROUP>();
    static_assert(LDS <= 160 * 1024, "the staged x, scales and zero points have to fit LDS twice");
    auto kern = qbatch_kernel<BITS, GROUP, MT, NTW, BF16, SUMS>;
    static uint64_t big_lds_devices = 0;                   // per instantiation
    if (LDS > 64 * 1024 && !bw_allow_big_lds(reinterpret_cast<const void*>(kern), big_lds_devices)) return BW_ELAUNCH;
    a.mtiles = (a.M + 16 * MT - 1) / (16 * MT);
    a.ntiles = (a.N + BatchCfg<MT, NTW>::BN - 1) / BatchCfg<MT, NTW>::BN;
    BW_NOTE_KERNEL("qbatch_kernel", BITS, GROUP, MT, NTW, (int)BF16, (int)SUMS);
    hipLaunchKernelGGL(kern, dim3((unsigned)(a.mtiles * a.ntiles * a.splits)), dim3(512), LDS, stream, a);
    return hipGetLastError() == hipSuccess ? BW_OK : BW_ELAUNCH;
}

template <int BITS>
int launch_qbatch_bits(int group, int mt, int ntw, const BatchArgs& a, hipStream_t stream) {
#define BW_CASE(G, T, W) \
    if (group == G && mt == T && ntw == W) {                                                                                          \
        if constexpr (bw_qbatch_sums(BITS, G, T, W))                                                                                  \
            if (a.sums) return a.x_bf16 ? launch_qbatch<BITS, G, T, W, true, true>(a, stream) : launch_qbatch<BITS, G, T, W, false, true>(a, stream); \
        return a.x_bf16 ? launch_qbatch<BITS, G, T, W, true, false>(a, stream) : launch_qbatch<BITS, G, T, W, false, false>(a, stream);  \
    }
#define BW_ROWS(G, T) BW_CASE(G, T, 1) BW_CASE(G, T, 2) BW_CASE(G, T, 3)
#define BW_WIDE(G) BW_CASE(G, 1, 4) BW_CASE(G, 2, 4) BW_CASE(G, 3, 4) BW_CASE(G, 4, 4)
#define BW_GROUP(G) BW_ROWS(G, 1) BW_ROWS(G, 2) BW_ROWS(G, 3) BW_ROWS(G, 4) BW_CASE(G, 6, 1) BW_CASE(G, 6, 2) BW_CASE(G, 6, 3) BW_CASE(G, 8, 1) BW_CASE(G, 8, 2)
    BW_GROUP(128) BW_GROUP(64) BW_GROUP(32)
    if constexpr (BITS != 8) {                                // (at 8 bits 64-row tiles of them spill 59 ... 135 registers)
        BW_WIDE(128) BW_WIDE(64) BW_WIDE(32)
    }
#undef BW_WIDE
#undef BW_GROUP
#undef BW_ROWS
#undef BW_CASE
    return BW_EUNSUPPORTED;
}

}  // namespace
