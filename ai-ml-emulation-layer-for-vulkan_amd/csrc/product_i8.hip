// int8 MATMUL whose operands lie at any alignment, on the matrix cores: what gemm_i8.hip's fetch modes do not take
// (reference arithmetic: matmul.comp:30-73; RESCALE and CLAMP of the fused form: rescale.comp:27-72, clamp.comp:24-53).
// int32 sums wrap, so the order of the additions is immaterial.
//
// out[m][n] = sum_k X[m][k] * W[k][n], W as [K][N] rows (KM) or as rows of K.  What bounds such a product is the trip to memory,
// not the arithmetic: so every load is 16 bytes wide, from whatever address, and none stands behind a condition (behind one the
// compiler no longer knows how many loads are on their way, and waits for all of them).  Rows beyond the operand are its last
// row; the one stage that reaches beyond K comes first, its addresses moved back inside the operand and its bytes shifted and
// cleared in registers, so that its loads travel together with those of the whole stages behind it.  A K-major W keeps its rows
// in shared memory and is transposed on its way out (ds_read_b64_tr_b8).  With the zero points
//     sum (x - zx) (w - zw) = sum x w - zx sum w - zw sum x + K zx zw,
// the sums of rows taken on the way to shared memory, those of a K-major W's columns from the matrix operands.
// What is left is bound by the loads: 16 bytes from any byte address move at 18 bytes per clock and compute unit (48 from aligned
// ones), and at 10 where a row gives only 32 bytes.
// Against the loop this replaces (a K-major W in conditional dwords, transposed in registers), us: 4095^3 390 -> 130,
// 1000^3 23 -> 7.0, 11 x 15 x 2541 x 1182 54 -> 12.5, 2 x 122 x 2933 x 137 32 -> 9.2, 10 x 2090 x 54 x 430 29 -> 10.6,
// 10 x 63 x 1296 x 46 18.5 -> 5.4.
#include <algorithm>

#include "common.hpp"
#include "dispatch.hpp"

namespace mlel {
namespace {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) v2i lds_v2i;

struct PArgs {
    const char *x, *w;
    char *out;
    int32_t M, N, K, batches;
    int32_t total_tiles, chunk;
    TileOrder order;
    int64_t x_batch, w_batch, o_batch;
    uint32_t ldx, ldw, x_bytes, w_bytes;  // bytes per row, bytes of a batch's operand (at least 16)
    int32_t whole;                        // whole stages in front of the last one
    int32_t zx, zw;
    const char *mult;
    const int8_t *shift;
    int32_t mult16;
    RescaleParams rp;
};

// a piece moved `by` (at most 15) bytes to the front, zeros behind, and its first `rem` bytes kept
__device__ __forceinline__ uint4 forward_keep(uint4 v, uint32_t by, int rem) {
    uint32_t w[5] = {v.x, v.y, v.z, v.w, 0};
    if (by & 4) w[0] = w[1], w[1] = w[2], w[2] = w[3], w[3] = 0;
    if (by & 8) w[0] = w[2], w[1] = w[3], w[2] = w[3] = 0;
    const uint32_t sh = (by & 3) * 8;
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = keep_bytes(__builtin_amdgcn_alignbit(w[i + 1], w[i], sh), rem - 4 * i);
    return make_uint4(w[0], w[1], w[2], w[3]);
}

constexpr int product_stage(int bm, int bn, int bkb, bool km) { return km ? bm * bkb + bkb * (bn + 16) : (bm + bn) * bkb; }
// two stages, or the tile of results
constexpr int product_tile(int bm, int bn, int bkb, bool km, int so) { return std::max(2 * product_stage(bm, bn, bkb, km), bm * (bn * so + 16)); }

// FUSED / SO: RESCALE to one byte, or the int32 sums; BM x BN tile; WM x WN x WK wavefronts over rows, columns and the K of a
// stage of BKB bytes; S register sets: a stage is asked for S stages before it is stored
template <bool FUSED, int BM, int BN, int WM, int WN, int WK, int BKB, int S, bool KM>
__global__ void __launch_bounds__(64 * WM * WN * WK) product_i8_kernel(const PArgs g) {
    constexpr int NT = 64 * WM * WN * WK, SO = FUSED ? 1 : 4;
    constexpr int PPR = BKB / 16, SH = BKB == 64 ? 2 : (BKB == 128 ? 1 : 0);
    constexpr int KKW = BKB / 32 / WK;
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
    constexpr int XI = BM * PPR / NT, WI = BN * PPR / NT;
    constexpr int WPITCH = BN + 16, WCH = BN / 16;  // K-major: pitch of a row of the tile, its pieces
    constexpr int STAGE = product_stage(BM, BN, BKB, KM), TILE = product_tile(BM, BN, BKB, KM, SO);
    static_assert((BM * PPR) % NT == 0 && (BN * PPR) % NT == 0 && KKW >= 1 && TM >= 1 && TN >= 1, "tile shape");
    static_assert((NT / PPR) % 16 == 0 && S % 2 == 0, "the rows of one thread share their swizzle; a set meets one buffer");
    extern __shared__ __align__(16) char smem[];
    int32_t *sums = reinterpret_cast<int32_t *>(smem + TILE);  // [BM] of X, [BN] of W
    struct Scale {
        int64_t pos, neg;
        int32_t mult, shift;
    };
    Scale *scales = reinterpret_cast<Scale *>(smem + TILE + (BM + BN) * 4);  // [BN]

    const int lin = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u));
    if (lin >= g.total_tiles) return;
    int batch, tile_m, tile_n;
    g.order.tile(lin, batch, tile_m, tile_n);
    const int m_base = tile_m * BM, n_base = tile_n * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_k = wave % WK, wave_n = (wave / WK) % WN, wave_m = wave / (WK * WN);
    const char *xp = g.x + (int64_t)batch * g.x_batch, *wp = g.w + (int64_t)batch * g.w_batch;

    // ---- this thread's pieces of a stage
    const int r0 = tid / PPR, p0 = (tid % PPR) ^ ((r0 >> SH) & (PPR - 1));
    uint32_t xo[XI], wo[WI];
#pragma unroll
    for (int i = 0; i < XI; i++) xo[i] = (uint32_t)min(m_base + r0 + i * (NT / PPR), g.M - 1) * g.ldx + (uint32_t)(p0 * 16);
#pragma unroll
    for (int i = 0; i < WI; i++) {
        const int id = i * NT + tid, n = n_base + (id % WCH) * 16;
        wo[i] = KM ? (uint32_t)(id / WCH) * g.ldw + (uint32_t)(n < g.N ? n : n_base)
                   : (uint32_t)min(n_base + r0 + i * (NT / PPR), g.N - 1) * g.ldw + (uint32_t)(p0 * 16);
    }
    struct Set {
        uint4 x[XI], w[WI];
    };
    auto ask = [&](Set &v, int stage) {  // whole stage `stage` (beyond the last one: that one again)
        stage = min(stage, g.whole - 1);
        const char *xa = xp + (int64_t)stage * BKB, *wa = wp + (int64_t)stage * (KM ? (int64_t)BKB * g.ldw : BKB);
#pragma unroll
        for (int i = 0; i < XI; i++) v.x[i] = load_any<16>(xa + xo[i]);
#pragma unroll
        for (int i = 0; i < WI; i++) v.w[i] = load_any<16>(wa + wo[i]);
    };
    // the stage at `k0` that may reach beyond K: loads inside the operand ...
    auto tail_x = [&](int i, int k0) { return xo[i] + (uint32_t)k0; };
    auto tail_w = [&](int i, int k0) {
        if constexpr (KM) return wo[i] + (uint32_t)min(k0, g.K - 1 - (i * NT + tid) / WCH) * g.ldw;  // (a row beyond K is the last one)
        return wo[i] + (uint32_t)k0;
    };
    auto ask_tail = [&](Set &v, int k0) {
#pragma unroll
        for (int i = 0; i < XI; i++) v.x[i] = load_any<16>(xp + min(tail_x(i, k0), g.x_bytes - 16));
#pragma unroll
        for (int i = 0; i < WI; i++) v.w[i] = load_any<16>(wp + min(tail_w(i, k0), g.w_bytes - 16));
    };
    // ... and what of them counts
    auto trim = [&](Set &v, int k0) {
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const uint32_t off = tail_x(i, k0);
            v.x[i] = forward_keep(v.x[i], min(off - min(off, g.x_bytes - 16), 15u), g.K - k0 - p0 * 16);
        }
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const uint32_t off = tail_w(i, k0);
            const int k = k0 + (i * NT + tid) / WCH;
            v.w[i] = forward_keep(v.w[i], min(off - min(off, g.w_bytes - 16), 15u), KM ? (k < g.K ? 16 : 0) : g.K - k0 - p0 * 16);
        }
    };
    const int nk = g.whole;
    int k0 = nk * BKB;
    Set r[S];
    // the scale of one column each, asked for in front of the operands
    static_assert(BN <= NT && BM + BN <= NT, "a thread per column");
    int32_t mu = 0, sh = 0;
    if constexpr (FUSED) {
        const int ch = g.rp.per_channel ? min(n_base + tid, g.N - 1) : 0;
        mu = g.mult16 ? (int32_t) reinterpret_cast<const int16_t *>(g.mult)[ch] : reinterpret_cast<const int32_t *>(g.mult)[ch];
        sh = g.shift[ch];
    }
    ask_tail(r[0], k0);

    v16i acc[TM][TN];
    int32_t xsum[XI], wsum[KM ? TN : WI];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0;
#pragma unroll
    for (int i = 0; i < XI; i++) xsum[i] = 0;
#pragma unroll
    for (int i = 0; i < (KM ? TN : WI); i++) wsum[i] = 0;

    auto store = [&](char *st, const Set &v) {
#pragma unroll
        for (int i = 0; i < XI; i++) {
            *reinterpret_cast<uint4 *>(st + (i * NT + tid) * 16) = v.x[i];
            if (g.zw != 0) xsum[i] = sum_bytes(v.x[i], xsum[i]);  // uniform
        }
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int id = i * NT + tid;
            *reinterpret_cast<uint4 *>(st + BM * BKB + (KM ? (id / WCH) * WPITCH + (id % WCH) * 16 : id * 16)) = v.w[i];
            if constexpr (!KM)
                if (g.zx != 0) wsum[i] = sum_bytes(v.w[i], wsum[i]);  // uniform
        }
    };
    const int h = lane >> 5, lrow = lane & 31;
    // K-major: 16-lane group q holds columns 16 (q & 1) .. of k 16 (q >> 1) ..; its lane s points at row s / 2, half s % 2
    const int tr_off = (h * 16 + ((lane & 15) >> 1)) * WPITCH + ((lane >> 4) & 1) * 16 + (lane & 1) * 8;
    const bool sum_w = KM && g.zx != 0 && wave_m == 0;
    auto compute = [&](const char *st) {
        v4i xf[KKW][TM], wf[KKW][TN];
#pragma unroll
        for (int k = 0; k < KKW; k++) {
            const int kk = wave_k * KKW + k, slot = ((kk * 2 + h) ^ ((lrow >> SH) & (PPR - 1))) * 16;
#pragma unroll
            for (int i = 0; i < TM; i++)
                xf[k][i] = *reinterpret_cast<const v4i *>(st + ((wave_m * TM + i) * 32 + lrow) * BKB + slot);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                if constexpr (KM) {
                    const char *p = st + BM * BKB + kk * 32 * WPITCH + tr_off + (wave_n * TN + j) * 32;
                    const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i *)p);
                    const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i *)(p + 8 * WPITCH));
                    wf[k][j] = v4i{lo.x, lo.y, hi.x, hi.y};
                } else {
                    wf[k][j] = *reinterpret_cast<const v4i *>(st + BM * BKB + ((wave_n * TN + j) * 32 + lrow) * BKB + slot);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < KKW; k++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[k][j], xf[k][i], acc[i][j], 0, 0, 0);
        if constexpr (KM)
            if (sum_w) {  // uniform
#pragma unroll
                for (int k = 0; k < KKW; k++)
#pragma unroll
                    for (int j = 0; j < TN; j++) wsum[j] = sum_bytes(__builtin_bit_cast(uint4, wf[k][j]), wsum[j]);
            }
    };
    // stage 0 is the last one of K, stage q the whole one q - 1; stage q passes through set q % S and buffer q % 2
    auto begin = [&] {
        if (tid < BM + BN) sums[tid] = 0;
        if (FUSED && tid < BN) {
            const ChanScale cs = make_chan_scale(mu, sh, g.rp);
            scales[tid] = Scale{cs.round_pos, cs.round_neg, cs.mult, cs.shift};
        }
        trim(r[0], k0);
        store(smem, r[0]);
    };
    if (nk > 0) {  // uniform
#pragma unroll
        for (int d = 1; d < S; d++) ask(r[d], d - 1);
        begin();
        ask(r[0], S - 1);
        __syncthreads();
        int step = 0;
        for (; step + S <= nk; step += S) {
#pragma unroll
            for (int d = 0; d < S; d++) {
                store(smem + ((d + 1) & 1) * STAGE, r[(d + 1) % S]);
                ask(r[(d + 1) % S], step + d + S);
                compute(smem + (d & 1) * STAGE);
                __syncthreads();
            }
        }
#pragma unroll
        for (int d = 0; d < S; d++) {
            if (step + d <= nk) {  // uniform
                if (step + d < nk) store(smem + ((d + 1) & 1) * STAGE, r[(d + 1) % S]);
                compute(smem + (d & 1) * STAGE);
                __syncthreads();
            }
        }
    } else {
        begin();
        for (;;) {  // K within one stage; rows of W so short that they are not read ahead
            __syncthreads();
            compute(smem);
            __syncthreads();
            k0 += BKB;
            if (k0 >= g.K) break;
            ask_tail(r[0], k0);
            trim(r[0], k0);
            store(smem, r[0]);
        }
    }

    // ---- sums of rows and columns, and the K shares of the wavefronts
    if (g.zw != 0) {
#pragma unroll
        for (int i = 0; i < XI; i++) atomicAdd(&sums[r0 + i * (NT / PPR)], xsum[i]);
    }
    if (g.zx != 0) {
        if constexpr (KM) {
            if (wave_m == 0) {
#pragma unroll
                for (int j = 0; j < TN; j++) atomicAdd(&sums[BM + (wave_n * TN + j) * 32 + lrow], wsum[j]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < WI; i++) atomicAdd(&sums[BM + r0 + i * (NT / PPR)], wsum[i]);
        }
    }
    // A register quad holds four columns of one row.  Wavefronts that share K leave their quads in shared memory, and each of the
    // first four takes an equal part of them (one alone over 112 shares and 16 results: 0.5 us more of a 32 x 32 tile).
    constexpr int NQ = WK == 1 ? 4 * TM * TN : (WK < 4 ? 4 / WK : 1);
    v4u own[NQ];
    if constexpr (WK > 1) {
        static_assert(TM * TN == 1 && WK * BM * BN * 4 <= TILE, "the shares fit the stage buffers");
        v4u *red = reinterpret_cast<v4u *>(smem) + wave / WK * 256 + lane;
#pragma unroll
        for (int q = 0; q < 4; q++)
            red[(wave_k * WM * WN * 4 + q) * 64] =
                v4u{(uint32_t)acc[0][0][4 * q], (uint32_t)acc[0][0][4 * q + 1], (uint32_t)acc[0][0][4 * q + 2], (uint32_t)acc[0][0][4 * q + 3]};
        __syncthreads();
        if (wave_k < 4) {
#pragma unroll
            for (int u = 0; u < NQ; u++) {
                own[u] = red[(wave_k * NQ + u) * 64];
#pragma unroll
                for (int s = 1; s < WK; s++) own[u] += red[(s * WM * WN * 4 + wave_k * NQ + u) * 64];
            }
        }
    } else {
#pragma unroll
        for (int u = 0; u < NQ; u++) {
            const v16i &t = acc[u / (4 * TN)][u / 4 % TN];
            own[u] = v4u{(uint32_t)t[u % 4 * 4], (uint32_t)t[u % 4 * 4 + 1], (uint32_t)t[u % 4 * 4 + 2], (uint32_t)t[u % 4 * 4 + 3]};
        }
    }
    __syncthreads();

    // ---- zero points and RESCALE; the tile goes through shared memory and leaves in runs of a row
    constexpr int OP = BN * SO + 16;
    const uint32_t kzz = (uint32_t)g.K * (uint32_t)g.zx * (uint32_t)g.zw;
    const int32_t hi_v = pin_vgpr(g.rp.out_hi);
    auto finish = [&](auto scale_of) {  // `scale_of(c)`: the scale of column c
#pragma unroll
        for (int u = 0; u < NQ; u++) {
            const int i = u / (4 * TN), j = u / 4 % TN, q = WK == 1 ? u % 4 : wave_k * NQ + u;
            const int row = (wave_m * TM + i) * 32 + lrow, c0 = (wave_n * TN + j) * 32 + 8 * q + 4 * h;
            const uint32_t xs = kzz - (uint32_t)sums[row] * (uint32_t)g.zw;
            uint32_t v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = own[u][e] + xs - (uint32_t)sums[BM + c0 + e] * (uint32_t)g.zx;
                if constexpr (FUSED) {
                    const Scale s = scale_of(c0 + e);
                    v[e] = (uint32_t)requant_acc((int32_t)v[e], ChanScale{s.pos, s.neg, s.mult, s.shift}, g.rp, hi_v);
                }
            }
            if constexpr (FUSED)
                *reinterpret_cast<uint32_t *>(smem + row * OP + c0) = __builtin_amdgcn_perm(
                    __builtin_amdgcn_perm(v[3], v[2], 0x00000400u), __builtin_amdgcn_perm(v[1], v[0], 0x00000400u), 0x05040100u);
            else
                *reinterpret_cast<uint4 *>(smem + row * OP + c0 * 4) = make_uint4(v[0], v[1], v[2], v[3]);
        }
    };
    if (WK == 1 || wave_k < 4) {
        if (FUSED && !g.rp.per_channel) {  // uniform: one scale, in registers
            const Scale one = scales[0];
            finish([&](int) { return one; });
        } else {
            finish([&](int c) { return scales[c]; });
        }
    }
    __syncthreads();
    char *ob = g.out + (int64_t)batch * g.o_batch + (int64_t)n_base * SO;
    const int rows = min(BM, g.M - m_base), bytes = min(BN, g.N - n_base) * SO;
    constexpr int OPPR = BN * SO / 16;
    for (int p = tid; p < BM * OPPR; p += NT) {
        const int row = p / OPPR, c = p % OPPR * 16;
        if (row >= rows || c >= bytes) continue;
        char *dst = ob + (int64_t)(m_base + row) * g.N * SO + c;
        const uint4 v = *reinterpret_cast<const uint4 *>(smem + row * OP + c);
        if (c + 16 <= bytes) {  // through the L2, which joins the lines that rows share (written through: 4095^3 137 us)
            __builtin_memcpy(dst, &v, 16);
        } else {                // the end of a row: halves, while there are bytes of them
            uint4 t = v;
            int left = bytes - c;
            if (left & 8) {
                const uint2 d = make_uint2(t.x, t.y);
                __builtin_memcpy(dst, &d, 8);
                t.x = t.z, t.y = t.w, dst += 8;
            }
            if (left & 4) {
                __builtin_memcpy(dst, &t.x, 4);
                t.x = t.y, dst += 4;
            }
            if (left & 2) {
                const uint16_t d = (uint16_t)t.x;
                __builtin_memcpy(dst, &d, 2);
                t.x >>= 16, dst += 2;
            }
            if (left & 1) *dst = (char)t.x;
        }
    }
}

template <bool FUSED, int BM, int BN, int WM, int WN, int WK, int BKB, int S, bool KM>
int launch_tile(PArgs &g, hipStream_t s) {
    constexpr size_t sm = (size_t)product_tile(BM, BN, BKB, KM, FUSED ? 1 : 4) + (BM + BN) * 4 + BN * 24;
    static_assert(sm <= 160 * 1024 && product_tile(BM, BN, BKB, KM, FUSED ? 1 : 4) % 16 == 0, "shared memory of a compute unit");
    // rows of W shorter than a piece: a piece may reach over several of them, so no stage counts as whole
    g.whole = KM && g.ldw < 16 ? 0 : (g.K - 1) / BKB;
    const int64_t tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
    const int64_t total = tiles_m * tiles_n * g.batches;
    MLEL_REQUIRE(total < (int64_t(1) << 30), MLEL_ERR_LIMIT, "matmul: %lld tiles", (long long)total);
    g.total_tiles = (int)total;
    g.chunk = (int)((total + 7) / 8);
    g.order = make_tile_order(tiles_m, tiles_n, g.chunk, BM, BN);
    auto kernel = product_i8_kernel<FUSED, BM, BN, WM, WN, WK, BKB, S, KM>;
    static const bool raised = sm <= 48 * 1024 || hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm) == hipSuccess;
    (void)raised;
    kernel<<<dim3((unsigned)(g.chunk * 8)), dim3(64 * WM * WN * WK), sm, s>>>(g);
    MLEL_TRY(check_launch("matmul int8, any alignment"));
    return 1;
}

// Tile choice.  128 x 128 from one tile per compute unit on, four wavefronts by two; 64 x 64 from half a tile per compute unit on,
// pairs of wavefronts sharing K; below that 32 x 32, eight of them.  Stages are short (64 and 128 bytes) where several blocks
// share a compute unit and hide each other's ends: 1 x 4095 x 200 x 4095 takes 18 us, with 128 bytes and half as many blocks 24.5.
// The small tile has the unit to itself and takes 256 bytes a stage; more register sets only lengthen the code (eight: 1 us).
template <bool FUSED, bool KM>
int launch_shape(mlel_ctx *ctx, PArgs &g, hipStream_t s) {
    const int64_t cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
    auto tiles = [&](int bm, int bn) { return (int64_t)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn) * g.batches; };
    if (g.M > 64 && g.N > 64 && tiles(128, 128) >= cus) return launch_tile<FUSED, 128, 128, 2, 4, 1, 64, 4, KM>(g, s);
    if (g.N > 32 && tiles(64, 64) * 2 >= cus) return launch_tile<FUSED, 64, 64, 2, 2, 2, 128, 4, KM>(g, s);
    return launch_tile<FUSED, 32, 32, 1, 1, 8, 256, 2, KM>(g, s);
}

constexpr int64_t kLim = (int64_t(1) << 31) - 4096;

}  // namespace

// Returns 1 when launched, 0 to decline.
int try_matmul_i8_ragged(mlel_ctx *ctx, hipStream_t s, const mlel_tensor *out, const mlel_tensor *a, const mlel_tensor *b,
                         const mlel_matmul_attr *attr, const FusedEpilogue *epi) {
    if (a->dtype != MLEL_I8 || b->dtype != MLEL_I8) return 0;
    PArgs g{};
    if (epi == nullptr) {
        if (out->dtype != MLEL_I32 || ((uintptr_t)out->ptr % 4) != 0) return 0;
    } else {
        if (dt_size(out->dtype) != 1 || epi->p.in_zp != 0) return 0;
        g.mult = static_cast<const char *>(epi->mult->ptr);
        g.shift = static_cast<const int8_t *>(epi->shift->ptr);
        g.mult16 = epi->scale32 ? 0 : 1;
        g.rp = epi->p;
    }
    if (attr->a_zp < -128 || attr->a_zp > 127 || attr->b_zp < -128 || attr->b_zp > 127) return 0;
    const int64_t NB = out->dims[0], M = out->dims[1], N = out->dims[2], K = a->dims[2];
    if (NB <= 0 || M <= 0 || N <= 0 || K <= 0 || !is_packed(out)) return 0;
    if (a->dims[0] < NB || b->dims[0] < NB || a->dims[1] < M || b->dims[1] != K || b->dims[2] < N) return 0;
    const bool rows = K > 1 && N > 1 && b->strides[1] == 1 && b->strides[2] >= K;
    if (a->strides[2] != 1 || a->strides[1] < K || (!rows && (b->strides[2] != 1 || b->strides[1] < N))) return 0;
    for (const mlel_tensor *t : {a, b})
        if (t->strides[0] < 0) return 0;
    const int64_t ldw = rows ? b->strides[2] : b->strides[1];
    const int64_t xb = (M - 1) * a->strides[1] + K, wb = ((rows ? N : K) - 1) * ldw + (rows ? K : N);
    // (a stage beyond the end adds up to 256 rows or bytes to an offset before it is moved back)
    if (xb >= kLim || wb >= kLim || xb < 16 || wb < 16 || M * N * 4 >= kLim || NB >= (1 << 20)) return 0;
    g.x = static_cast<const char *>(a->ptr), g.w = static_cast<const char *>(b->ptr), g.out = static_cast<char *>(out->ptr);
    g.M = (int)M, g.N = (int)N, g.K = (int)K, g.batches = (int)NB;
    g.x_batch = a->strides[0], g.w_batch = b->strides[0], g.o_batch = out->strides[0];
    g.ldx = (uint32_t)a->strides[1], g.ldw = (uint32_t)ldw, g.x_bytes = (uint32_t)xb, g.w_bytes = (uint32_t)wb;
    g.zx = attr->a_zp, g.zw = attr->b_zp;
    if (rows) return epi != nullptr ? launch_shape<true, false>(ctx, g, s) : launch_shape<false, false>(ctx, g, s);
    return epi != nullptr ? launch_shape<true, true>(ctx, g, s) : launch_shape<false, true>(ctx, g, s);
}

}  // namespace mlel
