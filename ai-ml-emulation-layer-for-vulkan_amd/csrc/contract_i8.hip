// int8 convolutions whose rows are not made of aligned 16-byte pieces, on the matrix cores: CONV2D with any channel count and
// TRANSPOSE_CONV2D -- what gemm_i8.hip's fetch modes and conv_direct.hip do not take (reference arithmetic: conv2d.comp:40-116,
// transpose_conv2d.comp:31-70; RESCALE and CLAMP of the fused forms: rescale.comp:27-72, clamp.comp:24-53).  int32 sums wrap,
// so the order of the additions is immaterial.
//
// out[m][n] = sum_k X[m][k] * W[n][k].  K is padded per tap: a tap's IC bytes are fetched in chunks of XC bytes (16, or 4
// for few channels) wherever they lie -- the chip loads dwords from any byte address, and a loop over single bytes, which
// this replaces, issues four to sixteen times the loads -- and the tail of a chunk, which holds the neighbouring pixel's
// channels, meets zero weights.  A tap outside the image is the input zero point, so that
//     sum (x - zx) (w - zw) = sum x w - zx sum w - zw sum x + K zx zw
// holds for every position alike; the sums of rows are taken from the pieces on their way to shared memory.
// TRANSPOSE_CONV2D by its phases: the outputs of one remainder class (oy mod sy, ox mod sx) meet the same taps and are a
// convolution of unit stride walking the input backwards; a launch holds the tiles of every phase, none of which
// multiplies the zeros between the input's positions.
// Pieces of 16 bytes sit in shared memory in XOR-swizzled slots as in contract_float.hip.  Registers hold the loads of the
// next two stages while one is multiplied: with a tile or two per compute unit that is what hides the trip to memory.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "dispatch.hpp"

namespace mlel {
namespace {

typedef int v16i __attribute__((ext_vector_type(16)));

struct IArgs {
    const int8_t *x, *x2, *w;           // x2: the second operand of a CONCAT along the channels, or null
    char *out;
    const int32_t *bias;  // or null
    int32_t bias_len;
    int32_t M, N;
    int32_t tiles_m, tiles_n, total_tiles, chunk, tiles_phase;
    DivMagic div_phase, div_tiles_n, div_ohw, div_ow;
    // row m of a phase: image, y', x'; its taps (jy, jx), jy < taps_y, read input row y' * sy + base_y + jy * dy.
    // CONV2D has one phase (phase_y = phase_x = 1); TRANSPOSE_CONV2D has sy x sx, of unit stride and dy = dx = -1
    int32_t IC, IC1, KH, KW, H, W, OHW, OW;  // OHW, OW: positions of a phase per image and per row; IC1: channels of x
    int32_t sy, sx, pt, pl, dy, dx, phase_y, phase_x;
    int32_t out_h, out_w;               // extents of the output image
    uint32_t x_pix, x_bytes, x2_bytes, ldw, w_bytes;  // x_pix: bytes from one position of x to the next
    int32_t zx, zw;
    const char *mult;
    const int8_t *shift;
    int32_t mult16;
    RescaleParams rp;
};

// B bytes at offset `off` of an operand of `bytes` bytes (at least B): a chunk that would reach beyond the end is loaded
// from further in front and shifted down
template <int B>
__device__ __forceinline__ uint4 load_chunk(const int8_t *base, uint32_t off, uint32_t bytes) {
    const uint32_t last = bytes - B;
    if (off <= last) return load_any<B>(base + off);
    const uint32_t by = off - last;  // 1 .. B - 1
    const uint4 v = load_any<B>(base + last);
    if constexpr (B == 4) return make_uint4(v.x >> (8 * by), 0, 0, 0);
    const uint32_t w[8] = {v.x, v.y, v.z, v.w, 0, 0, 0, 0};
    uint32_t r[4];
    const uint32_t d = by / 4, s = 8 * (by % 4);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (d == (uint32_t)j) lo = w[i + j], hi = i + j + 1 < 8 ? w[i + j + 1] : 0;
        r[i] = (uint32_t)((((uint64_t)hi << 32) | lo) >> s);
    }
    return make_uint4(r[0], r[1], r[2], r[3]);
}

// SO: bytes of a result (1: requantised int8 / uint8, 4: the int32 accumulator, or the requantised int32);
// XC: bytes per chunk; DUAL: X is two tensors side by side along the channels
// (CONCAT read in place: a tap's chunks are those of the first tensor, then those of the second)
template <bool FUSED, int SO, int BM, int BN, int WM, int WN, int WK, int BKB, int XC, bool DUAL>
__global__ void __launch_bounds__(64 * WM * WN * WK) contract_i8_kernel(const IArgs g) {
    constexpr int NT = 64 * WM * WN * WK;
    constexpr int PPR = BKB / 16, SH = BKB == 64 ? 2 : (BKB == 128 ? 1 : 0);
    constexpr int KK = BKB / 32, KKW = KK / WK;
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
    constexpr int XI = BM * PPR / NT, STAGE = (BM + BN) * BKB;
    constexpr int WI = (BN * PPR + NT - 1) / NT;  // pieces of W per thread
    static_assert((BM * PPR) % NT == 0 && KK % WK == 0 && TM >= 1 && TN >= 1 && (NT / PPR) % 16 == 0, "tile shape");
    static_assert(BM + BN <= NT, "a thread per sum");
    extern __shared__ __align__(16) char smem[];
    int32_t *sums = reinterpret_cast<int32_t *>(smem + 2 * STAGE);  // [BM] of X, [BN] of W
    struct Scale {
        int64_t pos, neg;
        int32_t mult, shift, bias, pad;
    };
    Scale *scales = reinterpret_cast<Scale *>(smem + 2 * STAGE + (BM + BN) * 4);  // [BN]

    const int lin_all = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u));
    if (lin_all >= g.total_tiles) return;
    const int phase = div_magic(lin_all, g.div_phase), lin = lin_all - phase * g.tiles_phase;
    const int tile_m = div_magic(lin, g.div_tiles_n), tile_n = lin - tile_m * g.tiles_n;
    const int m_base = tile_m * BM, n_base = tile_n * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_k = wave % WK, wave_n = (wave / WK) % WN, wave_m = wave / (WK * WN);

    // ---- the phase's taps: tap (jy, jx) is weight (ky0 + jy * phase_y, kx0 + jx * phase_x)
    const int ry = phase / g.phase_x, rx = phase - ry * g.phase_x;
    int ky0 = 0, kx0 = 0, by = -g.pt, bx = -g.pl, taps_y = g.KH, taps_x = g.KW;
    if (g.phase_y * g.phase_x > 1) {  // uniform; pt, pl: the output padding of TRANSPOSE_CONV2D
        ky0 = (ry - g.pt) % g.phase_y, kx0 = (rx - g.pl) % g.phase_x;
        if (ky0 < 0) ky0 += g.phase_y;
        if (kx0 < 0) kx0 += g.phase_x;
        taps_y = ky0 < g.KH ? (g.KH - 1 - ky0) / g.phase_y + 1 : 0;
        taps_x = kx0 < g.KW ? (g.KW - 1 - kx0) / g.phase_x + 1 : 0;
        by = (ry - g.pt - ky0) / g.phase_y, bx = (rx - g.pl - kx0) / g.phase_x;  // exact divisions
    }
    const int taps = taps_y * taps_x;
    constexpr int CP = 16 / XC;                // chunks per piece
    const int cpt1 = DUAL ? (g.IC1 + XC - 1) / XC : (g.IC + XC - 1) / XC;
    const int cpt = DUAL ? cpt1 + (g.IC - g.IC1 + XC - 1) / XC : cpt1;  // chunks per tap
    const int n_chunks = taps * cpt;
    const int nk = (n_chunks + PPR * CP - 1) / (PPR * CP);

    const int r0 = tid / PPR, p0 = (tid % PPR) ^ ((r0 >> SH) & (PPR - 1));
    int32_t xb[XI], iy0[XI], ix0[XI];  // xb: index of the position the first tap meets
#pragma unroll
    for (int i = 0; i < XI; i++) {
        const int m = m_base + r0 + i * (NT / PPR);
        const int img = div_magic(m, g.div_ohw), pos = m - img * g.OHW;
        const int y = div_magic(pos, g.div_ow), x = pos - y * g.OW;
        iy0[i] = m < g.M ? y * g.sy + by : -0x40000000;
        ix0[i] = x * g.sx + bx;
        xb[i] = (img * g.H + y * g.sy + by) * g.W + ix0[i];
    }
    if (tid < BM + BN) sums[tid] = 0;
    for (int c = tid; c < BN; c += NT) {
        const int n = n_base + c;
        Scale s{};
        if (n < g.N) {
            s.bias = g.bias != nullptr ? g.bias[g.bias_len == 1 ? 0 : n] : 0;
            if (FUSED) {
                const int ch = g.rp.per_channel ? n : 0;
                const int32_t mu = g.mult16 ? (int32_t) reinterpret_cast<const int16_t *>(g.mult)[ch]
                                            : reinterpret_cast<const int32_t *>(g.mult)[ch];
                const ChanScale cs = make_chan_scale(mu, g.shift[ch], g.rp);
                s.pos = cs.round_pos, s.neg = cs.round_neg, s.mult = cs.mult, s.shift = cs.shift;
            }
        }
        scales[c] = s;
    }

    // position along K of this thread's next piece: chunk cq of tap (jy, jx)
    int cq = p0 * CP, jy = 0, jx = 0;
    auto wrap = [&](int &c, int &y, int &x) {
        while (c >= cpt && y < taps_y) {
            c -= cpt;
            if (++x == taps_x) x = 0, y++;
        }
    };
    wrap(cq, jy, jx);
    const uint32_t zx4 = (uint32_t)(uint8_t)g.zx * 0x01010101u;
    // a tap's last chunk holds bytes of its neighbour
    const bool tail = DUAL ? (g.IC1 % XC != 0 || (g.IC - g.IC1) % XC != 0) : g.IC % XC != 0;
    const bool mask_x = tail && g.zw != 0;     // they count only where the weights' zero point does

    v16i acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0;

    // ---- fetch: X pieces and W pieces of the next stage into one of two register sets
    // chunk c of a tap: bytes of it that are channels, and its place among the weights of the tap
    auto remaining = [&](int c) { return DUAL ? (c < cpt1 ? g.IC1 - c * XC : g.IC - g.IC1 - (c - cpt1) * XC) : g.IC - c * XC; };
    auto channel = [&](int c) { return DUAL && c >= cpt1 ? g.IC1 + (c - cpt1) * XC : c * XC; };
    auto load_x = [&](int pix, int c) {
        if (DUAL && c >= cpt1)
            return load_chunk<XC>(g.x2, (uint32_t)pix * (uint32_t)(g.IC - g.IC1) + (uint32_t)((c - cpt1) * XC), g.x2_bytes);
        return load_chunk<XC>(g.x, (uint32_t)pix * g.x_pix + (uint32_t)(c * XC), g.x_bytes);
    };
    auto fetch = [&](uint4(&xr)[XI], uint4(&wr)[WI]) {
        const bool live = jy < taps_y && taps_x > 0;
#pragma unroll
        for (int i = 0; i < XI; i++) {
            if constexpr (XC == 16) {
                const int iy = iy0[i] + jy * g.dy, ix = ix0[i] + jx * g.dx;
                const uint32_t fill = live ? zx4 : 0u;  // (nothing beyond K, where the sums of rows end too)
                uint4 v = make_uint4(fill, fill, fill, fill);
                if (live && (uint32_t)iy < (uint32_t)g.H && (uint32_t)ix < (uint32_t)g.W) {
                    v = load_x(xb[i] + jy * g.dy * g.W + jx * g.dx, cq);
                }
                if (mask_x) {  // uniform
                    const int rem = remaining(cq);
                    v = make_uint4(keep_bytes(v.x, rem), keep_bytes(v.y, rem - 4), keep_bytes(v.z, rem - 8), keep_bytes(v.w, rem - 12));
                }
                xr[i] = v;
            } else {
                uint32_t v[4];
                int c = cq, y = jy, x = jx;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int iy = iy0[i] + y * g.dy, ix = ix0[i] + x * g.dx;
                    v[e] = y < taps_y ? zx4 : 0u;
                    if (y < taps_y && (uint32_t)iy < (uint32_t)g.H && (uint32_t)ix < (uint32_t)g.W)
                        v[e] = load_x(xb[i] + y * g.dy * g.W + x * g.dx, c).x;
                    if (mask_x) v[e] = keep_bytes(v[e], remaining(c));
                    if (++c == cpt) {
                        c = 0;
                        if (++x == taps_x) x = 0, y++;
                    }
                }
                xr[i] = make_uint4(v[0], v[1], v[2], v[3]);
            }
        }
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int r = r0 + i * (NT / PPR), n = n_base + r;
            const bool in = n < g.N && ((BN * PPR) % NT == 0 || r < BN);
            const uint32_t row = (uint32_t)n * g.ldw;
            if constexpr (XC == 16) {
                uint4 v = make_uint4(0, 0, 0, 0);
                if (in && live)
                    v = load_chunk<16>(g.w, row + (uint32_t)(((ky0 + jy * g.phase_y) * g.KW + kx0 + jx * g.phase_x) * g.IC + channel(cq)), g.w_bytes);
                if (tail) {  // uniform
                    const int rem = remaining(cq);
                    v = make_uint4(keep_bytes(v.x, rem), keep_bytes(v.y, rem - 4), keep_bytes(v.z, rem - 8), keep_bytes(v.w, rem - 12));
                }
                wr[i] = v;
            } else {
                uint32_t v[4];
                int c = cq, y = jy, x = jx;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[e] = 0;
                    if (in && y < taps_y)
                        v[e] = load_chunk<4>(g.w, row + (uint32_t)(((ky0 + y * g.phase_y) * g.KW + kx0 + x * g.phase_x) * g.IC + channel(c)), g.w_bytes).x;
                    if (tail) v[e] = keep_bytes(v[e], remaining(c));
                    if (++c == cpt) {
                        c = 0;
                        if (++x == taps_x) x = 0, y++;
                    }
                }
                wr[i] = make_uint4(v[0], v[1], v[2], v[3]);
            }
        }
        cq += PPR * CP;
        wrap(cq, jy, jx);
    };
    int32_t xsum[XI], wsum[WI];
#pragma unroll
    for (int i = 0; i < XI; i++) xsum[i] = 0;
#pragma unroll
    for (int i = 0; i < WI; i++) wsum[i] = 0;
    auto store = [&](char *st, const uint4(&xr)[XI], const uint4(&wr)[WI]) {
#pragma unroll
        for (int i = 0; i < XI; i++) {
            *reinterpret_cast<uint4 *>(st + (i * NT + tid) * 16) = xr[i];
            if (g.zw != 0) xsum[i] = sum_bytes(xr[i], xsum[i]);  // uniform
        }
#pragma unroll
        for (int i = 0; i < WI; i++) {
            if ((BN * PPR) % NT == 0 || i * NT + tid < BN * PPR)
                *reinterpret_cast<uint4 *>(st + BM * BKB + (i * NT + tid) * 16) = wr[i];
            if (g.zx != 0) wsum[i] = sum_bytes(wr[i], wsum[i]);  // uniform
        }
    };
    const int h = lane >> 5, lrow = lane & 31;
    auto compute = [&](const char *st) {
#pragma unroll
        for (int k = 0; k < KKW; k++) {
            const int slot = (((wave_k * KKW + k) * 2 + h) ^ ((lrow >> SH) & (PPR - 1))) * 16;
            v4i xf[TM], wf[TN];
#pragma unroll
            for (int i = 0; i < TM; i++)
                xf[i] = *reinterpret_cast<const v4i *>(st + ((wave_m * TM + i) * 32 + lrow) * BKB + slot);
#pragma unroll
            for (int j = 0; j < TN; j++)
                wf[j] = *reinterpret_cast<const v4i *>(st + BM * BKB + ((wave_n * TN + j) * 32 + lrow) * BKB + slot);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[j], xf[i], acc[i][j], 0, 0, 0);
        }
    };
    uint4 x0[XI], w0[WI], x1[XI], w1[WI];
    if (nk > 0) {
        fetch(x0, w0);
        if (nk > 1) fetch(x1, w1);
        store(smem, x0, w0);
        if (nk > 2) fetch(x0, w0);
        __syncthreads();
        for (int step = 0; step < nk; step += 2) {  // two register sets, two stage buffers: set s & 1 holds stage s
            if (step + 1 < nk) store(smem + STAGE, x1, w1);
            if (step + 3 < nk) fetch(x1, w1);
            compute(smem);
            __syncthreads();
            if (step + 1 < nk) {  // uniform
                if (step + 2 < nk) store(smem, x0, w0);
                if (step + 4 < nk) fetch(x0, w0);
                compute(smem + STAGE);
                __syncthreads();
            }
        }
    } else {
        __syncthreads();
    }

    // ---- sums of rows, and the K shares of the wavefronts
    if (g.zw != 0) {
#pragma unroll
        for (int i = 0; i < XI; i++) atomicAdd(&sums[r0 + i * (NT / PPR)], xsum[i]);
    }
    if (g.zx != 0) {
#pragma unroll
        for (int i = 0; i < WI; i++) {
            if ((BN * PPR) % NT == 0 || i * NT + tid < BN * PPR) atomicAdd(&sums[BM + r0 + i * (NT / PPR)], wsum[i]);
        }
    }
    if constexpr (WK > 1) {
        int32_t *red = reinterpret_cast<int32_t *>(smem);
        static_assert((WK - 1) * BM * BN * 4 <= 2 * STAGE, "the shares fit the stage buffers");
        if (wave_k > 0) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        red[((((wave_k - 1) * WM * WN + wave / WK) * TM * TN + i * TN + j) * 16 + r) * 64 + lane] = acc[i][j][r];
        }
        __syncthreads();
        if (wave_k == 0) {
#pragma unroll
            for (int s = 0; s < WK - 1; s++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int r = 0; r < 16; r++)
                            acc[i][j][r] = (int32_t)((uint32_t)acc[i][j][r] +
                                                     (uint32_t)red[(((s * WM * WN + wave / WK) * TM * TN + i * TN + j) * 16 + r) * 64 + lane]);
        }
    }
    __syncthreads();

    // ---- zero points, bias, RESCALE; the tile goes through shared memory and leaves in runs of a row
    constexpr int OP = BN * SO + 16;
    char *ob = g.out;
    // a tile that holds whole rows of a dense result is one run of memory: it is laid down without gaps and leaves in
    // 16-byte pieces whatever N is (m_base is a multiple of 32)
    const bool dense = g.phase_y * g.phase_x == 1 && g.tiles_n == 1 && (g.N * SO) % 16 != 0 && ((uintptr_t)ob % 16) == 0;
    const uint32_t kzz = (uint32_t)(taps * g.IC) * (uint32_t)g.zx * (uint32_t)g.zw;
    const int32_t hi_v = pin_vgpr(g.rp.out_hi);
    if (WK == 1 || wave_k == 0) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int row = (wave_m * TM + i) * 32 + lrow;
            const uint32_t xs = (uint32_t)sums[row] * (uint32_t)g.zw;
            char *orow = smem + row * (dense ? g.N * SO : OP);
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    uint32_t v[4];
                    const int c0 = (wave_n * TN + j) * 32 + 8 * q + 4 * h;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const Scale &s = scales[c0 + e];
                        const uint32_t a = (uint32_t)acc[i][j][4 * q + e] + (uint32_t)s.bias + kzz - xs -
                                           (uint32_t)sums[BM + c0 + e] * (uint32_t)g.zx;
                        if constexpr (FUSED)
                            v[e] = (uint32_t)requant_acc((int32_t)a, ChanScale{s.pos, s.neg, s.mult, s.shift}, g.rp, hi_v);
                        else
                            v[e] = a;
                    }
                    if (dense && g.N % 4 != 0) {  // uniform
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            if (c0 + e >= g.N) continue;
                            if constexpr (SO == 1) orow[c0 + e] = (char)v[e];
                            else *reinterpret_cast<uint32_t *>(orow + (c0 + e) * 4) = v[e];
                        }
                        continue;
                    }
                    if (dense && c0 >= g.N) continue;
                    if constexpr (SO == 1)
                        *reinterpret_cast<uint32_t *>(orow + c0) =
                            __builtin_amdgcn_perm(__builtin_amdgcn_perm(v[3], v[2], 0x00000400u),
                                                  __builtin_amdgcn_perm(v[1], v[0], 0x00000400u), 0x05040100u);
                    else
                        *reinterpret_cast<uint4 *>(orow + c0 * 4) = make_uint4(v[0], v[1], v[2], v[3]);
                }
        }
    }
    __syncthreads();
    if (dense) {  // uniform
        const int bytes = min(BM, g.M - m_base) * g.N * SO;
        char *run = ob + (int64_t)m_base * g.N * SO;
        for (int p = tid * 16; p < bytes; p += NT * 16) {
            if (p + 16 <= bytes)
                store16_result(run + p, *reinterpret_cast<const uint4 *>(smem + p));
            else
                for (int e = p; e < bytes; e++) run[e] = smem[e];
        }
        return;
    }
    // byte offset of row m of the phase; false for a position outside the image
    auto out_row = [&](int r, int64_t &off) {
        const int m = m_base + r;
        if (m >= g.M) return false;
        if (g.phase_y * g.phase_x == 1) {  // uniform
            off = (int64_t)m * g.N * SO;
            return true;
        }
        const int img = div_magic(m, g.div_ohw), pos = m - img * g.OHW;
        const int y = div_magic(pos, g.div_ow), x = pos - y * g.OW;
        const int oy = y * g.phase_y + ry, ox = x * g.phase_x + rx;
        off = (((int64_t)img * g.out_h + oy) * g.out_w + ox) * g.N * SO;
        return oy < g.out_h && ox < g.out_w;
    };
    const int cols = min(BN, g.N - n_base);
    if ((g.N * SO) % 16 == 0 && ((uintptr_t)ob % 16) == 0) {  // uniform
        constexpr int OPPR = BN * SO / 16;
        for (int p = tid; p < BM * OPPR; p += NT) {
            const int r = p / OPPR, c = p % OPPR;
            int64_t off;
            if (c * 16 >= cols * SO || !out_row(r, off)) continue;
            store16_result(ob + off + (int64_t)n_base * SO + c * 16, *reinterpret_cast<const uint4 *>(smem + r * OP + c * 16));
        }
    } else if ((g.N * SO) % 4 == 0 && ((uintptr_t)ob % 4) == 0) {  // uniform
        constexpr int OPPR = BN * SO / 4;
        for (int p = tid; p < BM * OPPR; p += NT) {
            const int r = p / OPPR, c = p % OPPR;
            int64_t off;
            if (c * 4 >= cols * SO || !out_row(r, off)) continue;
            *reinterpret_cast<uint32_t *>(ob + off + (int64_t)n_base * SO + c * 4) = *reinterpret_cast<const uint32_t *>(smem + r * OP + c * 4);
        }
    } else {
        for (int p = tid; p < BM * BN; p += NT) {
            const int r = p / BN, c = p % BN;
            int64_t off;
            if (c >= cols || !out_row(r, off)) continue;
            ob[off + n_base + c] = smem[r * OP + c];  // (SO == 4 rows are whole dwords)
        }
    }
}

template <bool FUSED, int SO, int BM, int BN, int WM, int WN, int WK, int BKB, int XC, bool DUAL>
int launch_tile(IArgs &g, hipStream_t s) {
    constexpr size_t operands = (size_t)2 * (BM + BN) * BKB, result = (size_t)BM * (BN * SO + 16);
    constexpr size_t sm = operands + (BM + BN) * 4 + BN * 32;
    static_assert(result <= operands && sm <= 64 * 1024 && operands % 16 == 0 && (BM + BN) % 4 == 0, "shared memory");
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    const int64_t per_phase = (int64_t)g.tiles_m * g.tiles_n, total = per_phase * g.phase_y * g.phase_x;
    MLEL_REQUIRE(total < (int64_t(1) << 30), MLEL_ERR_LIMIT, "contraction: %lld tiles", (long long)total);
    g.tiles_phase = (int)per_phase;
    g.total_tiles = (int)total;
    g.chunk = (int)((total + 7) / 8);
    g.div_phase = make_div_magic((uint32_t)per_phase);
    g.div_tiles_n = make_div_magic((uint32_t)g.tiles_n);
    auto kernel = contract_i8_kernel<FUSED, SO, BM, BN, WM, WN, WK, BKB, XC, DUAL>;
    static const bool raised = sm <= 48 * 1024 || hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm) == hipSuccess;
    (void)raised;
    kernel<<<dim3((unsigned)(g.chunk * 8)), dim3(64 * WM * WN * WK), sm, s>>>(g);
    MLEL_TRY(check_launch("int8 contraction, ragged rows"));
    return 1;
}

// Tile choice: 32 columns when N fits them, else 64; from half a tile per compute unit on four wavefronts share the rows,
// below that they share K over a 32 x 32 tile.
template <bool FUSED, int SO, int XC, bool DUAL>
int launch_shape(mlel_ctx *ctx, IArgs &g, hipStream_t s) {
    const int64_t cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
    const int64_t phases = (int64_t)g.phase_y * g.phase_x;
    auto tiles = [&](int bm, int bn) { return (int64_t)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn) * phases; };
    if (g.N <= 32 && tiles(128, 32) * 2 >= cus) return launch_tile<FUSED, SO, 128, 32, 4, 1, 1, 128, XC, DUAL>(g, s);
    if (g.N > 32 && tiles(64, 64) * 2 >= cus) return launch_tile<FUSED, SO, 64, 64, 2, 2, 1, 128, XC, DUAL>(g, s);
    return launch_tile<FUSED, SO, 32, 32, 1, 1, 4, 256, XC, DUAL>(g, s);
}

template <int XC>
int launch_out(mlel_ctx *ctx, IArgs &g, bool fused, hipStream_t s) {
    if (g.x2 != nullptr) return launch_shape<true, 1, XC, true>(ctx, g, s);
    return fused ? launch_shape<true, 1, XC, false>(ctx, g, s) : launch_shape<false, 4, XC, false>(ctx, g, s);
}

constexpr int64_t kLim = (int64_t(1) << 31) - 4096;

bool fill_epilogue(IArgs &g, const mlel_tensor *out, const FusedEpilogue *epi) {
    if (epi == nullptr) return out->dtype == MLEL_I32 && ((uintptr_t)out->ptr % 4) == 0;
    if (dt_size(out->dtype) != 1 || epi->p.in_zp != 0) return false;
    g.mult = static_cast<const char *>(epi->mult->ptr);
    g.shift = static_cast<const int8_t *>(epi->shift->ptr);
    g.mult16 = epi->scale32 ? 0 : 1;
    g.rp = epi->p;
    return true;
}

// CONV2D (over `in`, or over `in` and `in2` side by side along the channels) or TRANSPOSE_CONV2D; `probe`: judge types and
// extents only
int try_conv(mlel_ctx *ctx, hipStream_t s, const mlel_tensor *out, const mlel_tensor *in, const mlel_tensor *in2,
             const mlel_tensor *w, const mlel_tensor *bias, const FusedEpilogue *epi, uint32_t acc_type, int32_t zx, int32_t zw,
             const int32_t *pad, const int32_t *stride, const int32_t *dilation, bool transposed, bool probe) {
    if (in->dtype != MLEL_I8 || w->dtype != MLEL_I8 || bias->dtype != MLEL_I32 || acc_type != MLEL_ACC_I32) return 0;
    IArgs g{};
    if (probe ? dt_size(out->dtype) != 1 : !fill_epilogue(g, out, epi)) return 0;
    if (zx < -128 || zx > 127 || zw < -128 || zw > 127) return 0;
    if (!is_packed(in) || !is_packed(w) || !is_packed(out) || !is_packed(bias)) return 0;
    const int64_t N = in->dims[0], H = in->dims[1], W = in->dims[2], IC1 = in->dims[3], IC = IC1 + (in2 ? in2->dims[3] : 0);
    if (in2 != nullptr && (in2->dtype != MLEL_I8 || !is_packed(in2) || in2->dims[0] != N || in2->dims[1] != H || in2->dims[2] != W ||
                           epi == nullptr || in2->dims[3] <= 0 || N * H * W * in2->dims[3] < 16))
        return 0;
    const int64_t OC = w->dims[0], KH = w->dims[1], KW = w->dims[2], OH = out->dims[1], OW = out->dims[2], small = 1 << 20;
    if (w->dims[3] != IC || out->dims[0] != N || out->dims[3] != OC) return 0;
    if (N <= 0 || H <= 0 || W <= 0 || IC1 <= 0 || OC <= 0 || KH <= 0 || KW <= 0 || OH <= 0 || OW <= 0) return 0;
    if (bias->dims[0] != 1 && bias->dims[0] < OC) return 0;
    if (N * H * W * IC >= kLim || OC * KH * KW * IC >= kLim || N * H * W * IC1 < 16 || OC * KH * KW * IC < 16) return 0;
    if (N * OH * OW >= (int64_t(1) << 30) || H >= small || W >= small || OH >= small || OW >= small || KH >= 4096 || KW >= 4096) return 0;
    for (int i = 0; i < 2; i++)
        if (stride[i] <= 0 || stride[i] >= 1024 || dilation[i] <= 0 || dilation[i] >= 1024) return 0;
    for (int i = 0; i < 4; i++)
        if (pad[i] < -small || pad[i] > small) return 0;
    if (probe) return 1;
    const int few = try_conv_few_i8(ctx, s, out, in, in2, w, bias, epi, zx, zw, pad, stride, dilation, transposed);
    if (few != 0) return few;
    const int taken = try_conv_patch_i8(ctx, s, out, in, in2, w, bias, epi, zx, zw, pad, stride, dilation, transposed);
    if (taken != 0) return taken;
    g.x = static_cast<const int8_t *>(in->ptr), g.w = static_cast<const int8_t *>(w->ptr);
    if (in2 != nullptr) g.x2 = static_cast<const int8_t *>(in2->ptr), g.x2_bytes = (uint32_t)(N * H * W * in2->dims[3]);
    g.out = static_cast<char *>(out->ptr), g.bias = static_cast<const int32_t *>(bias->ptr), g.bias_len = (int)bias->dims[0];
    g.N = (int)OC;
    g.IC = (int)IC, g.IC1 = (int)IC1, g.KH = (int)KH, g.KW = (int)KW, g.H = (int)H, g.W = (int)W;
    g.pt = pad[0], g.pl = pad[2];
    g.out_h = (int)OH, g.out_w = (int)OW;
    int64_t ph = OH, pw = OW;
    if (transposed) {
        g.phase_y = stride[0], g.phase_x = stride[1], g.sy = g.sx = 1, g.dy = g.dx = -1;
        ph = (OH + stride[0] - 1) / stride[0], pw = (OW + stride[1] - 1) / stride[1];
    } else {
        g.phase_y = g.phase_x = 1, g.sy = stride[0], g.sx = stride[1], g.dy = dilation[0], g.dx = dilation[1];
    }
    g.M = (int)(N * ph * pw), g.OHW = (int)(ph * pw), g.OW = (int)pw;
    g.div_ohw = make_div_magic((uint32_t)g.OHW), g.div_ow = make_div_magic((uint32_t)g.OW);
    g.x_pix = (uint32_t)IC1;
    g.x_bytes = (uint32_t)(N * H * W * IC1), g.ldw = (uint32_t)(KH * KW * IC), g.w_bytes = (uint32_t)(OC * KH * KW * IC);
    g.zx = zx, g.zw = zw;
    // chunks of 16 bytes where they waste less than a quarter of the loads' width, dwords for fewer channels
    const auto fetched = [&](int64_t c) { return (IC1 + c - 1) / c * c + (IC - IC1 + c - 1) / c * c; };
    const bool wide = fetched(16) * 4 <= fetched(4) * 5;
    return wide ? launch_out<16>(ctx, g, epi != nullptr, s) : launch_out<4>(ctx, g, epi != nullptr, s);
}

}  // namespace

int try_conv2d_i8_ragged(mlel_ctx *ctx, hipStream_t s, const mlel_tensor *out, const mlel_tensor *in, const mlel_tensor *w,
                         const mlel_tensor *bias, const mlel_conv2d_attr *a, const FusedEpilogue *epi, const mlel_tensor *in2,
                         bool probe) {
    return try_conv(ctx, s, out, in, in2, w, bias, epi, a->acc_type, a->input_zp, a->weight_zp, a->pad, a->stride, a->dilation,
                    false, probe);
}

int try_tconv2d_i8(mlel_ctx *ctx, hipStream_t s, const mlel_tensor *out, const mlel_tensor *in, const mlel_tensor *w,
                   const mlel_tensor *bias, const mlel_tconv2d_attr *a, const FusedEpilogue *epi, bool probe) {
    const int32_t unit[2] = {1, 1};
    return try_conv(ctx, s, out, in, nullptr, w, bias, epi, a->acc_type, a->input_zp, a->weight_zp, a->out_pad, a->stride, unit,
                    true, probe);
}

}  // namespace mlel
