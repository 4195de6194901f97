// int8 CONV2D (+RESCALE +CLAMP) with a kernel of a few taps, over one image or two side by side along the channels (CONCAT
// read in place), and TRANSPOSE_CONV2D whose kernel is its stride: the block keeps its piece of the image in shared memory
// (reference arithmetic: conv2d.comp:40-116, transpose_conv2d.comp:31-70, rescale.comp:27-72, clamp.comp:24-53).
//
// The kernels that walk K in stages fetch every input byte once per tap, and for channel counts that are no multiple of 16
// each fetch is a handful of vector instructions: at 24 + 24 channels and nine taps they issued 32 dword loads per row and
// stage.  Here a block owns TH x TW output positions: the (TH - 1) stride + (KH - 1) dilation + 1 rows of the image they
// meet are fetched once, in the widest chunks the channel count allows, with the input zero point outside the image; the
// weights of the block's 32 NJ channels are fetched once per block.  All taps are then multiplied straight from shared
// memory without a barrier, a lane's operand being 16 bytes of one pixel ("piece"): a pixel is padded to an odd number of
// pieces, so that the lanes of a 128-bit read, neighbouring pixels, meet distinct banks.
//   K runs over the pieces of all taps in pairs, one piece per half of the wavefront (v_mfma_i32_32x32x32_i8); a pair may
//   straddle two taps, so only an odd total of pieces is padded.
//   NARROW (up to 8 channels, unit dilation): a pixel is 4 or 8 bytes and the taps of a kernel row are consecutive bytes,
//   so a piece holds several taps.
// The first matrix operand is X: a lane ends up with 16 positions of one channel, whose requantisation constants sit in
// registers.  The results leave through shared memory as the runs of whole pixels they are in the result.
// Two kernels.  In the first a block walks several tiles (the weights stay), with the next tile's pixels in registers while one
// is multiplied; it takes any channel count.  In the second (channels and weights in whole dwords) a block has one tile: the
// weights go straight to shared memory and nothing is kept from tile to tile, which leaves a third of the instructions and
// registers out; try_conv_patch_i8 has the figures of both.
// A TRANSPOSE_CONV2D whose kernel equals its stride meets one input position per output: it is a 1 x 1 convolution to
// sx * OC channels per output row phase, whose results are contiguous in the output row.
//
// Measured (360 x 640; the staged kernel, the first, the second): 24 + 24 -> 24 channels 3 x 3: 75, 15.6, 11.6 us; 3 -> 24: 25.6, 8.5 (the
// first only); 1 x 1 24 -> 19: 19, 8.3, 7.2; at half that size 96 -> 48: 12.9 and 10.3.  Bound by the vector and scalar instructions:
// 24 -> 24 channels, 904 blocks: 1003 vector and 522 scalar instructions per wavefront in the first, 666 and 461 in the second (11.4 ->
// 9.7 us), of which the requantisation is 270, and by the chain of one block: arguments, the way of the patch, 9 steps, results.
#include <algorithm>

#include "common.hpp"
#include "dispatch.hpp"

namespace mlel {
namespace {

typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kBlock = 256;
constexpr int kChunks = 8;  // chunks of the image per thread

struct PatchArgs {
    const int8_t *x, *x2, *w;
    int8_t *out;
    const int32_t *bias;
    const char *mult;
    const int8_t *shift;
    int32_t mult16, bias_len;
    RescaleParams rp;
    // image: H x W pixels of IC (= IC1 + IC2) bytes; x2: channels IC1 ..
    int32_t H, W, IC, IC1;
    uint32_t x_bytes, x2_bytes, w_bytes;
    int32_t sy, sx, dy, dx, pt, pl;
    // result: OH x OW positions of N bytes; position row y of phase p is row y * phases + p of the output image
    int32_t OH, OW, N, phases, KW, split;
    int32_t w_row;  // taps of a channel's weights; split: a result pixel holds N / split kernel columns (TRANSPOSE_CONV2D), else N
    // tile and patch
    int32_t log_tw, TH, PH, PW, pitch, patch_bytes;
    int32_t cpp[2], n_chunks[2], per_thread[2];  // chunks per pixel, per patch and per thread (at most) of x and of x2
    // the kernel without a loop: a patch row of x and of x2 in chunks and columns of 64 chunks; a wavefront takes `rows` rows at a
    // time (several where they are short), `turns` times
    int32_t row_chunks[2], columns[2], rows[2], turns[2];
    int32_t steps4, tap_bytes, row_bytes;  // steps, rounded up to a multiple of four; a tap and a row of taps in the patch
    int32_t ppt, taps_x, step_tap, step_row, pieces, steps;  // pieces of K: ppt per tap
    int32_t narrow_p;                                       // NARROW: bytes of a pixel in shared memory
    int32_t n_blocks, blocks, chunk, groups;  // groups: blocks (tiles, without the loop) per (phase, channel block)
    int32_t tiles_part, tiles_rest;           // tiles of a block; the first tiles_rest blocks have one more
    int32_t tiles_x, tiles_y;
    DivMagic div_taps, div_group, div_nb, div_tx, div_ty, div_pieces, div_ppt, div_split, div_run;
    uint32_t mul_cpp[2], mul_pw, mul_row[2];  // see quotient()
    int32_t stage_row;   // bytes of a staged run: tw * columns, rounded up to 16
    int32_t zx;
};

// n / d for n < 2^11 and n d < 2^20, `m` = 2^20 / d + 1: two full-rate instructions
__device__ __forceinline__ int quotient(int n, uint32_t m) { return (int)(__umul24((uint32_t)n, m) >> 20); }
// four bytes at offset `off` of an operand of `bytes` (at least 4): near the end from further in front, shifted down; what
// lies beyond the end is any value
__device__ __forceinline__ uint32_t load_dword(const int8_t *base, uint32_t off, uint32_t bytes) {
    const uint32_t at = min(off, bytes - 4);
    return load_any<4>(base + at).x >> (8 * (off - at) & 31);
}

// Blocks whose registers fit a compute unit.
constexpr int blocks_per_cu(int unit, int nj, int tm) { return nj * tm == 1 ? 4 : (nj * tm == 2 ? (unit == 16 ? 3 : 4) : 2); }

// U: bytes per chunk of the image; NJ: groups of 32 channels of a block; TM: groups of 32 positions per wavefront
template <int U, int NJ, int TM, bool NARROW, bool DUAL>
__global__ void __launch_bounds__(kBlock, blocks_per_cu(U, NJ, TM)) conv_patch_i8_kernel(const PatchArgs g) {
    extern __shared__ __align__(16) char smem[];
    constexpr int BN = 32 * NJ;
    constexpr int WP = (BN + 1) * 16;  // bytes of a piece of all channels: neighbouring pieces start four banks apart
    char *wl = smem + g.patch_bytes;   // [2 steps][WP]
    int32_t *wsum = reinterpret_cast<int32_t *>(wl + g.steps * 2 * WP);  // [BN] sums of the weights
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    char *stage = reinterpret_cast<char *>(wsum + BN) + wave * (32 * BN + 64);  // this wavefront's 32 positions on their way out

    const int lin = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u));
    if (lin >= g.blocks) return;
    const int pn = div_magic(lin, g.div_group), part = lin - pn * g.groups;
    const int phase = div_magic(pn, g.div_nb), n_base = (pn - phase * g.n_blocks) * BN;
    const int first = part * g.tiles_part + min(part, g.tiles_rest), last = first + g.tiles_part + (part < g.tiles_rest ? 1 : 0);
    const int cols = min(BN, g.N - n_base);

    // ---- this thread's chunks of a patch: those of x, then those of x2
    int32_t goff[kChunks], at[kChunks];  // at: row, column and place in shared memory (in dwords) of the patch, or -1
    const int c2 = g.IC - g.IC1;
#pragma unroll
    for (int i = 0; i < kChunks; i++) {
        goff[i] = 0, at[i] = -1;
        const int second = DUAL && i >= g.per_thread[0] ? 1 : 0;  // (uniform, like the break)
        if (i >= g.per_thread[0] + (DUAL ? g.per_thread[1] : 0)) break;
        const int id = (i - second * g.per_thread[0]) * kBlock + tid;
        const int pix = quotient(id, g.mul_cpp[second]), c = id - (int)__umul24(pix, g.cpp[second]);
        const int py = quotient(pix, g.mul_pw), px = pix - (int)__umul24(py, g.PW);
        const int place = (int)__umul24(pix, g.pitch) + c * U + second * g.IC1;  // below 64 KiB
        if (id < g.n_chunks[second]) at[i] = (py << 22) | (px << 14) | (place >> 2);
        goff[i] = (py * g.W + px) * (second ? c2 : g.IC1) + c * U;
    }
    const uint32_t zx4 = (uint32_t)(uint8_t)g.zx * 0x01010101u;
    uint4 pre[kChunks];
    auto tile_at = [&](int t, int &img, int &oy, int &ox) {
        const int ty = div_magic(t, g.div_tx);
        img = div_magic(ty, g.div_ty);
        oy = (ty - img * g.tiles_y) * g.TH;
        ox = (t - ty * g.tiles_x) << g.log_tw;
    };
    auto fetch = [&](int t) {
        int img, oy, ox;
        tile_at(t, img, oy, ox);
        const int iy = oy * g.sy - g.pt, ix = ox * g.sx - g.pl, pix0 = (img * g.H + iy) * g.W + ix;
#pragma unroll
        for (int i = 0; i < kChunks; i++) {
            const bool second = DUAL && i >= g.per_thread[0];
            if (i >= g.per_thread[0] + (DUAL ? g.per_thread[1] : 0)) break;
            pre[i] = make_uint4(zx4, zx4, zx4, zx4);
            int d = at[i];
            asm volatile("" : "+v"(d));  // (unpacked here, not kept unpacked from tile to tile)
            const int y = iy + (d >> 22), x = ix + ((d >> 14) & 0xff);
            if (d >= 0 && (uint32_t)y < (uint32_t)g.H && (uint32_t)x < (uint32_t)g.W) {
                const int8_t *base = second ? g.x2 : g.x;
                const uint32_t off = (uint32_t)(pix0 * (second ? c2 : g.IC1) + goff[i]);
                if constexpr (U == 4) pre[i].x = load_dword(base, off, second ? g.x2_bytes : g.x_bytes);
                else pre[i] = load_any<U>(base + off);
            }
        }
    };
    if (first < last) fetch(first);
    if (tid < BN) wsum[tid] = 0;
    __syncthreads();

    // ---- constants of this lane's channels
    const int h = lane >> 5, lrow = lane & 31;
    int32_t mult[NJ], shift[NJ], bias[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int n = min(n_base + j * 32 + lrow, g.N - 1);
        const int oc = n - div_magic(n, g.div_split) * g.split;
        const int ch = g.rp.per_channel ? oc : 0;
        mult[j] = g.mult16 ? (int32_t) reinterpret_cast<const int16_t *>(g.mult)[ch] : reinterpret_cast<const int32_t *>(g.mult)[ch];
        shift[j] = (int32_t)g.shift[ch];
        bias[j] = g.bias[g.bias_len == 1 ? 0 : oc];
    }

    // ---- weights of the block's channels, once
    // (a channel's pieces are consecutive bytes, so consecutive threads take consecutive pieces; every load of a round is on
    // its way before the first is used)
    const int items = g.steps * 2 * BN, n_pieces = g.steps * 2;
    for (int id0 = tid; id0 < items; id0 += 4 * kBlock) {
        uint32_t v[4][4], off[4];
        int dst[4], piece[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int id = min(id0 + k * kBlock, items - 1), c = div_magic(id, g.div_pieces), j = id - c * n_pieces, n = n_base + c;
            const int kx0 = div_magic(n, g.div_split), oc = n - kx0 * g.split;  // kx0: 0 unless TRANSPOSE_CONV2D
            const int tap = div_magic(j, g.div_ppt);
            dst[k] = j * WP + c * 16;
            piece[k] = j < g.pieces && n < g.N ? j - tap * g.ppt : 0x4000000;
            off[k] = n < g.N ? (uint32_t)((oc * g.w_row + (NARROW ? tap * g.KW : phase * g.KW + kx0 + tap)) * g.IC) : 0u;
            if constexpr (NARROW) {  // a "tap" is a kernel row of KW taps
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const int at = (piece[k] * 16 + d * 4) & 0xff, kx = at >> (g.narrow_p == 8 ? 3 : 2), ch = at & (g.narrow_p - 1);
                    v[k][d] = load_dword(g.w, off[k] + (uint32_t)(kx * g.IC + ch), g.w_bytes);
                }
            } else {
                off[k] += (uint32_t)(piece[k] & 0xff) * 16;
                const uint4 u = load_any<16>(g.w + min(off[k], g.w_bytes - 16));
                v[k][0] = u.x, v[k][1] = u.y, v[k][2] = u.z, v[k][3] = u.w;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (id0 + k * kBlock >= items) break;
            if (!NARROW && off[k] > g.w_bytes - 16) {  // the operand's last bytes: again, dword by dword
#pragma unroll
                for (int d = 0; d < 4; d++) v[k][d] = load_dword(g.w, off[k] + d * 4, g.w_bytes);
            }
            int32_t sum = 0;
#pragma unroll
            for (int d = 0; d < 4; d++) {
                const int at = piece[k] * 16 + d * 4;
                if constexpr (NARROW) {
                    const int kx = at >> (g.narrow_p == 8 ? 3 : 2), ch = at & (g.narrow_p - 1);
                    v[k][d] = kx < g.KW ? keep_bytes(v[k][d], g.IC - ch) : 0u;
                } else {
                    v[k][d] = keep_bytes(v[k][d], g.IC - at);
                }
                sum = __builtin_amdgcn_sdot4((int)v[k][d], 0x01010101, sum, false);
            }
            *reinterpret_cast<uint4 *>(wl + dst[k]) = make_uint4(v[k][0], v[k][1], v[k][2], v[k][3]);
            atomicAdd(reinterpret_cast<int32_t *>(wsum) + (dst[k] % WP) / 16, sum);
        }
    }

    ChanScale cs[NJ];
    int32_t start[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) cs[j] = make_chan_scale(mult[j], shift[j], g.rp);
    const int32_t hi_v = pin_vgpr(g.rp.out_hi);
    // shared-memory address of this lane's positions
    int32_t pos[TM];
#pragma unroll
    for (int t = 0; t < TM; t++) {
        const int m = (wave * TM + t) * 32 + lrow, y = m >> g.log_tw, x = m & ((1 << g.log_tw) - 1);
        pos[t] = (y * g.sy * g.PW + x * g.sx) * g.pitch;
    }
    const char *wlane = wl + h * WP + lrow * 16;

    for (int t = first; t < last; t++) {
#pragma unroll
        for (int i = 0; i < kChunks; i++) {
            if (i >= g.per_thread[0] + (DUAL ? g.per_thread[1] : 0)) break;  // uniform
            int d = at[i];
            asm volatile("" : "+v"(d));
            if (d >= 0) __builtin_memcpy(__builtin_assume_aligned(smem + (d & 0x3fff) * 4, U), &pre[i], U);
        }
        __syncthreads();
        if (t + 1 < last) fetch(t + 1);
        if (t == first) {  // uniform
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                start[j] = (int32_t)((uint32_t)bias[j] - (uint32_t)g.zx * (uint32_t)wsum[j * 32 + lrow]);
            }
        }

        v16i acc[TM][NJ];
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = start[j];
        // the piece of either half of the wavefront, advanced on the scalar unit
        int o = 0, p = 0, kx = 0;
        auto advance = [&]() {
            o += 16;
            if (++p == g.ppt) {
                p = 0;
                o += g.step_tap;
                if (++kx == g.taps_x) {
                    kx = 0;
                    o += g.step_row;
                }
            }
        };
        struct Operands {
            v4i w[NJ], x[TM];
        };
        auto read = [&](Operands &f, int s) {
            const int o0 = o;
            advance();
            const int o1 = o;
            advance();
            const int off = h ? o1 : o0;
#pragma unroll
            for (int j = 0; j < NJ; j++) f.w[j] = *reinterpret_cast<const v4i *>(wlane + s * (2 * WP) + j * 512);
#pragma unroll
            for (int i = 0; i < TM; i++) {
                if constexpr (NARROW) __builtin_memcpy(&f.x[i], __builtin_assume_aligned(smem + pos[i] + off, 4), 16);
                else f.x[i] = *reinterpret_cast<const v4i *>(smem + pos[i] + off);
            }
        };
        auto multiply = [&](const Operands &f) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.x[i], f.w[j], acc[i][j], 0, 0, 0);
        };
        if constexpr (NJ * TM == 1) {
            // one product per step: the operands of the next step are on their way while this one's are multiplied
            Operands fa, fb;
            read(fa, 0);
            for (int s = 0; s < g.steps; s += 2) {
                if (s + 1 < g.steps) read(fb, s + 1);
                multiply(fa);
                if (s + 2 < g.steps) read(fa, s + 2);
                if (s + 1 < g.steps) multiply(fb);
            }
        } else {
            for (int s = 0; s < g.steps; s++) {
                Operands f;
                read(f, s);
                multiply(f);
            }
        }
        __syncthreads();  // the patch has been read

        // ---- requantise; 32 positions at a time through this wavefront's staging rows
        int img, oy0, ox0;
        tile_at(t, img, oy0, ox0);
        const int tw = 1 << g.log_tw, rs = min(g.log_tw, 5), run_pos = 1 << rs, runs = 32 >> rs;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            // position m = 8 (r / 4) + 4 h + r % 4 of the 32: run m >> rs (it starts at a multiple of 16 bytes), of at least
            // eight positions, so that h moves the position inside its run
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int c = j * 32 + lrow;
                char *at = stage + 4 * h * cols + c;
                if (c < cols) {
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int m = 8 * (r >> 2) + (r & 3);
                        at[(m >> rs) * g.stage_row + (m & (run_pos - 1)) * cols] = (char)requant_acc(acc[i][j][r], cs[j], g.rp, hi_v);
                    }
                }
            }
            // a wavefront's own rows: its shared-memory accesses complete in order
            __builtin_amdgcn_wave_barrier();
            const int m0 = (wave * TM + i) * 32;
            if (g.n_blocks == 1) {  // uniform: a run is contiguous in the result
                const int per_run = g.stage_row >> 4;
                for (int q = lane; q < runs * per_run; q += 64) {
                    const int run = div_magic(q, g.div_run), at = (q - run * per_run) * 16;
                    const int m = m0 + run * run_pos, y = oy0 + (m >> g.log_tw), x = ox0 + (m & (tw - 1));
                    const int bytes = y < g.OH ? min(run_pos, g.OW - x) * cols : 0;
                    if (at >= bytes) continue;
                    int8_t *dst = g.out + ((int64_t)((img * g.OH + y) * g.phases + phase) * g.OW + x) * g.N + at;
                    const char *src = stage + run * g.stage_row + at;
                    if (at + 16 <= bytes)
                        store16_result(dst, *reinterpret_cast<const uint4 *>(src));
                    else
                        for (int e = 0; e < bytes - at; e++) dst[e] = (int8_t)src[e];
                }
            } else {
                for (int q = lane; q < 32 * 2 * NJ; q += 64) {  // 16-byte pieces of a position's `cols` bytes
                    const int m = q / (2 * NJ), at = (q % (2 * NJ)) * 16, run = m >> rs;
                    const int y = oy0 + ((m0 + m) >> g.log_tw), x = ox0 + ((m0 + m) & (tw - 1));
                    if (at >= cols || y >= g.OH || x >= g.OW) continue;
                    int8_t *dst = g.out + ((int64_t)((img * g.OH + y) * g.phases + phase) * g.OW + x) * g.N + n_base + at;
                    const char *src = stage + run * g.stage_row + (m & (run_pos - 1)) * cols + at;
                    if (at + 16 <= cols) {
                        uint4 v;
                        __builtin_memcpy(&v, src, 16);
                        store16_result(dst, v);
                    } else {
                        for (int e = 0; e < cols - at; e++) dst[e] = (int8_t)src[e];
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

constexpr uint32_t kFar = 0x40000000u;  // beyond any operand; twice that still is

// 16 bytes per lane from a buffer resource (zeros beyond its extent, dword by dword) straight to shared memory: lane i's
// land at lds_addr + 16 i.  The compiler does not count it among the outstanding loads.
__device__ __forceinline__ void load16_to_lds(v4i res, uint32_t lds_addr, uint32_t offset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds_addr), "v"(offset), "s"(res)
                 : "memory");
}

// The same for channels that are a multiple of four and weights at a multiple of four bytes: the weights go straight to
// shared memory, a block of NW wavefronts has one tile.
template <int U, int NJ, int TM, int NW, bool DUAL>
__global__ void __launch_bounds__(64 * NW, NJ * TM == 1 || U < 16 ? 4 : 3) conv_patch_direct_i8_kernel(const PatchArgs g) {
    extern __shared__ __align__(16) char smem[];
    constexpr int BN = 32 * NJ, WP = BN * 16;  // WP: bytes of a piece of all channels
    char *wl = smem + g.patch_bytes;           // [2 steps][WP]
    int32_t *wsum = reinterpret_cast<int32_t *>(wl + g.steps * 2 * WP);  // [BN][2 NW] sums of a wavefront's pieces of the weights
    int32_t *offs = wsum + BN * 2 * NW;  // [2][steps4] where a half's piece of a step lies behind a position
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    char *stage = reinterpret_cast<char *>(offs + 2 * g.steps4) + wave * (32 * BN + 64);  // this wavefront's 32 positions on their way out

    // the arguments in one batch: left alone the compiler loads them where they are used, a trip to memory each time
    asm volatile("" ::"s"(g.chunk), "s"(g.blocks), "s"(g.div_group.m), "s"(g.div_group.s), "s"(g.n_blocks), "s"(g.groups),
                 "s"(g.div_nb.m), "s"(g.div_nb.s), "s"(g.div_tx.m), "s"(g.div_tx.s), "s"(g.div_ty.m), "s"(g.div_ty.s),
                 "s"(g.tiles_x), "s"(g.tiles_y), "s"(g.TH), "s"(g.log_tw), "s"(g.N), "s"(g.div_split.m), "s"(g.div_split.s),
                 "s"(g.split), "s"(g.w_row), "s"(g.KW), "s"(g.IC), "s"(g.w), "s"(g.w_bytes), "s"(g.ppt), "s"(g.div_ppt.m),
                 "s"(g.div_ppt.s), "s"(g.pieces), "s"(g.steps));
    asm volatile("" ::"s"(g.mult), "s"(g.shift), "s"(g.bias), "s"(g.mult16), "s"(g.bias_len), "s"(g.rp.per_channel), "s"(g.x),
                 "s"(g.IC1), "s"(g.sy), "s"(g.sx), "s"(g.pt), "s"(g.pl), "s"(g.H), "s"(g.W), "s"(g.PH), "s"(g.PW), "s"(g.pitch),
                 "s"(g.cpp[0]), "s"(g.row_chunks[0]), "s"(g.columns[0]), "s"(g.rows[0]), "s"(g.turns[0]), "s"(g.mul_cpp[0]),
                 "s"(g.mul_row[0]), "s"(g.zx));
    const int lin = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u));
    if (lin >= g.blocks) return;
    // A channel block's tiles one after the other.  (A tile's channel blocks one after the other share its patch in the L2, but write
    // the same lines of the result at the same time.  TRANSPOSE_CONV2D 8 -> 68, 2 x 2, six images of 100 x 54: 19.8 us that way, 11.1 this
    // way; over 800 such sizes 4 % slower on average.)
    const int pn = div_magic(lin, g.div_group), t = lin - pn * g.groups;
    const int phase = div_magic(pn, g.div_nb), n_base = (pn - phase * g.n_blocks) * BN;
    const int ty = div_magic(t, g.div_tx), img = div_magic(ty, g.div_ty);
    const int oy0 = (ty - img * g.tiles_y) * g.TH, ox0 = (t - ty * g.tiles_x) << g.log_tw;
    const int cols = min(BN, g.N - n_base), h = lane >> 5, lrow = lane & 31;

    // ---- the weights: a wavefront's 64 lanes fill 64 consecutive slots of 16 bytes, which are one piece of 64 channels or two
    // pieces of 32.  A piece's bytes beyond its tap are the next tap's: they meet zeros of the patch.
    {
        const int n = n_base + (NJ == 1 ? lrow : lane);
        const int kx0 = div_magic(n, g.div_split), oc = n - kx0 * g.split;  // kx0: 0 unless TRANSPOSE_CONV2D
        const uint32_t row = n < g.N ? (uint32_t)((oc * g.w_row + phase * g.KW + kx0) * g.IC) : kFar;
        const uint64_t wa = reinterpret_cast<uint64_t>(g.w);
        const v4i wres = {(int)(uint32_t)wa, (int)((uint32_t)(wa >> 32) & 0xffffu), (int)g.w_bytes, 0x00020000};
        const uint32_t dst = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)wl);
        auto place = [&](int j) {
            const int tap = div_magic(j, g.div_ppt);
            return j < g.pieces ? (uint32_t)(tap * g.IC + (j - tap * g.ppt) * 16) : kFar;
        };
        for (int i = wave; i < g.steps * NJ; i += NW) {  // uniform
            if constexpr (NJ == 1) {
                const uint32_t o0 = place(2 * i), o1 = place(2 * i + 1);
                load16_to_lds(wres, dst + (uint32_t)i * 1024u, row + (h ? o1 : o0));
            } else {
                load16_to_lds(wres, dst + (uint32_t)i * 1024u, row + place(i));
            }
        }
    }

    // ---- constants of this lane's channels
    int32_t mult[NJ], shift[NJ], bias[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int n = min(n_base + j * 32 + lrow, g.N - 1);
        const int oc = n - div_magic(n, g.div_split) * g.split;
        const int ch = g.rp.per_channel ? oc : 0;
        mult[j] = g.mult16 ? (int32_t) reinterpret_cast<const int16_t *>(g.mult)[ch] : reinterpret_cast<const int32_t *>(g.mult)[ch];
        shift[j] = (int32_t)g.shift[ch];
        bias[j] = g.bias[g.bias_len == 1 ? 0 : oc];
    }

    // ---- the patch: a wavefront takes whole rows of it, 64 chunks at a time.  Where a lane's chunk lies in its row is found once
    // per column of 64, the rest is uniform; two columns of four rows of either operand are on their way at a time.
    {
        const int c2 = g.IC - g.IC1;
        const uint32_t zx4 = (uint32_t)(uint8_t)g.zx * 0x01010101u;
        const int iy = oy0 * g.sy - g.pt, ix = ox0 * g.sx - g.pl, pix0 = (img * g.H + iy) * g.W + ix;
        // a patch that lies in the image: nothing to decide per chunk
        const bool inside = iy >= 0 && ix >= 0 && iy + g.PH <= g.H && ix + g.PW <= g.W;
        struct Chunks {
            uint4 v[2][4];
            int32_t to[2], row_in[2];
        };
        auto fetch = [&](Chunks &p, int second, int col0, int turn0) {
            const int ch = second ? c2 : g.IC1;
            const int row0 = (turn0 * (NW) + wave) * g.rows[second], step = NW * g.rows[second];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (k > 0 && col0 + k >= g.columns[second]) break;  // uniform
                int q = (col0 + k) * 64 + lane, row_in = quotient(q, g.mul_row[second]);
                q -= (int)__umul24(row_in, g.row_chunks[second]);
                const int px = quotient(q, g.mul_cpp[second]), at = (q - (int)__umul24(px, g.cpp[second])) * U;
                const uint32_t off = (uint32_t)((row_in * g.W + px) * ch + at);
                p.to[k] = (int)__umul24((int)__umul24(row0 + row_in, g.PW) + px, g.pitch) + at + second * g.IC1;
                if (row_in >= g.rows[second] || q >= g.row_chunks[second]) row_in = 1 << 20;
                p.row_in[k] = row_in;
                const int8_t *from = (second ? g.x2 : g.x) + (int64_t)(pix0 + row0 * g.W) * ch;
                const bool x_in = (uint32_t)(ix + px) < (uint32_t)g.W;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int row = row0 + u * step;
                    if (u > 0 && row >= g.PH) break;  // uniform
                    if (inside) {                     // uniform
                        if (row_in < g.PH - row) p.v[k][u] = load_any<U>(from + off);
                    } else {
                        p.v[k][u] = make_uint4(zx4, zx4, zx4, zx4);
                        if (row_in < g.PH - row && x_in && (uint32_t)(iy + row + row_in) < (uint32_t)g.H) p.v[k][u] = load_any<U>(from + (int32_t)off);
                    }
                    from += step * g.W * ch;
                }
            }
        };
        auto store = [&](const Chunks &p, int second, int col0, int turn0) {
            const int row0 = (turn0 * (NW) + wave) * g.rows[second], step = NW * g.rows[second];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (k > 0 && col0 + k >= g.columns[second]) break;
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int row = row0 + u * step;
                    if (u > 0 && row >= g.PH) break;
                    if (p.row_in[k] < g.PH - row)
                        __builtin_memcpy(__builtin_assume_aligned(smem + p.to[k] + u * step * g.PW * g.pitch, U), &p.v[k][u], U);
                }
            }
        };
        Chunks a, b;
        fetch(a, 0, 0, 0);
        if constexpr (DUAL) fetch(b, 1, 0, 0);
        store(a, 0, 0, 0);
        if constexpr (DUAL) store(b, 1, 0, 0);
        for (int second = 0; second < (DUAL ? 2 : 1); second++)  // what a large patch has beyond that
            for (int c0 = 0; c0 < g.columns[second]; c0 += 2)
                for (int t0 = c0 == 0 ? 4 : 0; t0 < g.turns[second]; t0 += 4) fetch(a, second, c0, t0), store(a, second, c0, t0);
    }
    // zeros between a pixel's channels and the next piece, which the products read
    for (int pix = tid; pix < g.PH * g.PW && g.ppt * 16 != g.IC; pix += 64 * NW)
        for (int c = g.IC; c < g.ppt * 16; c += 4) *reinterpret_cast<uint32_t *>(smem + pix * g.pitch + c) = 0u;
    for (int j = tid; j < g.pieces; j += 64 * NW) {
        const int tap = div_magic(j, g.div_ppt), ky = div_magic(tap, g.div_taps);
        offs[(j & 1) * g.steps4 + (j >> 1)] = ky * g.row_bytes + (tap - ky * g.taps_x) * g.tap_bytes + (j - tap * g.ppt) * 16;
    }
    if (tid == 0 && (g.pieces & 1)) offs[g.steps4 + g.steps - 1] = 0;  // (multiplied by zeros)
    {
        // the weights are there: each wavefront adds up what it brought (dwords beyond a tap left out)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        int32_t sum = 0;
        const int tail = g.ppt * 4 - g.IC / 4;  // dwords of a tap's last piece that are not its own
        for (int i = wave; i < g.steps * NJ; i += NW) {  // uniform
            const uint4 v = *reinterpret_cast<const uint4 *>(wl + i * 1024 + lane * 16);
            const int j = NJ == 1 ? 2 * i + h : i;
            const int own = j + 1 == (div_magic(j, g.div_ppt) + 1) * g.ppt ? 4 - tail : 4;
            sum = __builtin_amdgcn_sdot4((int)v.x, 0x01010101, sum, false);
            sum = __builtin_amdgcn_sdot4((int)v.y, own > 1 ? 0x01010101 : 0, sum, false);
            sum = __builtin_amdgcn_sdot4((int)v.z, own > 2 ? 0x01010101 : 0, sum, false);
            sum = __builtin_amdgcn_sdot4((int)v.w, own > 3 ? 0x01010101 : 0, sum, false);
        }
        wsum[NJ == 1 ? lrow * (2 * NW) + wave * 2 + h : lane * NW + wave] = sum;
    }
    // shared-memory address of this lane's positions
    int32_t pos[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = (wave * TM + i) * 32 + lrow, y = m >> g.log_tw, x = m & ((1 << g.log_tw) - 1);
        pos[i] = (y * g.sy * g.PW + x * g.sx) * g.pitch;
    }
    __syncthreads();

    v16i acc[TM][NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int4 *p = reinterpret_cast<const int4 *>(wsum + (j * 32 + lrow) * (NJ == 1 ? 2 * NW : NW));
        int32_t sum = 0;
#pragma unroll
        for (int e = 0; e < (NJ == 1 ? 2 * NW : NW) / 4; e++) {
            const int4 v = p[e];
            sum += v.x + v.y + v.z + v.w;
        }
        const int32_t start = (int32_t)((uint32_t)bias[j] - (uint32_t)g.zx * (uint32_t)sum);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = start;
    }
    {
        struct Operands {
            v4i w[NJ], x[TM];
        };
        auto read = [&](Operands &f, const char *w, int off) {
#pragma unroll
            for (int j = 0; j < NJ; j++) f.w[j] = *reinterpret_cast<const v4i *>(w + j * 512);
#pragma unroll
            for (int i = 0; i < TM; i++) f.x[i] = *reinterpret_cast<const v4i *>(smem + pos[i] + off);
        };
        auto multiply = [&](const Operands &f) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.x[i], f.w[j], acc[i][j], 0, 0, 0);
        };
        const int32_t *o = offs + h * g.steps4;
        const char *w = wl + h * WP + lrow * 16;
        int s = 0;
        for (; s + 4 <= g.steps; s += 4, o += 4, w += 8 * WP) {
            const int4 off = *reinterpret_cast<const int4 *>(o);
            Operands f[2];
            read(f[0], w, off.x), read(f[1], w + 2 * WP, off.y);
            multiply(f[0]), multiply(f[1]);
            read(f[0], w + 4 * WP, off.z), read(f[1], w + 6 * WP, off.w);
            multiply(f[0]), multiply(f[1]);
        }
        for (; s < g.steps; s++, o++, w += 2 * WP) {
            Operands f;
            read(f, w, *o);
            multiply(f);
        }
    }

    // ---- requantise; 32 positions at a time through this wavefront's staging rows
    const int32_t hi_v = pin_vgpr(g.rp.out_hi);
    const int tw = 1 << g.log_tw, rs = min(g.log_tw, 5), run_pos = 1 << rs, runs = 32 >> rs;
    ChanScale cs[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) cs[j] = make_chan_scale(mult[j], shift[j], g.rp);
#pragma unroll
    for (int i = 0; i < TM; i++) {
        // position m = 8 (r / 4) + 4 h + r % 4 of the 32: run m >> rs (it starts at a multiple of 16 bytes), of at least
        // eight positions, so that 4 h + r % 4 moves the position inside its run
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int c = j * 32 + lrow;
            char *at = stage + 4 * h * cols + c;
            if (c < cols) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    char *row = at + ((8 * q) >> rs) * g.stage_row + ((8 * q) & (run_pos - 1)) * cols;
#pragma unroll
                    for (int e = 0; e < 4; e++) row[e * cols] = (char)requant_acc(acc[i][j][4 * q + e], cs[j], g.rp, hi_v);
                }
            }
        }
        // a wavefront's own rows: its shared-memory accesses complete in order
        __builtin_amdgcn_wave_barrier();
        const int m0 = (wave * TM + i) * 32;
        if (g.n_blocks == 1) {  // uniform: a run is contiguous in the result
            const int per_run = g.stage_row >> 4;
            for (int q = lane; q < runs * per_run; q += 64) {
                const int run = div_magic(q, g.div_run), at = (q - run * per_run) * 16;
                const int m = m0 + run * run_pos, y = oy0 + (m >> g.log_tw), x = ox0 + (m & (tw - 1));
                const int bytes = y < g.OH ? min(run_pos, g.OW - x) * cols : 0;
                if (at >= bytes) continue;
                int8_t *dst = g.out + ((int64_t)((img * g.OH + y) * g.phases + phase) * g.OW + x) * g.N + at;
                const char *src = stage + run * g.stage_row + at;
                if (at + 16 <= bytes)
                    store16_result(dst, *reinterpret_cast<const uint4 *>(src));
                else
                    for (int e = 0; e < bytes - at; e++) dst[e] = (int8_t)src[e];
            }
        } else {
            for (int q = lane; q < 32 * 2 * NJ; q += 64) {  // 16-byte pieces of a position's `cols` bytes
                const int m = q / (2 * NJ), at = (q % (2 * NJ)) * 16, run = m >> rs;
                const int y = oy0 + ((m0 + m) >> g.log_tw), x = ox0 + ((m0 + m) & (tw - 1));
                if (at >= cols || y >= g.OH || x >= g.OW) continue;
                int8_t *dst = g.out + ((int64_t)((img * g.OH + y) * g.phases + phase) * g.OW + x) * g.N + n_base + at;
                const char *src = stage + run * g.stage_row + (m & (run_pos - 1)) * cols + at;
                if (at + 16 <= cols) {
                    uint4 v;
                    __builtin_memcpy(&v, src, 16);
                    store16_result(dst, v);
                } else {
                    for (int e = 0; e < cols - at; e++) dst[e] = (int8_t)src[e];
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

template <int U, int NJ, int TM, bool NARROW, bool DUAL>
int launch_kernel(const PatchArgs &g, size_t sm, hipStream_t s) {
    auto kernel = conv_patch_i8_kernel<U, NJ, TM, NARROW, DUAL>;
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   160 * 1024) == hipSuccess;
    (void)raised;
    kernel<<<dim3((unsigned)(g.chunk * 8)), dim3(kBlock), sm, s>>>(g);
    MLEL_TRY(check_launch("conv2d int8, image pieces in shared memory"));
    return 1;
}
template <int NJ, int TM, bool NARROW>
int launch_unit(const PatchArgs &g, int unit, bool dual, size_t sm, hipStream_t s) {
    if constexpr (NARROW) {
        return launch_kernel<4, NJ, TM, true, false>(g, sm, s);
    } else {
        if (dual) {
            if (unit == 16) return launch_kernel<16, NJ, TM, false, true>(g, sm, s);
            if (unit == 8) return launch_kernel<8, NJ, TM, false, true>(g, sm, s);
            return launch_kernel<4, NJ, TM, false, true>(g, sm, s);
        }
        if (unit == 16) return launch_kernel<16, NJ, TM, false, false>(g, sm, s);
        if (unit == 8) return launch_kernel<8, NJ, TM, false, false>(g, sm, s);
        return launch_kernel<4, NJ, TM, false, false>(g, sm, s);
    }
}
template <int U, int NJ, int TM, int NW, bool DUAL>
int launch_direct_unit(const PatchArgs &g, size_t sm, hipStream_t s) {
    auto kernel = conv_patch_direct_i8_kernel<U, NJ, TM, NW, DUAL>;
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   160 * 1024) == hipSuccess;
    (void)raised;
    kernel<<<dim3((unsigned)(g.chunk * 8)), dim3(64 * NW), sm, s>>>(g);
    MLEL_TRY(check_launch("conv2d int8, image pieces in shared memory"));
    return 1;
}
template <int NJ, int TM, int NW>
int launch_direct(const PatchArgs &g, int unit, bool dual, size_t sm, hipStream_t s) {
    if (dual) {
        if (unit == 16) return launch_direct_unit<16, NJ, TM, NW, true>(g, sm, s);
        return unit == 8 ? launch_direct_unit<8, NJ, TM, NW, true>(g, sm, s) : launch_direct_unit<4, NJ, TM, NW, true>(g, sm, s);
    }
    if (unit == 16) return launch_direct_unit<16, NJ, TM, NW, false>(g, sm, s);
    return unit == 8 ? launch_direct_unit<8, NJ, TM, NW, false>(g, sm, s) : launch_direct_unit<4, NJ, TM, NW, false>(g, sm, s);
}

}  // namespace

// The operands are checked by the caller (contract_i8.hip): packed int8 tensors whose extents in bytes fit 31 bits, an
// epilogue to 8 bits.  `transposed`: TRANSPOSE_CONV2D, `pad` its output padding.  0: not a case for this kernel.
int try_conv_patch_i8(mlel_ctx *ctx, hipStream_t s, const mlel_tensor *out, const mlel_tensor *in, const mlel_tensor *in2,
                      const mlel_tensor *w, const mlel_tensor *bias, const FusedEpilogue *epi, int32_t zx, int32_t zw,
                      const int32_t *pad, const int32_t *stride, const int32_t *dilation, bool transposed) {
    if (epi == nullptr || zw != 0 || dt_size(out->dtype) != 1) return 0;
    const int64_t B = in->dims[0], H = in->dims[1], W = in->dims[2], IC1 = in->dims[3], IC = IC1 + (in2 ? in2->dims[3] : 0);
    const int64_t OC = w->dims[0], KH = w->dims[1], KW = w->dims[2];
    PatchArgs g{};
    g.sy = g.sx = g.dy = g.dx = g.phases = 1;
    g.KW = (int)KW, g.w_row = (int)(KH * KW);
    int64_t N = OC, OH = out->dims[1], OW = out->dims[2], kh = KH, kw = KW;
    if (transposed) {
        if (KH != stride[0] || KW != stride[1] || pad[0] != 0 || pad[1] != 0 || pad[2] != 0 || pad[3] != 0 || OH != H * KH || OW != W * KW)
            return 0;
        g.phases = (int)KH;
        N = OC * KW, OH = H, OW = W, kh = kw = 1;
    } else {
        g.sy = stride[0], g.sx = stride[1], g.dy = dilation[0], g.dx = dilation[1], g.pt = pad[0], g.pl = pad[2];
        if (pad[0] < 0 || pad[2] < 0) return 0;
    }
    // what the kernel was written for: kernels and strides of a few, channels whose weights fit beside a patch
    if (kh > 7 || kw > 7 || g.sy > 3 || g.sx > 3 || g.dy > 2 || g.dx > 2 || IC > 256 || N > 4096 || B * H * W >= (1 << 28)) return 0;
    g.split = (int)OC;
    if (!transposed) g.split = (int)N;
    const bool narrow = IC <= 8 && in2 == nullptr && kw > 1 && g.dx == 1;
    // the widest chunk that divides a pixel's channels; dwords (the last one partly a neighbour's) for the rest
    int unit = 4;
    if (in2 != nullptr && (IC1 % 4 != 0 || (IC - IC1) % 4 != 0)) return 0;
    for (int u : {16, 8})
        if (unit == 4 && !narrow && IC1 % u == 0 && (IC - IC1) % u == 0) unit = u;
    if (OC * KH * KW * IC < 16 || B * H * W * IC1 < 4) return 0;
    g.cpp[0] = (int)((IC1 + unit - 1) / unit), g.cpp[1] = (int)((IC - IC1 + unit - 1) / unit);
    const auto per_thread = [&](int64_t pixels, int which) { return (pixels * g.cpp[which] + kBlock - 1) / kBlock; };
    if (narrow) {
        g.narrow_p = g.pitch = IC <= 4 ? 4 : 8;
        g.ppt = (int)((kw * g.pitch + 15) / 16);
        g.taps_x = 1;
        g.pieces = (int)(kh * g.ppt);
    } else {
        g.ppt = (int)((IC + 15) / 16);
        g.pitch = 16 * (g.ppt | 1);
        g.taps_x = (int)kw;
        g.pieces = (int)(kh * kw * g.ppt);
    }
    g.steps = (g.pieces + 1) / 2, g.steps4 = (g.steps + 3) / 4 * 4;
    g.div_taps = make_div_magic((uint32_t)g.taps_x);
    const int64_t cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
    const int64_t positions = B * OH * OW;
    // the kernel without a loop, its wavefronts per block, channels per block / 32 and positions per wavefront / 32
    bool direct = false;
    int nw = 4, nj = 1, tm = 1;
    size_t sm = 0;
    // how often a wavefront of the kernel without a loop asks for two columns of four rows of the patch and waits for them: a patch
    // that is wide and low takes as many trips to memory in a row (1 x 1, 108 -> 16 channels at 101 x 188, batch 11, in tiles of 64 x 2:
    // 14 of them, 27 us; as before, 13)
    const auto fetches = [&](int64_t ph, int64_t pw, int which) {
        const int64_t row = std::max<int64_t>(1, pw * g.cpp[which]), turn = nw * std::max<int64_t>(1, 64 / row);
        return ((row + 63) / 64 + 1) / 2 * (((ph + turn - 1) / turn + 3) / 4);
    };
    // the tile: the shape of its positions with the least padding, then the smallest patch; false: none whose shared memory
    // leaves room for two blocks on a compute unit
    const auto choose = [&]() {
        int64_t best = -1, best_patch = 0;
        for (int lt = 3; lt <= 6; lt++) {
            const int64_t tw = int64_t(1) << lt, th = 32 * nw * tm / tw;
            const int64_t ph = (th - 1) * g.sy + (kh - 1) * g.dy + 1, pw = (tw - 1) * g.sx + (kw - 1) * g.dx + 1;
            const int64_t area = ((OH + th - 1) / th) * ((OW + tw - 1) / tw);
            const int64_t patch = ph * pw;
            if (ph > 511 || pw > 255 || patch * g.pitch > 65536) continue;  // what a thread's chunk descriptors hold
            if (per_thread(patch, 0) + per_thread(patch, 1) > kChunks * nw / (direct && unit == 4 ? 2 : 4)) continue;
            if (direct && std::max(fetches(ph, pw, 0), fetches(ph, pw, 1)) > 3) continue;
            if (best >= 0 && (area > best || (area == best && patch >= best_patch))) continue;
            best = area, best_patch = patch;
            g.log_tw = lt, g.TH = (int)th, g.PH = (int)ph, g.PW = (int)pw;
        }
        if (best < 0) return false;
        const int bn = 32 * nj;
        // slack: an odd number of pieces, and NARROW's whole pieces, read a little beyond the patch
        const int64_t slack = (int64_t)g.PW * g.dy * g.pitch + (int64_t)g.pitch * (g.dx + 1) + 64;
        g.patch_bytes = (int)((g.PH * g.PW * (int64_t)g.pitch + slack + 15) / 16 * 16);
        sm = (size_t)g.patch_bytes + nw * (32 * bn + 64) +
             (direct ? (size_t)g.steps * bn * 32 + bn * 8 * nw + g.steps4 * 8 : (size_t)g.steps * 2 * (bn + 1) * 16 + bn * 4);
        const int tw = 1 << g.log_tw;
        g.n_blocks = (int)((N + bn - 1) / bn);
        g.tiles_x = (int)((OW + tw - 1) / tw), g.tiles_y = (int)((OH + g.TH - 1) / g.TH);
        return sm <= 80 * 1024;
    };
    const auto blocks = [&]() { return B * g.tiles_x * g.tiles_y * g.n_blocks * g.phases; };
    // 256 positions per block from a block and a half per compute unit on: a step's weights then serve two products (48 + 48 ->
    // 48 channels at 180 x 320, 450 blocks: 18.7 -> 15.2 us; with 1.4 blocks per unit 7.3 -> 7.9 us)
    const auto wide = [&]() { return positions * ((N + 32 * nj - 1) / (32 * nj)) * g.phases * 2 >= 256 * 3 * cus ? 2 : 1; };
    // ---- blocks that walk tiles.  64 channels per block when that leaves fewer idle columns or the work fills the machine anyway
    const bool even = N > 32 && (N % 64 == 0 || N % 64 > 32);
    nj = even && positions * ((N + 63) / 64) * g.phases >= 128 * 2 * cus ? 2 : 1;
    tm = wide();
    bool looped = choose();
    if (!looped && tm == 2) tm = 1, looped = choose();
    const auto resident = [&]() { return std::max<int64_t>(1, std::min<int64_t>(blocks_per_cu(unit, nj, tm), (int64_t)(160 * 1024 / sm))) * cus; };
    // ---- a block per tile, unless the weights of many steps or of many channels would be fetched for each of three rounds of
    // blocks: 24 -> 24 channels 3 x 3 (9 steps) at 360 x 640, batch 4: 25.2 us looped, 26.5 with a block per tile, batch 3 20.7
    // and 20.4, batch 1 10.9 and 9.3; 16 -> 8 (5 steps), batch 4: 21.3 and 19.1; 32 -> 320 at 112 x 112, batch 16: 44.9 and 50.9
    if (!narrow && IC % 4 == 0 && reinterpret_cast<uintptr_t>(w->ptr) % 4 == 0 &&
        !(looped && blocks() >= 3 * resident() && (g.steps >= 8 || N > 128))) {
        const int nj0 = nj, tm0 = tm;
        direct = true;
        // 64 channels per block, 128 positions, from 1.4 blocks per unit on: 24 -> 48, stride 2, to 180 x 320 (450 blocks) 10.1 ->
        // 8.2 us; 20 -> 40 at 160 x 160, batch 2 (400) 8.1 -> 7.1; 36 -> 60 at 120 x 120 (113) 7.0 -> 7.2
        nj = even && g.ppt <= 3 && positions * ((N + 63) / 64) * g.phases * 5 >= 128 * 7 * cus ? 2 : 1;
        tm = nj == 2 ? 1 : wide();
        bool fits = choose();
        if (!fits && nj == 2) nj = 1, tm = wide(), fits = choose();
        if (!fits && tm == 2) tm = 1, fits = choose();
        // eight wavefronts where the shared memory of four leaves room for three blocks on a unit at most (96 -> 96 at 90 x 160,
        // 352 blocks of four: 7.9 -> 6.6 us; 48 -> 64 at 256 x 320, batch 4: 25.1 -> 21.9; 36 -> 60, 30 KiB: 7.0 -> 8.0), and where the
        // launching of blocks takes longer than their few products (1 x 1, 8 -> 19 at 480 x 640, batch 4, 4800: 28 -> 22 us; 900: 7.2 -> 7.7)
        if (fits && ((sm > 44 * 1024 && blocks() * 10 >= 13 * cus) || (g.steps <= 2 && blocks() >= 16 * cus))) {
            nw = 8;
            if (!choose()) nw = 4, choose();
        }
        // Where the other kernel has 64 channels to a block and this one's shared memory leaves 32, twice as many blocks fetch the
        // patch: TRANSPOSE_CONV2D 192 -> 97, 3 x 3, eight images of 95 x 18 20.9 us looped, 27.0 here; 9 of 17 such sizes longer, by up to 38 %
        if (looped && nj0 == 2 && nj == 1) fits = false;
        // What the other kernel does not take: not where most of a tile lies outside a small image, nor kernels of one or two
        // taps, for which contract_i8.hip's stages are short (68 -> 398, 2 x 2, over 105 x 1, batch 15: 9.1 us there, 15.6 here; 1 x 1,
        // 124 -> 128 at 69 x 177, batch 2: 8.3, 19.6; 2 x 1, 84 -> 186 at 139 x 39, batch 4: 11.9, 15.0; 3 x 3 and larger: 23 % faster here on
        // average over 67 sizes)
        if (!looped && fits && (positions * 3 < B * g.tiles_x * g.tiles_y * 32 * nw * tm || (!transposed && in2 == nullptr && kh * kw < 3)))
            fits = false;
        if (!fits) {
            direct = false, nw = 4, nj = nj0, tm = tm0;
            if (looped) choose();
        }
    }
    if (!direct && !looped) return 0;
    if (narrow) {
        g.step_tap = -g.ppt * 16;  // (one "tap" per kernel row)
        g.step_row = g.dy * g.PW * g.pitch;
    } else {
        g.step_tap = g.dx * g.pitch - g.ppt * 16;
        g.step_row = g.dy * g.PW * g.pitch - g.taps_x * g.dx * g.pitch;
    }
    g.tap_bytes = g.dx * g.pitch, g.row_bytes = g.dy * g.PW * g.pitch;
    g.x = static_cast<const int8_t *>(in->ptr), g.w = static_cast<const int8_t *>(w->ptr);
    g.x_bytes = (uint32_t)(B * H * W * IC1), g.w_bytes = (uint32_t)(OC * KH * KW * IC);
    if (in2 != nullptr) g.x2 = static_cast<const int8_t *>(in2->ptr), g.x2_bytes = (uint32_t)(B * H * W * (IC - IC1));
    g.out = static_cast<int8_t *>(out->ptr), g.bias = static_cast<const int32_t *>(bias->ptr), g.bias_len = (int)bias->dims[0];
    g.mult = static_cast<const char *>(epi->mult->ptr), g.shift = static_cast<const int8_t *>(epi->shift->ptr);
    g.mult16 = epi->scale32 ? 0 : 1;
    g.rp = epi->p;
    g.H = (int)H, g.W = (int)W, g.IC = (int)IC, g.IC1 = (int)IC1;
    g.OH = (int)OH, g.OW = (int)OW, g.N = (int)N;
    for (int k = 0; k < 2; k++) {
        g.n_chunks[k] = g.PH * g.PW * g.cpp[k], g.per_thread[k] = (int)per_thread(g.PH * g.PW, k);
        g.row_chunks[k] = std::max(1, g.PW * g.cpp[k]), g.columns[k] = (g.PW * g.cpp[k] + 63) / 64;
        g.rows[k] = std::max(1, 64 / g.row_chunks[k]);
        g.turns[k] = (g.PH + nw * g.rows[k] - 1) / (nw * g.rows[k]);
        g.mul_cpp[k] = (1u << 20) / (uint32_t)std::max(1, g.cpp[k]) + 1;
        g.mul_row[k] = g.rows[k] == 1 ? 0u : (1u << 20) / (uint32_t)g.row_chunks[k] + 1;
    }
    g.zx = zx;
    const int tw = 1 << g.log_tw;
    const int cols = g.n_blocks == 1 ? (int)N : 32 * nj;
    g.stage_row = (std::min(tw, 32) * cols + 15) / 16 * 16;
    const int64_t tiles = B * g.tiles_x * g.tiles_y, shares = (int64_t)g.n_blocks * g.phases;
    if (tiles * shares >= (int64_t(1) << 28)) return 0;
    // as many blocks as the machine holds at once, each with an equal share of the tiles of its channels
    const int64_t rounds = (tiles * shares + resident() - 1) / resident();
    g.groups = (int)((tiles + rounds - 1) / rounds);
    g.tiles_part = (int)(tiles / g.groups), g.tiles_rest = (int)(tiles % g.groups);
    g.blocks = (int)(g.groups * shares);
    g.chunk = (g.blocks + 7) / 8;
    g.div_group = make_div_magic((uint32_t)g.groups), g.div_nb = make_div_magic((uint32_t)g.n_blocks);
    g.div_tx = make_div_magic((uint32_t)g.tiles_x), g.div_ty = make_div_magic((uint32_t)g.tiles_y);
    g.mul_pw = (1u << 20) / (uint32_t)g.PW + 1;
    g.div_pieces = make_div_magic((uint32_t)g.steps * 2);
    g.div_ppt = make_div_magic((uint32_t)g.ppt), g.div_split = make_div_magic((uint32_t)g.split);
    g.div_run = make_div_magic((uint32_t)(g.stage_row / 16));
    const bool dual = in2 != nullptr;
    if (direct) {
        g.blocks = (int)(tiles * shares), g.chunk = (g.blocks + 7) / 8;
        g.groups = (int)tiles, g.div_group = make_div_magic((uint32_t)tiles);
        if (nj == 2) return nw == 8 ? launch_direct<2, 1, 8>(g, unit, dual, sm, s) : launch_direct<2, 1, 4>(g, unit, dual, sm, s);
        if (tm == 1) return nw == 8 ? launch_direct<1, 1, 8>(g, unit, dual, sm, s) : launch_direct<1, 1, 4>(g, unit, dual, sm, s);
        return nw == 8 ? launch_direct<1, 2, 8>(g, unit, dual, sm, s) : launch_direct<1, 2, 4>(g, unit, dual, sm, s);
    }
    if (narrow) {
        if (nj == 1) return tm == 1 ? launch_unit<1, 1, true>(g, unit, dual, sm, s) : launch_unit<1, 2, true>(g, unit, dual, sm, s);
        return tm == 1 ? launch_unit<2, 1, true>(g, unit, dual, sm, s) : launch_unit<2, 2, true>(g, unit, dual, sm, s);
    }
    if (nj == 1) return tm == 1 ? launch_unit<1, 1, false>(g, unit, dual, sm, s) : launch_unit<1, 2, false>(g, unit, dual, sm, s);
    return tm == 1 ? launch_unit<2, 1, false>(g, unit, dual, sm, s) : launch_unit<2, 2, false>(g, unit, dual, sm, s);
}

}  // namespace mlel
