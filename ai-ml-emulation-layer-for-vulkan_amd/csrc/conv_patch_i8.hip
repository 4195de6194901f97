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
// Blocks walk several tiles (the weights stay), with the next tile's pixels in registers while one is multiplied.
// A TRANSPOSE_CONV2D whose kernel equals its stride meets one input position per output: it is a 1 x 1 convolution to
// sx * OC channels per output row phase, whose results are contiguous in the output row.
//
// Measured (360 x 640, before -> after): 24 + 24 -> 24 channels 3 x 3: 75 -> 15.6 us; 3 -> 24: 25.6 -> 10.3 us; 1 x 1 24 -> 19: 19 -> 9.2 us;
// TRANSPOSE_CONV2D 48 -> 24 to 360 x 640: 20.5 -> 9.9 us; at half that size 48 + 48 -> 48: 17.2 -> 15.2 us.  Bound by the vector
// instructions of the requantisation (8 per result) and of the addresses, half of the time, and by the latency of a tile's
// fetch.  A channel count whose pieces and taps fill whole stages (64 channels, 3 x 3) stays with gemm_i8.hip, whose loads
// and products overlap from the first stage on (1 x 56 x 56 x 64: 6.5 us there, 8.3 us here).
#include <algorithm>

#include "common.hpp"
#include "dispatch.hpp"

namespace mlel {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
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
    int32_t ppt, taps_x, step_tap, step_row, pieces, steps;  // pieces of K: ppt per tap
    int32_t narrow_p;                                       // NARROW: bytes of a pixel in shared memory
    int32_t n_blocks, blocks, chunk, tiles, groups;         // groups: blocks per (phase, channel block)
    int32_t tiles_x, tiles_y;
    DivMagic div_group, div_nb, div_tx, div_ty, div_pieces, div_ppt, div_split, div_run;
    uint32_t mul_cpp[2], mul_pw;  // see quotient()
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
    const int first = (int)((int64_t)part * g.tiles / g.groups), last = (int)((int64_t)(part + 1) * g.tiles / g.groups);
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
    g.steps = (g.pieces + 1) / 2;
    const int64_t cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
    // 64 channels per block when that leaves fewer idle columns or the work fills the machine anyway
    int nj = N <= 32 ? 1 : (N % 64 == 0 || N % 64 > 32 ? 2 : 1);
    const int64_t positions = B * OH * OW;
    if (nj == 2 && positions * ((N + 63) / 64) * g.phases < 128 * 2 * cus) nj = 1;
    // tile: the shape of 256 (128) positions with the least padding, then the smallest patch
    // 256 positions per block from a block and a half per compute unit on: a step's weights then serve two products (48 + 48 ->
    // 48 channels at 180 x 320, 450 blocks: 18.7 -> 15.2 us; with 1.4 blocks per unit 7.3 -> 7.9 us)
    int tm = positions * ((N + 32 * nj - 1) / (32 * nj)) * g.phases * 2 >= 256 * 3 * cus ? 2 : 1;
    size_t sm = 0;
    for (; tm >= 1; tm--) {
        int64_t best = -1, best_patch = 0;
        for (int lt = 3; lt <= 6; lt++) {
            const int64_t tw = int64_t(1) << lt, th = 128 * tm / tw;
            const int64_t ph = (th - 1) * g.sy + (kh - 1) * g.dy + 1, pw = (tw - 1) * g.sx + (kw - 1) * g.dx + 1;
            const int64_t area = ((OH + th - 1) / th) * ((OW + tw - 1) / tw);
            const int64_t patch = ph * pw;
            if (ph > 511 || pw > 255 || patch * g.pitch > 65536) continue;  // what a thread's chunk descriptors hold
            if (per_thread(patch, 0) + per_thread(patch, 1) > kChunks) continue;
            if (best >= 0 && (area > best || (area == best && patch >= best_patch))) continue;
            best = area, best_patch = patch;
            g.log_tw = lt, g.TH = (int)th, g.PH = (int)ph, g.PW = (int)pw;
        }
        if (best < 0) continue;
        const int bn = 32 * nj;
        // slack: an odd number of pieces, and NARROW's whole pieces, read a little beyond the patch
        const int64_t slack = (int64_t)g.PW * g.dy * g.pitch + (int64_t)g.pitch * (g.dx + 1) + 64;
        g.patch_bytes = (int)((g.PH * g.PW * (int64_t)g.pitch + slack + 15) / 16 * 16);
        sm = (size_t)g.patch_bytes + (size_t)g.steps * 2 * (bn + 1) * 16 + bn * 4 + 4 * (32 * bn + 64);
        if (sm <= 80 * 1024) break;  // two blocks per compute unit
    }
    if (tm < 1) return 0;
    if (narrow) {
        g.step_tap = -g.ppt * 16;  // (one "tap" per kernel row)
        g.step_row = g.dy * g.PW * g.pitch;
    } else {
        g.step_tap = g.dx * g.pitch - g.ppt * 16;
        g.step_row = g.dy * g.PW * g.pitch - g.taps_x * g.dx * g.pitch;
    }
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
        g.mul_cpp[k] = (1u << 20) / (uint32_t)std::max(1, g.cpp[k]) + 1;
    }
    g.zx = zx;
    const int tw = 1 << g.log_tw;
    g.n_blocks = (int)((N + 32 * nj - 1) / (32 * nj));
    const int cols = g.n_blocks == 1 ? (int)N : 32 * nj;
    g.stage_row = (std::min(tw, 32) * cols + 15) / 16 * 16;
    g.tiles_x = (int)((OW + tw - 1) / tw), g.tiles_y = (int)((OH + g.TH - 1) / g.TH);
    const int64_t tiles = B * g.tiles_x * g.tiles_y, shares = (int64_t)g.n_blocks * g.phases;
    if (tiles * shares >= (int64_t(1) << 28)) return 0;
    g.tiles = (int)tiles;
    // as many blocks as the machine holds at once, each with an equal share of the tiles of its channels
    const int64_t resident = std::max<int64_t>(1, std::min<int64_t>(blocks_per_cu(unit, nj, tm), (int64_t)(160 * 1024 / sm))) * cus;
    const int64_t rounds = (tiles * shares + resident - 1) / resident;
    g.groups = (int)((tiles + rounds - 1) / rounds);
    g.blocks = (int)(g.groups * shares);
    g.chunk = (g.blocks + 7) / 8;
    g.div_group = make_div_magic((uint32_t)g.groups), g.div_nb = make_div_magic((uint32_t)g.n_blocks);
    g.div_tx = make_div_magic((uint32_t)g.tiles_x), g.div_ty = make_div_magic((uint32_t)g.tiles_y);
    g.mul_pw = (1u << 20) / (uint32_t)g.PW + 1;
    g.div_pieces = make_div_magic((uint32_t)g.steps * 2);
    g.div_ppt = make_div_magic((uint32_t)g.ppt), g.div_split = make_div_magic((uint32_t)g.split);
    g.div_run = make_div_magic((uint32_t)(g.stage_row / 16));
    const bool dual = in2 != nullptr;
    if (narrow) {
        if (nj == 1) return tm == 1 ? launch_unit<1, 1, true>(g, unit, dual, sm, s) : launch_unit<1, 2, true>(g, unit, dual, sm, s);
        return tm == 1 ? launch_unit<2, 1, true>(g, unit, dual, sm, s) : launch_unit<2, 2, true>(g, unit, dual, sm, s);
    }
    if (nj == 1) return tm == 1 ? launch_unit<1, 1, false>(g, unit, dual, sm, s) : launch_unit<1, 2, false>(g, unit, dual, sm, s);
    return tm == 1 ? launch_unit<2, 1, false>(g, unit, dual, sm, s) : launch_unit<2, 2, false>(g, unit, dual, sm, s);
}

}  // namespace mlel
