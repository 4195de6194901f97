// int8 CONV2D + RESCALE (+CLAMP) of few output tiles, over one image or two side by side along the channels (CONCAT read in
// place), and TRANSPOSE_CONV2D whose kernel is its stride (reference arithmetic: conv2d.comp:40-116,
// transpose_conv2d.comp:31-70, rescale.comp:27-72, clamp.comp:24-53).
//
// A network's inner layers on a small image have a few dozen tiles of 64 x 64 or of 128 positions, each the serial chain of its
// whole K: a handful of blocks, one wavefront on a SIMD, which issues an instruction every seven clocks.  Here a tile is
// 32 x 32 (or 16 x 16) and the four wavefronts of its block share K, whose order is free: sums of int32 wrap.  What is left is
// the bytes a block takes from the L2, 64 K (32 K) bytes at 41 per clock, and the fixed part of a launch.
//   Stages of 256 bytes of K for the tile's rows of X and W, requested straight into shared memory, four stages deep, one
//   barrier per stage; 16-byte pieces in XOR-swizzled slots (piece p of row r in slot p ^ (r & 15)), read as the operands of
//   v_mfma_i32_32x32x32_i8 (16x16x64).  A piece lies inside one tap (channels in multiples of 16; a second kernel below
//   pads the taps of the others).
//   A tap outside the image contributes nothing, so its piece must hold the input's zero point: such lanes fetch it from a
//   table of all 256 of them (a load through a buffer resource would leave zeros).
//   zx sum w: a second multiply of the same weights with a splat of -zx, into the same accumulator.
//   The shares of the tile are added through shared memory by a thread per four channels of a position, which requantises and
//   stores them.
//
// Measured (us, one image, 3 x 3, before -> after): 56 x 56 x 64 -> 64 5.7 -> 3.8, 16 x 16 x 64 -> 64 5.7 -> 3.2, 8 x 8 x 128 -> 128
// 9.7 -> 3.6, 14 x 14 x 256 -> 512 13.4 -> 5.2; 7 x 7 x 320 -> 512, 5 x 5: 15.2 -> 8.4.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "dispatch.hpp"

namespace mlel {
namespace {

typedef int v16i __attribute__((ext_vector_type(16)));

constexpr uint32_t kOob = 0x80000000u;
constexpr int kStages = 4;

struct ZeroPoints {  // sixteen bytes of every value
    uint32_t v[256 * 4];
};
constexpr ZeroPoints make_zero_points() {
    ZeroPoints z{};
    for (uint32_t i = 0; i < 256 * 4; i++) z.v[i] = (i >> 2) * 0x01010101u;
    return z;
}
__device__ const ZeroPoints zero_points = make_zero_points();

struct FewArgs {
    const int8_t *x, *x2, *w;
    int8_t *out;
    const int32_t *bias;
    const char *mult;
    const int8_t *shift;
    int32_t mult16, bias_len;
    RescaleParams rp;
    // image: H x W pixels of IC (= IC1 + IC2) bytes; x2: channels IC1 ..
    int32_t H, W, IC1, IC2;
    int32_t ppt, ppt1;  // pieces of a tap, and those of x
    uint32_t x_bytes, x2_bytes, w_bytes, o_bytes;
    int32_t sy, sx, dy, dx, pt, pl, KW;
    // M positions of N bytes; position row y of phase p is row y * phases + p of the output image; columns N / split kernel
    // columns of `split` channels (TRANSPOSE_CONV2D), else split = N
    int32_t M, N, pieces, OHW, OW, phases, split, w_row;  // w_row: bytes of a channel's weights
    int32_t total_tiles, chunk;
    TileOrder order;  // its batches: the phases
    DivMagic div_ohw, div_ow, div_split;
    uint32_t ppt_magic, kw_magic;  // piece / ppt = mulhi(piece, ppt_magic) for ppt > 1, tap / KW = tap kw_magic >> 16
    int32_t zx;
    int32_t ragged;  // (for the launch) pieces at any address
};

__device__ __forceinline__ v16i multiply(v4i w, v4i x, v16i acc) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(w, x, acc, 0, 0, 0); }
__device__ __forceinline__ v4i multiply(v4i w, v4i x, v4i acc) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(w, x, acc, 0, 0, 0); }

// ---- what both kernels share: the constants of a thread's four channels, and the end of a tile
struct Channels {
    int32_t bias[4], mult[4], shift[4];
};
__device__ __forceinline__ Channels load_channels(const FewArgs &g, int n0) {
    Channels c;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int n = min(n0 + e, g.N - 1), oc = g.split == g.N ? n : n - div_magic(n, g.div_split) * g.split;
        const int ch = g.rp.per_channel ? oc : 0;
        c.mult[e] = g.mult16 ? (int32_t) reinterpret_cast<const int16_t *>(g.mult)[ch] : reinterpret_cast<const int32_t *>(g.mult)[ch];
        c.shift[e] = (int32_t)g.shift[ch];
        c.bias[e] = g.bias[g.bias_len == 1 ? 0 : oc];
    }
    return c;
}
// The four shares of the tile, [4][BT][RP], in the shared memory of the stages (which have been read): a lane holds position
// lane % BT and, per register quad q, channels 4 MP q + 4 (lane / BT) ..; a thread then adds, requantises and stores four
// channels of a position.
template <int BT, typename acc_t>
__device__ __forceinline__ void finish(const FewArgs &g, char *smem, const acc_t &acc, const Channels &c, int phase, int m_base, int n_base) {
    constexpr int MP = 64 / BT, AR = BT * BT / 64, RP = BT + 4, QPR = BT / 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane / BT, lrow = lane % BT, qm = tid / QPR, qn = tid % QPR * 4;
    int32_t *shares = reinterpret_cast<int32_t *>(smem);
#pragma unroll
    for (int q = 0; q < AR / 4; q++)
        *reinterpret_cast<v4i *>(shares + (wave * BT + lrow) * RP + 4 * MP * q + 4 * h) = v4i{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    __syncthreads();
    if (BT * QPR < 256 && tid >= BT * QPR) return;
    const int m = m_base + qm, n = n_base + qn;
    v4i sum = v4i{c.bias[0], c.bias[1], c.bias[2], c.bias[3]};
#pragma unroll
    for (int k = 0; k < 4; k++) sum += *reinterpret_cast<const v4i *>(shares + (k * BT + qm) * RP + qn);
    const int32_t hi_v = pin_vgpr(g.rp.out_hi);
    uint32_t bytes = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const ChanScale cs = make_chan_scale(c.mult[e], c.shift[e], g.rp);
        bytes |= ((uint32_t)requant_acc(sum[e], cs, g.rp, hi_v) & 0xffu) << (8 * e);
    }
    if (m >= g.M || n >= g.N) return;
    const int row = g.phases == 1 ? 0 : div_magic(m, g.div_ow) * (g.phases - 1) + phase;
    const uint32_t at = (uint32_t)(m + row * g.OW) * (uint32_t)g.N + (uint32_t)n;
    const __amdgpu_buffer_rsrc_t ores = rsrc(g.out, g.o_bytes);
    if ((g.N & 3) == 0 && ((uintptr_t)g.out & 3) == 0) {  // uniform
        __builtin_amdgcn_raw_buffer_store_b32((int)bytes, ores, (int)at, 0, kOutAux);
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (n + e < g.N) __builtin_amdgcn_raw_buffer_store_b8((char)(bytes >> (8 * e)), ores, (int)(at + e), 0, 0);
    }
}

// BT x BT tile of positions and channels; DUAL: two images
template <int BT, bool DUAL>
__global__ void __launch_bounds__(256) conv_few_i8_kernel(const FewArgs g) {
    constexpr int NT = 256, WK = 4, BK = 256, PPR = BK / 16, MP = 64 / BT, AR = BT * BT / 64, S = kStages;
    constexpr int XI = BT * PPR / NT, STAGE = 2 * BT * BK, KKW = PPR / MP / WK, QPR = BT / 4, NLA = 2 * XI;
    static_assert(XI >= 1 && KKW >= 1 && (S - 1) * NLA < 16, "tile shape");
    typedef typename std::conditional<BT == 32, v16i, v4i>::type acc_t;
    extern __shared__ __align__(16) char smem[];
    // every argument in front of the first request, in one batch
    asm volatile("" ::"s"(g.chunk), "s"(g.total_tiles), "s"(g.order.tiles_m), "s"(g.order.tiles_n), "s"(g.order.rows), "s"(g.order.m_batch),
                 "s"(g.order.m_band), "s"(g.order.m_rows), "s"(g.order.m_last), "s"(g.order.shifts), "s"(g.div_ohw.m), "s"(g.div_ohw.s),
                 "s"(g.div_ow.m), "s"(g.div_ow.s), "s"(g.x), "s"(g.w), "s"(g.H), "s"(g.W), "s"(g.IC1), "s"(g.ppt), "s"(g.w_bytes), "s"(g.sy),
                 "s"(g.sx), "s"(g.dy), "s"(g.dx), "s"(g.pt), "s"(g.pl));
    asm volatile("" ::"s"(g.KW), "s"(g.M), "s"(g.N), "s"(g.pieces), "s"(g.OHW), "s"(g.OW), "s"(g.split), "s"(g.w_row), "s"(g.ppt_magic),
                 "s"(g.kw_magic), "s"(g.zx), "s"(g.bias), "s"(g.mult), "s"(g.shift), "s"(g.out), "s"(g.bias_len), "s"(g.mult16),
                 "s"(g.rp.per_channel), "s"(g.rp.double_round), "s"(g.rp.out_lo), "s"(g.rp.out_hi), "s"(g.rp.out_zp), "s"(g.o_bytes));
    const int lin = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u));
    if (lin >= g.total_tiles) return;
    int phase, tile_m, tile_n;
    g.order.tile(lin, phase, tile_m, tile_n);
    const int m_base = tile_m * BT, n_base = tile_n * BT;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // ---- this thread's pieces: rows r0 + i NT / PPR of X and of W, the same piece of each
    const int r0 = tid / PPR, p0 = (tid % PPR) ^ (r0 & 15);
    int32_t iy0[XI], ix0[XI], pix[XI];
    uint32_t wo[XI];
#pragma unroll
    for (int i = 0; i < XI; i++) {
        const int m = m_base + r0 + i * (NT / PPR), n = n_base + r0 + i * (NT / PPR);
        const int img = div_magic(m, g.div_ohw), pos = m - img * g.OHW, oy = div_magic(pos, g.div_ow), ox = pos - oy * g.OW;
        iy0[i] = m < g.M ? oy * g.sy - g.pt : -0x40000000;
        ix0[i] = ox * g.sx - g.pl;
        pix[i] = (img * g.H + oy * g.sy - g.pt) * g.W + ix0[i];
        if (g.split == g.N) {  // uniform
            wo[i] = n < g.N ? (uint32_t)(n * g.w_row + phase * g.KW * g.ppt * 16 + p0 * 16) : kOob;
        } else {
            const int kx = div_magic(n, g.div_split), oc = n - kx * g.split;
            wo[i] = n < g.N ? (uint32_t)(oc * g.w_row + (phase * g.KW + kx) * g.ppt * 16 + p0 * 16) : kOob;
        }
    }
    const v4i wres = rsrc_words(g.w, g.w_bytes);
    const char *outside = reinterpret_cast<const char *>(zero_points.v + 4 * (g.zx & 0xff));
    const uint32_t lds0 = (uint32_t) reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem) + (uint32_t)(wave * 1024);
    const int nk = (g.pieces + PPR - 1) / PPR;
    int piece = p0;  // of K, in the stage that is requested next
    auto request = [&](int step, int buf) {
        const uint32_t d = lds0 + (uint32_t)(buf * STAGE);
        const int tap = g.ppt == 1 ? piece : (int)__umulhi((uint32_t)piece, g.ppt_magic), c = piece - (int)__umul24(tap, g.ppt);
        const int y = (int)(__umul24(tap, g.kw_magic) >> 16), x = tap - (int)__umul24(y, g.KW);
        int yd = (int)__umul24(y, g.dy);
        const int xd = (int)__umul24(x, g.dx), away = (int)__umul24(yd, g.W) + xd;
        const bool partial = (step + 1) * PPR > g.pieces;  // uniform: the last stage ends beyond K
        if (partial) {
            yd = piece < g.pieces ? yd : 0x20000000;  // no tap
            asm volatile("" : "+v"(yd));  // (a branch, not a select in every stage)
        }
        const bool second = DUAL && c >= g.ppt1;
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const bool in = (uint32_t)(iy0[i] + yd) < (uint32_t)g.H && (uint32_t)(ix0[i] + xd) < (uint32_t)g.W;
            const char *from;
            if constexpr (DUAL) {
                const int pitch = second ? g.IC2 : g.IC1, first = second ? g.ppt1 : 0;
                from = reinterpret_cast<const char *>(second ? g.x2 : g.x) + (uint32_t)((pix[i] + away) * pitch + (c - first) * 16);
            } else {
                from = reinterpret_cast<const char *>(g.x) + (uint32_t)((pix[i] + away) * g.IC1 + c * 16);
            }
            load16_to_lds(in ? from : outside, d + i * NT * 16);
        }
#pragma unroll
        for (int i = 0; i < XI; i++) {
            uint32_t off = wo[i];
            if (partial) {
                off = piece < g.pieces ? off : kOob;
                asm volatile("" : "+v"(off));
            }
            load16_to_lds(wres, d + BT * BK + i * NT * 16, off, (uint32_t)(step * BK));
        }
        piece += PPR;
    };
#pragma unroll
    for (int d = 0; d < S - 1; d++)
        if (d < nk) request(d, d);  // uniform

    // ---- the constants of this thread's four channels, behind the first stages (younger than they are and older than every later
    // request: the counted waits hold)
    const Channels channels = load_channels(g, n_base + tid % QPR * 4);

    acc_t acc;
#pragma unroll
    for (int r = 0; r < AR; r++) acc[r] = 0;
    const int h = lane / BT, lrow = lane % BT;
    const char *x_at[KKW];
#pragma unroll
    for (int k = 0; k < KKW; k++) x_at[k] = smem + lrow * BK + ((((wave * KKW + k) * MP + h) ^ (lrow & 15)) * 16);
    // (-zx) as a byte; 128 is twice 64
    const int nz = g.zx == -128 ? 0x40404040 : (int)((uint32_t)(-g.zx & 0xff) * 0x01010101u);
    const v4i zeros = v4i{nz, nz, nz, nz};
    auto meet = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto step_of = [&](int buf, auto between) {
        v4i xf[KKW], wf[KKW];
#pragma unroll
        for (int k = 0; k < KKW; k++) {
            xf[k] = *reinterpret_cast<const v4i *>(x_at[k] + buf * STAGE);
            wf[k] = *reinterpret_cast<const v4i *>(x_at[k] + buf * STAGE + BT * BK);
        }
        __builtin_amdgcn_sched_barrier(0);
        between();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < KKW; k++) acc = multiply(wf[k], xf[k], acc);
        if (g.zx != 0) {  // uniform
#pragma unroll
            for (int k = 0; k < KKW; k++) acc = multiply(wf[k], zeros, acc);
            if (g.zx == -128) {
#pragma unroll
                for (int k = 0; k < KKW; k++) acc = multiply(wf[k], zeros, acc);
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // (every read has arrived before the next barrier)
    };
    // this thread's part of a stage has landed when at most the later stages are outstanding; the barrier extends that to the
    // block, and says that every wavefront has read the buffer that the next request overwrites
    int step = 0;
    while (step + S - 1 < nk) {  // unrolled over the ring: a stage's place is a constant
#pragma unroll
        for (int d = 0; d < S; d++) {
            if (step + S - 1 < nk) {  // uniform
                wait_vmcnt<(S - 2) * NLA>();
                meet();
                step_of(d, [&] { request(step + S - 1, (d + S - 1) % S); });
                step++;
            }
        }
    }
    int cur = step % S;
    auto drain = [&](auto self, auto left) {  // the last S - 1 stages: nothing is left to request
        constexpr int R = decltype(left)::value;
        if constexpr (R > 0) {
            if (nk - step >= R) {  // uniform
                wait_vmcnt<(R - 1) * NLA>();
                meet();
                step_of(cur, [] {});
                cur = cur + 1 == S ? 0 : cur + 1;
                step++;
            }
            self(self, std::integral_constant<int, R - 1>{});
        }
    };
    drain(drain, std::integral_constant<int, S - 1>{});
    __syncthreads();

    finish<BT>(g, smem, acc, channels, phase, m_base, n_base);
}

// The same for channel counts that are no whole pieces: a tap's last piece holds bytes of its neighbour, which meet zeros among the
// weights.  The pieces lie at any address, so they pass through registers, S stages ahead of their use, and two stage buffers.
template <int BT, int S, bool DUAL>
__global__ void __launch_bounds__(256) conv_few_ragged_i8_kernel(const FewArgs g) {
    constexpr int NT = 256, WK = 4, BK = 256, PPR = BK / 16, MP = 64 / BT, AR = BT * BT / 64;
    constexpr int XI = BT * PPR / NT, STAGE = 2 * BT * BK, KKW = PPR / MP / WK, QPR = BT / 4;
    static_assert(XI >= 1 && KKW >= 1 && S % 2 == 0, "tile shape; a set meets one buffer");
    typedef typename std::conditional<BT == 32, v16i, v4i>::type acc_t;
    extern __shared__ __align__(16) char smem[];
    asm volatile("" ::"s"(g.chunk), "s"(g.total_tiles), "s"(g.order.tiles_m), "s"(g.order.tiles_n), "s"(g.order.rows), "s"(g.order.m_batch),
                 "s"(g.order.m_band), "s"(g.order.m_rows), "s"(g.order.m_last), "s"(g.order.shifts), "s"(g.div_ohw.m), "s"(g.div_ohw.s),
                 "s"(g.div_ow.m), "s"(g.div_ow.s), "s"(g.x), "s"(g.w), "s"(g.H), "s"(g.W), "s"(g.IC1), "s"(g.ppt), "s"(g.w_bytes), "s"(g.sy),
                 "s"(g.sx), "s"(g.dy), "s"(g.dx), "s"(g.pt), "s"(g.pl), "s"(g.x_bytes));
    asm volatile("" ::"s"(g.KW), "s"(g.M), "s"(g.N), "s"(g.pieces), "s"(g.OHW), "s"(g.OW), "s"(g.split), "s"(g.w_row), "s"(g.ppt_magic),
                 "s"(g.kw_magic), "s"(g.zx), "s"(g.bias), "s"(g.mult), "s"(g.shift), "s"(g.out), "s"(g.bias_len), "s"(g.mult16),
                 "s"(g.rp.per_channel), "s"(g.rp.double_round), "s"(g.rp.out_lo), "s"(g.rp.out_hi), "s"(g.rp.out_zp), "s"(g.o_bytes));
    const int lin = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u));
    if (lin >= g.total_tiles) return;
    int phase, tile_m, tile_n;
    g.order.tile(lin, phase, tile_m, tile_n);
    const int m_base = tile_m * BT, n_base = tile_n * BT;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int IC = g.IC1 + g.IC2;

    const int r0 = tid / PPR, p0 = (tid % PPR) ^ (r0 & 15);
    int32_t iy0[XI], ix0[XI], pix[XI];
    uint32_t wo[XI];
#pragma unroll
    for (int i = 0; i < XI; i++) {
        const int m = m_base + r0 + i * (NT / PPR), n = min(n_base + r0 + i * (NT / PPR), g.N - 1);  // (beyond N: not stored)
        const int img = div_magic(m, g.div_ohw), pos = m - img * g.OHW, oy = div_magic(pos, g.div_ow), ox = pos - oy * g.OW;
        iy0[i] = m < g.M ? oy * g.sy - g.pt : -0x40000000;
        ix0[i] = ox * g.sx - g.pl;
        pix[i] = (img * g.H + oy * g.sy - g.pt) * g.W + ix0[i];
        const int kx = g.split == g.N ? 0 : div_magic(n, g.div_split), oc = n - kx * g.split;
        wo[i] = (uint32_t)(oc * g.w_row + (phase * g.KW + kx) * IC);
    }
    const char *outside = reinterpret_cast<const char *>(zero_points.v + 4 * (g.zx & 0xff));
    // bytes of the last piece of a tap (DUAL: of x, and of x2)
    const int rem1 = g.IC1 - (g.ppt1 - 1) * 16, rem2 = DUAL ? g.IC2 - (g.ppt - g.ppt1 - 1) * 16 : rem1;
    uint32_t tail1[4], tail2[4];
#pragma unroll
    for (int d = 0; d < 4; d++) tail1[d] = keep_bytes(0xffffffffu, rem1 - 4 * d), tail2[d] = keep_bytes(0xffffffffu, rem2 - 4 * d);

    // A piece that would reach beyond its operand is loaded from further in front (`back`: by how many bytes) and moved when it
    // is stored; `tail`: what of W's piece belongs to its tap.
    struct Set {
        uint4 x[XI], w[XI];
        uint32_t back;  // a byte per piece: those of x, then those of w
        int tail;       // 0: all of it, 1: tail1, 2: tail2, 3: nothing
    };
    const int nk = (g.pieces + PPR - 1) / PPR;
    auto fetch = [&](Set &r, int stage) {  // (beyond the last one: nothing of it is used)
        const int piece = min(stage, nk) * PPR + p0;
        const int tap = g.ppt == 1 ? piece : (int)__umulhi((uint32_t)piece, g.ppt_magic), c = piece - (int)__umul24(tap, g.ppt);
        const int y = (int)(__umul24(tap, g.kw_magic) >> 16), x = tap - (int)__umul24(y, g.KW);
        const bool live = piece < g.pieces, second = DUAL && c >= g.ppt1;
        const int yd = live ? (int)__umul24(y, g.dy) : 0x20000000, xd = (int)__umul24(x, g.dx), away = (int)__umul24(__umul24(y, g.dy), g.W) + xd;
        const int pitch = second ? g.IC2 : g.IC1, cb = (second ? c - g.ppt1 : c) * 16;
        const char *base = reinterpret_cast<const char *>(second ? g.x2 : g.x);
        const uint32_t last = (second ? g.x2_bytes : g.x_bytes) - 16;
        r.back = 0;
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const bool in = (uint32_t)(iy0[i] + yd) < (uint32_t)g.H && (uint32_t)(ix0[i] + xd) < (uint32_t)g.W;
            const uint32_t off = (uint32_t)((pix[i] + away) * pitch + cb), at = min(off, last);
            r.back |= in ? (off - at) << (8 * i) : 0u;
            r.x[i] = load_any<16>(in ? base + at : outside);
        }
        const uint32_t k = live ? (uint32_t)(tap * IC + (second ? g.IC1 : 0) + cb) : 0u;
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const uint32_t off = wo[i] + k, at = min(off, g.w_bytes - 16);
            r.back |= (off - at) << (8 * (XI + i));
            r.w[i] = load_any<16>(g.w + at);
        }
        r.tail = !live ? 3 : (c == g.ppt - 1 ? 2 : (DUAL && c == g.ppt1 - 1 ? 1 : 0));
    };
    auto forward = [&](uint4 v, uint32_t by) {  // `by` bytes (below 16) to the front
        uint32_t w[5] = {v.x, v.y, v.z, v.w, 0};
        if (by & 4) w[0] = w[1], w[1] = w[2], w[2] = w[3], w[3] = 0;
        if (by & 8) w[0] = w[2], w[1] = w[3], w[2] = w[3] = 0;
        const uint32_t sh = (by & 3) * 8;
        return make_uint4(__builtin_amdgcn_alignbit(w[1], w[0], sh), __builtin_amdgcn_alignbit(w[2], w[1], sh),
                          __builtin_amdgcn_alignbit(w[3], w[2], sh), __builtin_amdgcn_alignbit(w[4], w[3], sh));
    };
    auto store = [&](char *st, const Set &from) {
        Set r = from;
        if (r.back != 0) {  // the ends of the operands
#pragma unroll
            for (int i = 0; i < XI; i++) {
                r.x[i] = forward(r.x[i], (r.back >> (8 * i)) & 0xff);
                r.w[i] = forward(r.w[i], (r.back >> (8 * (XI + i))) & 0xff);
            }
        }
        if (r.tail != 0) {
            uint32_t keep[4];
#pragma unroll
            for (int d = 0; d < 4; d++) keep[d] = r.tail == 3 ? 0u : (r.tail == 2 ? tail2[d] : tail1[d]);
#pragma unroll
            for (int i = 0; i < XI; i++) r.w[i] = make_uint4(r.w[i].x & keep[0], r.w[i].y & keep[1], r.w[i].z & keep[2], r.w[i].w & keep[3]);
        }
#pragma unroll
        for (int i = 0; i < XI; i++) {
            *reinterpret_cast<uint4 *>(st + (i * NT + tid) * 16) = r.x[i];
            *reinterpret_cast<uint4 *>(st + BT * BK + (i * NT + tid) * 16) = r.w[i];
        }
    };
    Set r[S];
#pragma unroll
    for (int d = 0; d < S; d++) fetch(r[d], d);
    const Channels channels = load_channels(g, n_base + tid % QPR * 4);

    acc_t acc;
#pragma unroll
    for (int i = 0; i < AR; i++) acc[i] = 0;
    const int h = lane / BT, lrow = lane % BT;
    const char *x_at[KKW];
#pragma unroll
    for (int k = 0; k < KKW; k++) x_at[k] = smem + lrow * BK + ((((wave * KKW + k) * MP + h) ^ (lrow & 15)) * 16);
    const int nz = g.zx == -128 ? 0x40404040 : (int)((uint32_t)(-g.zx & 0xff) * 0x01010101u);
    const v4i zeros = v4i{nz, nz, nz, nz};
    auto compute = [&](int buf) {
        v4i xf[KKW], wf[KKW];
#pragma unroll
        for (int k = 0; k < KKW; k++) {
            xf[k] = *reinterpret_cast<const v4i *>(x_at[k] + buf * STAGE);
            wf[k] = *reinterpret_cast<const v4i *>(x_at[k] + buf * STAGE + BT * BK);
        }
#pragma unroll
        for (int k = 0; k < KKW; k++) acc = multiply(wf[k], xf[k], acc);
        if (g.zx != 0) {  // uniform
#pragma unroll
            for (int k = 0; k < KKW; k++) acc = multiply(wf[k], zeros, acc);
            if (g.zx == -128) {
#pragma unroll
                for (int k = 0; k < KKW; k++) acc = multiply(wf[k], zeros, acc);
            }
        }
    };
    store(smem, r[0]);
    __syncthreads();
    for (int step = 0; step < nk; step += S) {
#pragma unroll
        for (int d = 0; d < S; d++) {
            if (step + d < nk) {  // uniform
                fetch(r[d], step + d + S);
                if (step + d + 1 < nk) store(smem + ((d + 1) & 1) * STAGE, r[(d + 1) % S]);
                compute(d & 1);
                __syncthreads();
            }
        }
    }
    finish<BT>(g, smem, acc, channels, phase, m_base, n_base);
}

template <int BT, bool DUAL>
int launch_kernel(FewArgs &g, hipStream_t s) {
    const int64_t tiles_m = (g.M + BT - 1) / BT, tiles_n = (g.N + BT - 1) / BT;
    g.total_tiles = (int)(tiles_m * tiles_n * g.phases);
    g.chunk = (g.total_tiles + 7) / 8;
    // (the rows of a tile meet the same pixels tap after tap)
    g.order = make_tile_order(tiles_m, tiles_n, g.chunk, (int64_t)BT * (g.IC1 + g.IC2) * g.sy * g.sx, (int64_t)BT * g.pieces * 16);
    constexpr size_t sm = (size_t)kStages * 2 * BT * 256;
    static_assert(sm <= 64 * 1024 && sm / 2 >= 4 * BT * (BT + 4) * 4, "the default limit of dynamic shared memory; the shares");
    const dim3 grid((unsigned)(g.chunk * 8));
    if (!g.ragged)
        conv_few_i8_kernel<BT, DUAL><<<grid, dim3(256), sm, s>>>(g);
    else if (g.pieces <= 32)  // (two stages: no more are asked for)
        conv_few_ragged_i8_kernel<BT, 2, DUAL><<<grid, dim3(256), sm / 2, s>>>(g);
    else
        conv_few_ragged_i8_kernel<BT, 4, DUAL><<<grid, dim3(256), sm / 2, s>>>(g);
    MLEL_TRY(check_launch("conv2d int8, few tiles"));
    return 1;
}

}  // namespace

// The operands are checked by the caller: packed int8 tensors whose extents in bytes fit 31 bits, an epilogue to 8 bits.
// `transposed`: TRANSPOSE_CONV2D, `pad` its output padding.  0: not a case for this kernel.
int try_conv_few_i8(mlel_ctx *ctx, hipStream_t s, const mlel_tensor *out, const mlel_tensor *in, const mlel_tensor *in2,
                    const mlel_tensor *w, const mlel_tensor *bias, const FusedEpilogue *epi, int32_t zx, int32_t zw,
                    const int32_t *pad, const int32_t *stride, const int32_t *dilation, bool transposed) {
    if (epi == nullptr || epi->p.in_zp != 0 || zw != 0 || dt_size(out->dtype) != 1) return 0;
    if (zx < -128 || zx > 127) return 0;  // (-zx is a byte of an operand here; the kernels of more tiles multiply in 32 bits)
    const int64_t B = in->dims[0], H = in->dims[1], W = in->dims[2], IC1 = in->dims[3], IC2 = in2 ? in2->dims[3] : 0, IC = IC1 + IC2;
    const int64_t OC = w->dims[0], KH = w->dims[1], KW = w->dims[2];
    FewArgs g{};
    // pieces of 16 bytes that lie inside one tap
    g.ragged = IC1 % 16 != 0 || IC2 % 16 != 0 || (uintptr_t)in->ptr % 16 != 0 || (uintptr_t)w->ptr % 16 != 0 || (in2 && (uintptr_t)in2->ptr % 16 != 0);
    if (B * H * W * IC1 < 16 || (in2 && B * H * W * IC2 < 16) || OC * KH * KW * IC < 16) return 0;
    g.sy = g.sx = g.dy = g.dx = g.phases = 1;
    int64_t N = OC, OH = out->dims[1], OW = out->dims[2], taps = KH * KW, kw = KW;
    if (transposed) {
        if (KH != stride[0] || KW != stride[1] || pad[0] != 0 || pad[1] != 0 || pad[2] != 0 || pad[3] != 0 || OH != H * KH || OW != W * KW)
            return 0;
        g.phases = (int)KH;
        N = OC * KW, OH = H, OW = W, taps = kw = 1;
    } else {
        g.sy = stride[0], g.sx = stride[1], g.dy = dilation[0], g.dx = dilation[1], g.pt = pad[0], g.pl = pad[2];
    }
    const int64_t M = B * OH * OW, ppt1 = (IC1 + 15) / 16, ppt = ppt1 + (IC2 + 15) / 16, K = taps * ppt * 16;
    if (KH > 32 || KW > 32 || N >= 65536 || M >= (1 << 28) || H >= 65536 || W >= 65536 || g.sy >= 1024 || g.sx >= 1024 || g.dy >= 1024 || g.dx >= 1024)
        return 0;
    for (int i = 0; i < 4; i++)
        if (pad[i] < -65536 || pad[i] > 65536) return 0;
    if ((K / 16 + 64) * ppt >= (int64_t(1) << 32) || B * H * W * IC >= (int64_t(1) << 31) - 4096 || OC * KH * KW * IC >= (int64_t(1) << 31) - 4096 ||
        M * N * g.phases >= (int64_t(1) << 31) - 4096)
        return 0;
    const int64_t cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
    const auto tiles = [&](int64_t t) { return (M + t - 1) / t * ((N + t - 1) / t) * g.phases; };
    // us, before / tiles of 32 / tiles of 16 (3 x 3 over one image): 64 x 64 x 32 -> 16 (256 tiles of 16) 5.5 / 3.4 / 3.1, 40 x 40 x 16
    // -> 32 twice, 5 x 5 (400) 6.0 / 3.4 / 3.5, 14 x 14 x 256 -> 512 (416) 13.4 / 5.5 / 5.2, 56 x 56 x 64 -> 64 (784; 196 of 32) 5.7 /
    // 3.8 / 4.9; 128 x 128 x 32 -> 32 (512 of 32) 5.6 / 4.1, 76 x 76 x 64 -> 96 (543) 6.8 / 6.5, 120 x 160 x 32 -> 32 (600) 5.5 / 5.8,
    // 56 x 56 x 64 -> 64 four times (784) 5.9 / 7.4; longer: 28 x 28 x 256 -> 512 twice (784) 13.3 / 11.9
    const bool small = tiles(16) * 2 <= 3 * cus || (tiles(16) <= 2 * cus && K >= 1024);
    if (!small && !(tiles(32) <= 2 * cus || (tiles(32) <= 3 * cus && K >= 1024))) return 0;
    // pieces at any address, conv_patch_i8.hip / tiles of 32 here: 28 x 28 x 100 -> 300 (250 tiles) 9.0 / 6.3, 64 x 64 x 40 -> 60 (256) 7.0 /
    // 4.9, 60 x 60 x 50 -> 100 (452) 8.3 / 7.8, 50 x 50 x 100 -> 170 (474) 10.0 / 7.6; 100 x 100 x 10 -> 20 (313) 5.5 / 5.8, 70 x 70 x 18 ->
    // 64, 5 x 5 (308) 9.2 / 9.5: beyond one tile per unit not where the pieces are more than half as much again as the channels
    if (g.ragged && !small && tiles(32) > cus && (tiles(32) > 2 * cus || 3 * IC < 2 * 16 * ppt)) return 0;
    // nor where large kernels of a few channels are mostly padding, from a tile of 16 per unit on: 7 x 35 x 3 -> 144 four times, 7 x 7
    // (558) 5.4 / 7.5, 8 x 248 of 1 channel eleven times (464) 5.5 / 7.6; 18 of 1200 random sizes, on average 14 % longer here
    if (g.ragged && 2 * IC < 16 * ppt && K - taps * IC > 350 && tiles(16) > cus) return 0;
    g.x = static_cast<const int8_t *>(in->ptr), g.w = static_cast<const int8_t *>(w->ptr);
    g.x2 = in2 != nullptr ? static_cast<const int8_t *>(in2->ptr) : g.x;
    g.out = static_cast<int8_t *>(out->ptr), g.bias = static_cast<const int32_t *>(bias->ptr), g.bias_len = (int)bias->dims[0];
    g.mult = static_cast<const char *>(epi->mult->ptr), g.shift = static_cast<const int8_t *>(epi->shift->ptr);
    g.mult16 = epi->scale32 ? 0 : 1;
    g.rp = epi->p;
    g.H = (int)H, g.W = (int)W, g.IC1 = (int)IC1, g.IC2 = (int)IC2;
    g.ppt = (int)ppt, g.ppt1 = (int)ppt1;
    g.x_bytes = (uint32_t)(B * H * W * IC1), g.x2_bytes = (uint32_t)(B * H * W * IC2);
    g.w_bytes = (uint32_t)(OC * KH * KW * IC), g.o_bytes = (uint32_t)(M * N * g.phases);
    g.KW = (int)KW;
    g.M = (int)M, g.N = (int)N, g.pieces = (int)(K / 16), g.OHW = (int)(OH * OW), g.OW = (int)OW;
    g.split = transposed ? (int)OC : (int)N, g.w_row = (int)(KH * KW * IC);
    g.div_ohw = make_div_magic((uint32_t)g.OHW), g.div_ow = make_div_magic((uint32_t)g.OW), g.div_split = make_div_magic((uint32_t)g.split);
    g.ppt_magic = (uint32_t)((uint64_t(1) << 32) / (uint32_t)ppt + 1), g.kw_magic = 65536u / (uint32_t)kw + 1;
    g.zx = zx;
    if (in2 != nullptr) return small ? launch_kernel<16, true>(g, s) : launch_kernel<32, true>(g, s);
    return small ? launch_kernel<16, false>(g, s) : launch_kernel<32, false>(g, s);
}

}  // namespace mlel
