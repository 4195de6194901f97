// Floating-point contractions on the matrix cores: CONV2D (NHWC x OHWI, fp32 accumulator) over fp16, bf16 and fp32
// tensors, and MATMUL over the same types with an fp32 result, for whatever extents and alignment gemm_f16.hip does not
// take (reference arithmetic: conv2d.comp:40-116, matmul.comp:30-73; the order of the fp32 additions differs from the
// shaders' sequential loops, the operands and the accumulator keep their types).
//
// One kernel body.  out[m][n] = sum_k X[m][k] * W[n][k]; k runs over 16-byte pieces (eight 16-bit or four 32-bit
// elements), and a piece of X lies inside one tap of the convolution.  A block keeps stages of BKB bytes of K for its
// BM rows and BN columns in shared memory, as pieces in XOR-swizzled slots (piece p of row r in slot
// p ^ ((r >> SH) & mask), so that the sixteen lanes an LDS cycle serves meet sixteen different 16-byte banks), and every
// type reads the same 128-bit operands: one v_mfma_f32_32x32x16 per piece pair for 16-bit types, four
// v_mfma_f32_32x32x2_f32 for fp32 (the K order inside a piece pair is permuted alike on both sides).
//   DIRECT: every piece is 16-byte aligned: buffer loads straight into shared memory, S stages deep, one barrier per
//           stage.  A lane carries the position of its piece along K, from which tap and channel follow, so that padding,
//           strides, dilation and channel counts that are no multiple of a stage cost a few vector instructions.
//   else:   pieces from any address are loaded into registers, S stages ahead, and stored into two stage buffers; a K-major W
//           keeps its rows in shared memory and is transposed by the reads (ds_read_b64_tr_b16; fp32 reads columns).
// Small problems: with one tile of 64 x 64 per compute unit nothing but the stage depth hides the trip to memory, so the
// tile shrinks to 32 x 32 and the four wavefronts of a block share a stage's K instead of its rows (WK = 4), summed
// through shared memory at the end -- no exchange between blocks.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "dispatch.hpp"

namespace mlel {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) v4s lds_v4s;

constexpr uint32_t kOob = 0x80000000u;

struct BF16 {};  // tag: bf16 storage

template <typename T> struct Elem;  // size, decode, encode of a storage type
template <> struct Elem<_Float16> {
    static constexpr int size = 2;
    static __device__ __forceinline__ float get(uint32_t bits) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits); }
    static __device__ __forceinline__ uint32_t put(float v, bool) {
        return __half_as_ushort(f2h(v));
    }
};
template <> struct Elem<BF16> {
    static constexpr int size = 2;
    static __device__ __forceinline__ float get(uint32_t bits) { return decode_bf16((uint16_t)bits); }
    static __device__ __forceinline__ uint32_t put(float v, bool nearest) {
        return nearest ? encode_bf16_rne(v) : encode_bf16_trunc(v);
    }
};
template <> struct Elem<float> {
    static constexpr int size = 4;
    static __device__ __forceinline__ float get(uint32_t bits) { return __uint_as_float(bits); }
    static __device__ __forceinline__ uint32_t put(float v, bool) { return __float_as_uint(v); }
};

struct FArgs {
    const char *x, *w;
    const char *bias, *res;  // of the output's type; res: of the output's shape and layout, or null
    char *out;
    int32_t M, N, K;                    // K in elements
    int32_t total_tiles, chunk;
    TileOrder order;
    DivMagic div_ohw, div_ow, div_ppr;
    // X: row m is output position (image, oy, ox) of a convolution (a product: one "image" of M positions, one tap)
    int32_t IC, KW, KH, H, W, sy, sx, pt, pl, dy, dx, OHW, OW;
    uint32_t x_img, x_row, x_pix, x_bytes;  // byte strides and extent of one batch
    // W: row-wise [N][K] with a pitch of ldw, or (w_kmajor) [K][N] with a pitch of ldw
    uint32_t ldw, w_bytes;
    int64_t x_batch, w_batch, o_batch;
    uint32_t ldo, o_bytes;
    uint32_t ic_magic, kw_magic;  // k / IC = mulhi(k, ic_magic), tap / KW = tap kw_magic >> 16 (DIRECT)
    int32_t bias_len;
    int32_t wide_out;  // rows of the result in whole aligned 16-byte pieces
    int32_t border;    // some tap of some position lies outside the image
    int32_t in_order;  // (for the tile choice) K is to be added in one sequence, as gemm_f16.hip does
    int32_t has_clamp, clamp_nan_ignore;
    float clamp_lo, clamp_hi;
};

__device__ __forceinline__ uint4 load16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const v4i v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
    return make_uint4((uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w);
}
template <int BYTES>
__device__ __forceinline__ uint4 load_piece(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    if constexpr (BYTES == 16) return load16(r, off);
    const v2i v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
    return make_uint4((uint32_t)v.x, (uint32_t)v.y, 0, 0);
}
template <int BYTES>
__device__ __forceinline__ void store_piece(__amdgpu_buffer_rsrc_t r, uint32_t off, uint4 v) {
    if constexpr (BYTES == 16) __builtin_amdgcn_raw_buffer_store_b128(v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w}, r, (int)off, 0, kOutAux);
    else __builtin_amdgcn_raw_buffer_store_b64(v2i{(int)v.x, (int)v.y}, r, (int)off, 0, kOutAux);
}
template <int SIZE>
__device__ __forceinline__ uint32_t load_elem(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    if constexpr (SIZE == 2) return (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0);
    else return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
}

// 16 x 16: the same over four pieces
template <typename T>
__device__ __forceinline__ v4f multiply(uint4 w, uint4 x, v4f acc) {
    if constexpr (std::is_same<T, _Float16>::value) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, w), __builtin_bit_cast(v8h, x), acc, 0, 0, 0);
    } else if constexpr (std::is_same<T, BF16>::value) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8b, w), __builtin_bit_cast(v8b, x), acc, 0, 0, 0);
    } else {
        const v4f a = __builtin_bit_cast(v4f, w), b = __builtin_bit_cast(v4f, x);
#pragma unroll
        for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
        return acc;
    }
}
template <typename T>
__device__ __forceinline__ v16f multiply(uint4 w, uint4 x, v16f acc) {
    if constexpr (std::is_same<T, _Float16>::value) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, w), __builtin_bit_cast(v8h, x), acc, 0, 0, 0);
    } else if constexpr (std::is_same<T, BF16>::value) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, w), __builtin_bit_cast(v8b, x), acc, 0, 0, 0);
    } else {
        const v4f a = __builtin_bit_cast(v4f, w), b = __builtin_bit_cast(v4f, x);
#pragma unroll
        for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], acc, 0, 0, 0);
        return acc;
    }
}

// how a register-staged operand is fetched
enum { F_PIECES = 0,   // aligned 16-byte pieces
       F_ROWS = 1,     // products: 16-byte pieces of rows from any address
       F_RUNS = 2,     // convolutions: the taps of a kernel row are one run of KW IC elements, padded to whole pieces of K, that
                       // lie anywhere; elements outside the image or beyond the run are zeros
       F_ELEMS = 3,    // element by element along K (convolutions dilated along the row)
       F_KMAJOR = 4,   // W of a product only: pieces of the rows of [K][N], from any address, transposed on their way out of
                       // shared memory
       F_TAPS = 5 };   // X, DIRECT: F_PIECES with the taps inside the image as a bit each

// What position m gives for column n before its rounding, over the taps inside the image one after the other, until the sum is
// NaN for good; false for a position whose taps all lie inside.
template <typename T, typename TO>
__device__ __forceinline__ bool sum_inside(const FArgs &g, int m, int n, float &s) {
    constexpr int SZ = Elem<T>::size, SO = Elem<TO>::size;
    const int img = div_magic(m, g.div_ohw), pos = m - img * g.OHW, oy = div_magic(pos, g.div_ow), ox = pos - oy * g.OW;
    const int iy0 = oy * g.sy - g.pt, ix0 = ox * g.sx - g.pl;
    if (iy0 >= 0 && ix0 >= 0 && iy0 + (g.KH - 1) * g.dy < g.H && ix0 + (g.KW - 1) * g.dx < g.W) return false;
    const __amdgpu_buffer_rsrc_t xres = rsrc(g.x, g.x_bytes), wres = rsrc(g.w, g.w_bytes), bres = rsrc(g.bias, (uint32_t)(g.bias_len * SO));
    s = 0.f;
    for (int tap = 0; tap < g.KH * g.KW && s == s; tap++) {
        const int ky = tap / g.KW, kx = tap - ky * g.KW, iy = iy0 + ky * g.dy, ix = ix0 + kx * g.dx;
        if ((uint32_t)iy >= (uint32_t)g.H || (uint32_t)ix >= (uint32_t)g.W) continue;
        const uint32_t xo = (uint32_t)img * g.x_img + (uint32_t)iy * g.x_row + (uint32_t)ix * g.x_pix;
        const uint32_t wo = (uint32_t)n * g.ldw + (uint32_t)(tap * g.IC * SZ);
#pragma unroll 4
        for (int c = 0; c < g.IC; c++)
            s += Elem<T>::get(load_elem<SZ>(xres, xo + (uint32_t)(c * SZ))) * Elem<T>::get(load_elem<SZ>(wres, wo + (uint32_t)(c * SZ)));
    }
    s += Elem<TO>::get(load_elem<SO>(bres, g.bias_len == 1 ? 0u : (uint32_t)(n * SO)));
    return true;
}

// elements lo .. hi - 1 of a piece, the others zeros
template <int SZ>
__device__ __forceinline__ uint4 keep_elems(uint4 v, int lo, int hi) {
    uint32_t *w = &v.x;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if constexpr (SZ == 4) {
            w[k] = k >= lo && k < hi ? w[k] : 0u;
        } else {
            const uint32_t low = 2 * k >= lo && 2 * k < hi ? 0xffffu : 0u, high = 2 * k + 1 >= lo && 2 * k + 1 < hi ? 0xffff0000u : 0u;
            w[k] &= low | high;
        }
    }
    return v;
}
// the words of a piece that keep its first `n` (any value) elements
template <int SZ>
__device__ __forceinline__ uint4 first_elems(int n) {
    uint4 v;
    uint32_t *w = &v.x;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if constexpr (SZ == 4) w[k] = n > k ? 0xffffffffu : 0u;
        else w[k] = n > 2 * k + 1 ? 0xffffffffu : (n > 2 * k ? 0xffffu : 0u);
    }
    return v;
}
__device__ __forceinline__ uint4 both(const uint4 &a, const uint4 &b) { return make_uint4(a.x & b.x, a.y & b.y, a.z & b.z, a.w & b.w); }
// a piece moved `by` elements to the front (zeros behind)
template <int SZ>
__device__ __forceinline__ uint4 move_elems(uint4 v, int by) {
    const uint32_t d = (uint32_t)by * SZ / 4, sh = (uint32_t)by * SZ % 4 * 8;
    uint32_t w[5] = {v.x, v.y, v.z, v.w, 0};
    if (d & 1) w[0] = w[1], w[1] = w[2], w[2] = w[3], w[3] = 0;
    if (d & 2) w[0] = w[2], w[1] = w[3], w[2] = w[3] = 0;
    return make_uint4(__builtin_amdgcn_alignbit(w[1], w[0], sh), __builtin_amdgcn_alignbit(w[2], w[1], sh),
                      __builtin_amdgcn_alignbit(w[3], w[2], sh), __builtin_amdgcn_alignbit(w[4], w[3], sh));
}
// ADD of the residual (one rounding, to nearest) and CLAMP, as the stand-alone operators compute them
template <typename TO>
__device__ __forceinline__ uint32_t finish_bits(const FArgs &g, uint32_t bits, uint32_t res_bits) {
    if (g.res != nullptr) bits = Elem<TO>::put(Elem<TO>::get(bits) + Elem<TO>::get(res_bits), true);
    if (g.has_clamp) {
        float v = Elem<TO>::get(bits);
        if (v != v && g.clamp_nan_ignore) v = g.clamp_lo;
        if (v < g.clamp_lo) v = g.clamp_lo;
        if (v > g.clamp_hi) v = g.clamp_hi;
        bits = Elem<TO>::put(v, false);
    }
    return bits;
}
template <typename TO, int WORDS>
__device__ __forceinline__ uint4 finish_words(const FArgs &g, uint4 v, const uint4 &r) {
    uint32_t *w = reinterpret_cast<uint32_t *>(&v);
    const uint32_t *rw = reinterpret_cast<const uint32_t *>(&r);
#pragma unroll
    for (int e = 0; e < WORDS; e++) {
        if constexpr (Elem<TO>::size == 2)
            w[e] = finish_bits<TO>(g, w[e] & 0xffffu, rw[e] & 0xffffu) | (finish_bits<TO>(g, w[e] >> 16, rw[e] >> 16) << 16);
        else
            w[e] = finish_bits<TO>(g, w[e], rw[e]);
    }
    return v;
}

constexpr int stage_bytes(int bm, int bn, int bkb, int size, bool km) {
    return km ? bm * bkb + (bkb / size) * (bn * size + 32) : (bm + bn) * bkb;
}

// T: operand type, TO: result type; BM x BN tile; WM x WN x WK wavefronts over rows, columns and the K of a stage
template <typename T, typename TO, int BM, int BN, int WM, int WN, int WK, int BKB, int S, bool DIRECT, int XF, int WF>
__global__ void __launch_bounds__(64 * WM * WN * WK) contract_float_kernel(const FArgs g) {
    constexpr int NT = 64 * WM * WN * WK, E = 16 / Elem<T>::size, SZ = Elem<T>::size, SO = Elem<TO>::size;
    constexpr int PPR = BKB / 16, SH = BKB == 64 ? 2 : (BKB == 128 ? 1 : 0);
    constexpr int MT = BM / WM >= 32 ? 32 : 16, MP = 64 / MT, AR = MT * MT / 64;  // matrix tile; its pieces of K and result registers
    constexpr int KK = BKB / (16 * MP), KKW = KK / WK;  // matrix steps per stage, and per wavefront
    constexpr int TM = BM / WM / MT, TN = BN / WN / MT;
    typedef typename std::conditional<MT == 32, v16f, v4f>::type acc_t;
    constexpr int XI = BM * PPR / NT, WI = BN * PPR / NT;
    constexpr bool KM = WF == F_KMAJOR, CONV = std::is_same<T, TO>::value && XF != F_ROWS;  // (or an fp32 product of aligned pieces)
    // a K-major W keeps its rows: the pad puts the four rows a transposing read meets (16 bits), or the two the halves of a
    // wavefront read (fp32), on distinct banks
    constexpr int WPITCH = BN * SZ + 32, KROWS = BKB / SZ, WCH = BN * SZ / 16;
    constexpr int STAGE = stage_bytes(BM, BN, BKB, SZ, KM);
    static_assert((BM * PPR) % NT == 0 && (BN * PPR) % NT == 0 && KK % WK == 0 && TM >= 1 && TN >= 1, "tile shape");
    static_assert((NT / PPR) % 16 == 0, "the rows of one thread share their swizzle");
    extern __shared__ __align__(16) char smem[];

    // every argument that stands in front of the first request is asked for here, in one batch (left alone the compiler loads
    // them where they are first used, one trip to memory behind the other)
    asm volatile("" ::"s"(g.chunk), "s"(g.total_tiles), "s"(g.order.tiles_m), "s"(g.order.tiles_n), "s"(g.order.rows), "s"(g.order.m_batch),
                 "s"(g.order.m_band), "s"(g.order.m_rows), "s"(g.order.m_last), "s"(g.order.shifts),
                 "s"(g.div_ohw.m), "s"(g.div_ohw.s), "s"(g.div_ow.m), "s"(g.div_ow.s),
                 "s"(g.x), "s"(g.w), "s"(g.bias), "s"(g.res), "s"(g.out), "s"(g.M), "s"(g.N), "s"(g.K), "s"(g.IC), "s"(g.KW), "s"(g.KH),
                 "s"(g.H), "s"(g.W), "s"(g.sy), "s"(g.sx), "s"(g.pt), "s"(g.pl), "s"(g.dy), "s"(g.dx), "s"(g.OHW), "s"(g.OW));
    asm volatile("" ::"s"(g.x_img), "s"(g.x_row), "s"(g.x_pix), "s"(g.x_bytes), "s"(g.ldw), "s"(g.w_bytes), "s"(g.x_batch),
                 "s"(g.w_batch), "s"(g.o_batch), "s"(g.ldo), "s"(g.o_bytes), "s"(g.ic_magic), "s"(g.kw_magic), "s"(g.bias_len), "s"(g.wide_out));
    const int lin = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u));
    if (lin >= g.total_tiles) return;
    int batch, tile_m, tile_n;
    g.order.tile(lin, batch, tile_m, tile_n);
    const int m_base = tile_m * BM, n_base = tile_n * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_k = wave % WK, wave_n = (wave / WK) % WN, wave_m = wave / (WK * WN);

    // ---- this thread's pieces: rows r0 + i * NT / PPR of X and of W, the same piece p of each (the swizzle repeats)
    const int r0 = tid / PPR, p0 = (tid % PPR) ^ ((r0 >> SH) & (PPR - 1));
    int32_t xb[XI], iy0[XI], ix0[XI];
#pragma unroll
    for (int i = 0; i < XI; i++) {
        const int m = m_base + r0 + i * (NT / PPR);
        const int img = div_magic(m, g.div_ohw), pos = m - img * g.OHW;
        const int oy = div_magic(pos, g.div_ow), ox = pos - oy * g.OW;
        iy0[i] = m < g.M ? oy * g.sy - g.pt : -0x40000000;
        ix0[i] = ox * g.sx - g.pl;
        xb[i] = (int32_t)((uint32_t)img * g.x_img + (uint32_t)(oy * g.sy - g.pt) * g.x_row + (uint32_t)ix0[i] * g.x_pix);
    }
    // position along K of this thread's piece in the stage that is fetched next: element kpos = tap * IC + ic
    int kpos = p0 * E, ic = kpos, ky = 0, kx = 0;  // (DIRECT keeps kpos alone)
    auto wrap = [&](int &c, int &y, int &x) {
        while (c >= g.IC && y < g.KH) {
            c -= g.IC;
            if (++x == g.KW) x = 0, y++;
        }
    };
    if constexpr (!DIRECT) wrap(ic, ky, kx);
    auto tap_off = [&](int i, int c, int y, int x) {  // offset of channel c of a tap of row i, or beyond the extent
        const int iy = iy0[i] + y * g.dy, ix = ix0[i] + x * g.dx;
        const bool in = (uint32_t)iy < (uint32_t)g.H && (uint32_t)ix < (uint32_t)g.W && y < g.KH;
        return in ? (uint32_t)xb[i] + (uint32_t)(y * g.dy) * g.x_row + (uint32_t)(x * g.dx) * g.x_pix + (uint32_t)(c * SZ) : kOob;
    };
    auto step_on = [&]() {
        kpos += PPR * E;
        ic += PPR * E;
        wrap(ic, ky, kx);
    };
    const int n0 = n_base + r0;

    acc_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < AR; r++) acc[i][j][r] = 0.f;

    const int h = lane / MT, lrow = lane % MT;

    // ---- what the epilogue needs: the bias of this lane's columns and the pieces of the residual.  Asked for in front of the
    // operands (behind the loop its trip to memory stands alone) where the loop's loads are counted; a loop whose loads stand
    // behind conditions would wait for it first (the 3-channel convolution of four images of 224 x 224: 7.7 -> 10.4 us).  NQ: register quads of a wavefront that has K to itself, of NB columns' worth
    constexpr int NQ = AR / 4 * TM * TN, NB = AR / 4 * TN;
    static_assert(WK == 1 || TM * TN == 1, "one sub-tile where K is shared");
    auto quad_col = [&](int u) {  // first column of quad u, within the tile
        return (wave_n * TN + u / (AR / 4) % TN) * MT + 4 * MP * (u % (AR / 4)) + 4 * h;
    };
    // where K is shared a thread finishes four columns of a row at a time: NP quads, of the same columns
    constexpr int QPR = BN / 4, EO = WK > 1 ? 4 : 16 / SO, OP = BN * SO + 16, OPPR = BN / EO, NP = (BM * OPPR + NT - 1) / NT;
    static_assert(WK == 1 || NT % QPR == 0, "a thread's quads share their columns");
    const __amdgpu_buffer_rsrc_t bres = rsrc(g.bias, g.bias != nullptr ? (uint32_t)(g.bias_len * SO) : 0u);
    const __amdgpu_buffer_rsrc_t ores = rsrc(g.out + (int64_t)batch * g.o_batch, g.o_bytes);
    const __amdgpu_buffer_rsrc_t rres = rsrc(g.res, g.res != nullptr ? g.o_bytes : 0u);
    uint32_t bias_bits[WK > 1 ? 1 : NB][4], off[NP];
    uint4 res[NP];
    auto ask_epilogue = [&] {
#pragma unroll
        for (int u = 0; u < (WK > 1 ? 1 : NB); u++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                bias_bits[u][e] = load_elem<SO>(bres, g.bias_len == 1 ? 0u : (uint32_t)((n_base + (WK > 1 ? tid % QPR * 4 : quad_col(u)) + e) * SO));
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int p = i * NT + tid, m = m_base + p / OPPR, n = n_base + (p % OPPR) * EO;
            off[i] = p < BM * OPPR && m < g.M && n < g.N ? (uint32_t)m * g.ldo + (uint32_t)(n * SO) : kOob;
            res[i] = load_piece<EO * SO>(rres, g.wide_out ? off[i] : kOob);
        }
    };
    constexpr bool AHEAD = DIRECT || XF == F_ROWS;
    if constexpr (AHEAD) ask_epilogue();
    // this wavefront's operands of a stage; `between` runs while they are on their way, then they are multiplied
    auto compute = [&](const char *st, auto between) {
        uint4 xf[KKW][TM], wf[KKW][TN];
#pragma unroll
        for (int k = 0; k < KKW; k++) {
            const int slot = (((wave_k * KKW + k) * MP + h) ^ ((lrow >> SH) & (PPR - 1))) * 16;
#pragma unroll
            for (int i = 0; i < TM; i++)
                xf[k][i] = *reinterpret_cast<const uint4 *>(st + ((wave_m * TM + i) * MT + lrow) * BKB + slot);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                if constexpr (!KM) {
                    wf[k][j] = *reinterpret_cast<const uint4 *>(st + BM * BKB + ((wave_n * TN + j) * MT + lrow) * BKB + slot);
                } else if constexpr (SZ == 2) {
                    // 16-lane group q covers columns 16 (q & 1) .., k group q / 2; its lane s points at row s / 4, columns 4 (s % 4)
                    const char *p = st + BM * BKB + ((wave_k * KKW + k) * 16 + 8 * (lane >> 5) + ((lane & 15) >> 2)) * WPITCH +
                                    ((wave_n * TN + j) * 32 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
                    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)p);
                    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(p + 4 * WPITCH));
                    const v8s both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                    wf[k][j] = __builtin_bit_cast(uint4, both);
                } else {
                    const char *p = st + BM * BKB + ((wave_k * KKW + k) * 8 + 4 * h) * WPITCH + ((wave_n * TN + j) * 32 + lrow) * 4;
                    wf[k][j] = make_uint4(*reinterpret_cast<const uint32_t *>(p), *reinterpret_cast<const uint32_t *>(p + WPITCH),
                                          *reinterpret_cast<const uint32_t *>(p + 2 * WPITCH), *reinterpret_cast<const uint32_t *>(p + 3 * WPITCH));
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        between();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < KKW; k++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = multiply<T>(wf[k][j], xf[k][i], acc[i][j]);
    };
    auto nothing = [] {};

    const int run = g.KW * g.IC, ppr = (run + E - 1) / E;  // F_RUNS: elements and pieces of a kernel row
    const int nk = XF == F_RUNS ? (g.KH * ppr + PPR - 1) / PPR : (g.K + PPR * E - 1) / (PPR * E);
    const char *xp = g.x + (int64_t)batch * g.x_batch, *wp = g.w + (int64_t)batch * g.w_batch;
    if constexpr (DIRECT) {
        constexpr int NLA = XI + WI;
        const v4i xres = rsrc_words(xp, g.x_bytes), wres = rsrc_words(wp, g.w_bytes);
        const uint32_t lds0 =
            (uint32_t) reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem) + (uint32_t)(wave * 1024);
        // A wavefront that has its SIMD to itself issues an instruction every 7 clocks or so, and the loop is a few dozen of
        // them beside eight matrix instructions: what a request costs is what the loop takes.  So the place of a piece among the
        // taps comes from two multiplications, and W's rows advance by the scalar offset alone.  F_TAPS makes the taps that a
        // row meets inside the image a bit each in front of the loop: 1400 clocks there, for fewer instructions per request.
        uint32_t wo[WI], my[XI], mx[XI];
        if constexpr (XF == F_TAPS) {
#pragma unroll
            for (int i = 0; i < XI; i++) {
                my[i] = mx[i] = 0;
                for (int y = 0; y < g.KH; y++) my[i] |= (uint32_t)(iy0[i] + y * g.dy) < (uint32_t)g.H ? 1u << y : 0u;  // uniform trip count
                for (int x = 0; x < g.KW; x++) mx[i] |= (uint32_t)(ix0[i] + x * g.dx) < (uint32_t)g.W ? 1u << x : 0u;
            }
        }
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int n = n0 + i * (NT / PPR);
            wo[i] = n < g.N ? (uint32_t)n * g.ldw + (uint32_t)(p0 * 16) : kOob;
        }
        const uint32_t y_step = (uint32_t)g.dy * g.x_row, x_step = (uint32_t)g.dx * g.x_pix;
        int asked = 0;  // stages requested so far
        auto request = [&](int buf) {  // the next stage into buffer `buf`; beyond K there is no tap, and W is zeros
            const uint32_t d = lds0 + (uint32_t)(buf * STAGE);
            const int tap = (int)__umulhi((uint32_t)kpos, g.ic_magic), c = kpos - (int)__umul24((uint32_t)tap, (uint32_t)g.IC);
            const int y = (int)(__umul24((uint32_t)tap, g.kw_magic) >> 16), x = tap - (int)__umul24((uint32_t)y, (uint32_t)g.KW);
            const uint32_t t = __umul24((uint32_t)y, y_step) + __umul24((uint32_t)x, x_step) + (uint32_t)(c * SZ);
            const bool partial = (asked + 1) * PPR * E > g.K;  // uniform: the last stage ends beyond K
            if constexpr (XF == F_TAPS) {  // (beyond the last tap: bits that are not set; 32 rows of taps are whole stages)
#pragma unroll
                for (int i = 0; i < XI; i++) {
                    const uint32_t in = (uint32_t)(__builtin_amdgcn_sbfe((int)my[i], y, 1) & __builtin_amdgcn_sbfe((int)mx[i], x, 1));
                    load16_to_lds(xres, d + i * NT * 16, (in & ((uint32_t)xb[i] + t)) | (~in & kOob), 0);
                }
            } else {
                int yd = y * g.dy;
                const int xd = x * g.dx;
                if (partial) {
                    yd = kpos < g.K ? yd : 0x20000000;  // no tap: outside the image
                    asm volatile("" : "+v"(yd));  // (a branch, not a select in every stage)
                }
#pragma unroll
                for (int i = 0; i < XI; i++) {
                    const bool in = (uint32_t)(iy0[i] + yd) < (uint32_t)g.H && (uint32_t)(ix0[i] + xd) < (uint32_t)g.W;
                    const uint32_t off = in ? (uint32_t)xb[i] + t : kOob;
                    load16_to_lds(xres, d + i * NT * 16, off, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < WI; i++) {
                uint32_t off = wo[i];
                if (partial) {
                    off = kpos < g.K ? off : kOob;
                    asm volatile("" : "+v"(off));  // (a branch, not a select in every stage)
                }
                load16_to_lds(wres, d + BM * BKB + i * NT * 16, off, (uint32_t)(asked * BKB));
            }
            kpos += PPR * E;
            asked++;
        };
#pragma unroll
        for (int d = 0; d < S - 1; d++)
            if (d < nk) request(d);  // uniform
        // this thread's part of a stage has landed when at most the later stages are outstanding; the barrier extends that to
        // the block, and says that every wavefront is done with the buffer the next request overwrites
        auto meet = [&]() {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        int step = 0;
        while (step + S - 1 < nk) {  // unrolled over the ring: a stage's place is a constant
#pragma unroll
            for (int d = 0; d < S; d++) {
                if (step + S - 1 < nk) {  // uniform
                    wait_vmcnt<(S - 2) * NLA>();
                    meet();
                    compute(smem + d * STAGE, [&] { request((d + S - 1) % S); });
                    step++;
                }
            }
        }
        int cur = step % S;
        // the last S - 1 stages: nothing is left to request
        auto drain = [&](auto self, auto left) {
            constexpr int R = decltype(left)::value;
            if constexpr (R > 0) {
                if (nk - step >= R) {  // uniform
                    wait_vmcnt<(R - 1) * NLA>();
                    meet();
                    compute(smem + cur * STAGE, nothing);
                    cur = cur + 1 == S ? 0 : cur + 1;
                    step++;
                }
                self(self, std::integral_constant<int, R - 1>{});
            }
        };
        drain(drain, std::integral_constant<int, S - 1>{});
        __syncthreads();
    } else {
        const __amdgpu_buffer_rsrc_t xres = rsrc(xp, g.x_bytes), wres = rsrc(wp, g.w_bytes);
        struct Set {
            uint4 x[XI], w[WI];
        };
        auto pack = [](const uint32_t *v) {
            if constexpr (SZ == 2)
                return make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
            else
                return make_uint4(v[0], v[1], v[2], v[3]);
        };
        auto keep = [](uint4 v, int lo, int hi) { return keep_elems<SZ>(v, lo, hi); };
        // elements lo .. hi - 1 of the piece at byte `off`: one load where the whole piece lies inside the operand, else
        // element by element
        auto load_run = [&](const char *base, __amdgpu_buffer_rsrc_t res, uint32_t bytes, int64_t off, int lo, int hi) {
            uint4 v = make_uint4(0, 0, 0, 0);
            if (lo >= hi) return v;
            if (off >= 0 && off + 16 <= (int64_t)bytes) {
                __builtin_memcpy(&v, base + off, 16);
            } else {
                uint32_t e[E];
#pragma unroll
                for (int k = 0; k < E; k++) e[k] = load_elem<SZ>(res, k >= lo && k < hi ? (uint32_t)(off + k * SZ) : kOob);
                return pack(e);
            }
            return lo > 0 || hi < E ? keep(v, lo, hi) : v;
        };
        // F_ROWS and F_KMAJOR walk K by a scalar offset; a row beyond the operand is its last row (its results are not stored).
        // The stage that reaches beyond K, and whole operands of less than a piece, take load_run.
        uint32_t xo[XI], wo[WI];
        int back[WI];  // F_KMAJOR: elements by which the piece that would reach beyond a row lies further in front
#pragma unroll
        for (int i = 0; i < XI; i++) xo[i] = XF == F_ROWS ? (uint32_t)min(m_base + r0 + i * (NT / PPR), g.M - 1) * g.x_pix + (uint32_t)(p0 * 16) : 0u;
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int id = i * NT + tid, n = n_base + (id % WCH) * E;
            back[i] = KM ? min(max(n + E - g.N, 0), n) : 0;
            wo[i] = KM ? (uint32_t)(id / WCH) * g.ldw + (uint32_t)((n - back[i]) * SZ)
                       : (uint32_t)min(n0 + i * (NT / PPR), g.N - 1) * g.ldw + (uint32_t)(p0 * 16);
        }
        const bool edge = KM && n_base + BN > g.N;  // uniform
        auto forward = [](uint4 v, int by) { return move_elems<SZ>(v, by); };
        const bool tiny = (XF == F_ROWS && g.x_bytes < 16) || g.w_bytes < 16 || (KM && g.N < E);
        int stage_k = 0;            // first element (F_RUNS: first piece) of the stage that is fetched next
        auto fetch = [&](Set &r) {
            if constexpr (XF == F_RUNS) {
                const int pi = stage_k + p0, y = div_magic(pi, g.div_ppr), q = pi - y * ppr, e0 = q * E;
#pragma unroll
                for (int i = 0; i < XI; i++) {
                    const bool in = (uint32_t)(iy0[i] + y * g.dy) < (uint32_t)g.H && y < g.KH;
                    const int lo = min(max(-ix0[i], 0), g.KW) * g.IC - e0, hi = min(g.W - ix0[i], g.KW) * g.IC - e0;
                    r.x[i] = load_run(xp, xres, g.x_bytes, (int64_t)xb[i] + (int64_t)(y * g.dy) * g.x_row + e0 * SZ, lo, in ? hi : INT32_MIN);
                }
#pragma unroll
                for (int i = 0; i < WI; i++) {
                    const int n = n0 + i * (NT / PPR);
                    r.w[i] = load_run(wp, wres, g.w_bytes, (int64_t)n * g.ldw + (int64_t)(y * run + e0) * SZ, 0,
                                      n < g.N && y < g.KH ? run - e0 : 0);
                }
            } else if constexpr (XF == F_ELEMS) {
#pragma unroll
                for (int i = 0; i < XI; i++) {
                    uint32_t v[E];
                    int c = ic, y = ky, x = kx;
#pragma unroll
                    for (int e = 0; e < E; e++) {
                        v[e] = load_elem<SZ>(xres, tap_off(i, c, y, x));
                        c++;
                        if (c == g.IC) {
                            c = 0;
                            if (++x == g.KW) x = 0, y++;
                        }
                    }
                    r.x[i] = pack(v);
                }
#pragma unroll
                for (int i = 0; i < WI; i++) {
                    const int n = n0 + i * (NT / PPR);
                    uint32_t v[E];
#pragma unroll
                    for (int e = 0; e < E; e++)
                        v[e] = load_elem<SZ>(wres, n < g.N && kpos + e < g.K ? (uint32_t)n * g.ldw + (uint32_t)((kpos + e) * SZ) : kOob);
                    r.w[i] = pack(v);
                }
            } else {  // the stage that reaches beyond K, and operands of less than a piece
#pragma unroll
                for (int i = 0; i < XI; i++)
                    r.x[i] = load_run(xp, xres, g.x_bytes, (int64_t)stage_k * SZ + xo[i], 0, g.K - stage_k - p0 * E);
#pragma unroll
                for (int i = 0; i < WI; i++) {
                    if constexpr (KM) {
                        const int id = i * NT + tid, k = stage_k + id / WCH, n = n_base + (id % WCH) * E;
                        r.w[i] = load_run(wp, wres, g.w_bytes, (int64_t)k * g.ldw + (int64_t)(n - back[i]) * SZ, 0, k < g.K && n < g.N ? E : 0);
                    } else {
                        r.w[i] = load_run(wp, wres, g.w_bytes, (int64_t)stage_k * SZ + wo[i], 0, g.K - stage_k - p0 * E);
                    }
                }
            }
            if constexpr (XF == F_ELEMS) step_on();
            stage_k += XF == F_RUNS ? PPR : PPR * E;
        };
        auto store = [&](char *st, const Set &r) {
#pragma unroll
            for (int i = 0; i < XI; i++) *reinterpret_cast<uint4 *>(st + (i * NT + tid) * 16) = r.x[i];
#pragma unroll
            for (int i = 0; i < WI; i++) {
                const int id = i * NT + tid;
                uint4 v = r.w[i];
                if (edge) v = forward(v, back[i]);
                *reinterpret_cast<uint4 *>(st + BM * BKB + (KM ? (id / WCH) * WPITCH + (id % WCH) * 16 : id * 16)) = v;
            }
        };
        // S register sets, two stage buffers: stage s passes through set s % S and buffer s % 2, and is asked for S stages
        // before it is stored
        static_assert(S % 2 == 0, "a set meets one buffer");
        Set r[S];
        if constexpr (XF == F_ROWS) {
            // The whole stages without a condition around a load -- behind one the compiler no longer knows how many loads are
            // on their way, and waits for all of them; requests beyond the last whole stage ask for it again.
            const int nkw = tiny ? 0 : g.K / (PPR * E);
            auto ask = [&](Set &v, int stage) {
                stage = min(stage, nkw - 1);
                const char *xa = xp + (int64_t)stage * BKB, *wa = wp + (int64_t)stage * (KM ? (int64_t)KROWS * g.ldw : BKB);
#pragma unroll
                for (int i = 0; i < XI; i++) __builtin_memcpy(&v.x[i], xa + xo[i], 16);
#pragma unroll
                for (int i = 0; i < WI; i++) __builtin_memcpy(&v.w[i], wa + wo[i], 16);
            };
            if (nkw > 0) {  // uniform
#pragma unroll
                for (int d = 0; d < S; d++) ask(r[d], d);
                store(smem, r[0]);
                ask(r[0], S);
                __syncthreads();
                int step = 0;
                for (; step + S <= nkw; step += S) {
#pragma unroll
                    for (int d = 0; d < S; d++) {
                        store(smem + ((d + 1) & 1) * STAGE, r[(d + 1) % S]);
                        ask(r[(d + 1) % S], step + d + 1 + S);
                        compute(smem + (d & 1) * STAGE, nothing);
                        __syncthreads();
                    }
                }
#pragma unroll
                for (int d = 0; d + 1 < S; d++) {
                    if (step + d < nkw) {  // uniform
                        store(smem + ((d + 1) & 1) * STAGE, r[(d + 1) % S]);
                        compute(smem + (d & 1) * STAGE, nothing);
                        __syncthreads();
                    }
                }
            }
            stage_k = nkw * PPR * E;
            while (stage_k < g.K) {  // (tiny operands: all of their stages)
                fetch(r[0]);
                store(smem, r[0]);
                __syncthreads();
                compute(smem, nothing);
                __syncthreads();
            }
        } else {
#pragma unroll
            for (int d = 0; d < S; d++)
                if (d < nk) fetch(r[d]);
            store(smem, r[0]);
            if (S < nk) fetch(r[0]);
            __syncthreads();
            for (int step = 0; step < nk; step += S) {
#pragma unroll
                for (int d = 0; d < S; d++) {
                    if (step + d < nk) {  // uniform
                        if (step + d + 1 < nk) store(smem + ((d + 1) & 1) * STAGE, r[(d + 1) % S]);
                        if (step + d + 1 + S < nk) fetch(r[(d + 1) % S]);
                        compute(smem + (d & 1) * STAGE, nothing);
                        __syncthreads();
                    }
                }
            }
        }
    }

    if constexpr (!AHEAD) ask_epilogue();
    auto finish = [&](uint32_t bits, uint32_t res_bits) { return finish_bits<TO>(g, bits, res_bits); };
    auto finish_piece = [&](uint4 v, uint4 r) { return finish_words<TO, EO * SO / 4>(g, v, r); };
    // piece `v` of the result, column n of the tile's row at byte `at` of the output
    auto put_piece = [&](uint4 v, uint4 r, uint32_t at, int n) {
        if (g.wide_out) {  // uniform
            if (g.res != nullptr || g.has_clamp) v = finish_piece(v, r);
            store_piece<EO * SO>(ores, at, v);
            return;
        }
        // rows that are no whole pieces: a piece at any element's address, through the L2, which joins the lines that rows
        // share; the end of a row element by element
        if (at == kOob) return;
        if (n + EO <= g.N) {
            if (g.res != nullptr) __builtin_memcpy(&r, g.res + at, EO * SO);
            if (g.res != nullptr || g.has_clamp) v = finish_piece(v, r);
            __builtin_memcpy(g.out + (int64_t)batch * g.o_batch + at, &v, EO * SO);
            return;
        }
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < EO; e++) {
            if (e >= g.N - n) break;
            const uint32_t to = at + (uint32_t)(e * SO);
            const uint32_t x = finish(SO == 2 ? (w[e / 2] >> (16 * (e & 1))) & 0xffffu : w[e % 4], g.res != nullptr ? load_elem<SO>(rres, to) : 0u);
            if constexpr (SO == 2) __builtin_amdgcn_raw_buffer_store_b16((short)x, ores, (int)to, 0, 0);
            else __builtin_amdgcn_raw_buffer_store_b32((int)x, ores, (int)to, 0, 0);
        }
    };
    // A tap outside the image contributes nothing (conv2d.comp:40-116), but here it is a zero times its weight: no change to
    // a finite sum, NaN where the weight is infinite or NaN.  So a position with such taps whose sum came out as NaN is
    // summed again over the taps inside the image, by the lane that holds it.  One comparison per two results where
    // none is.
    auto late_args = [] {  // (the arguments again, from where the launch left them: held from the start they took 30 scalar registers)
        typedef const FArgs __attribute__((address_space(4))) *args_t;
        args_t again = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(again));
        return (const FArgs *)again;
    };

    // ---- K shared: every wavefront leaves its share of the tile in shared memory, a lane holding row m = lane % MT of a
    // sub-tile and, per register quad q, columns 4 MP q + 4 * (lane / MT) ..; each thread then adds the shares of four columns
    // of a row, in ascending order of K, finishes them and stores them -- one trip through shared memory for sum and
    // layout.  A wavefront alone on its SIMD is bound by the instructions it issues, in front of the loop and behind it as well
    // (4 x 14 x 14 x 256 -> 256, 3 x 3: of 14 600 clocks 4 400 in front of the first product and 2 200 behind the last): with
    // this, the arguments in one batch and no bit masks of the taps, a network of twelve such convolutions over four images
    // of 224 x 224 takes 81.9 us, 87.9 before (fp16), one image of 112 x 208 57.4, 60.4 before (fp32).
    if constexpr (WK > 1) {
        constexpr int RP = BN + 4;  // floats per row of a share
        float *shares = reinterpret_cast<float *>(smem);
#pragma unroll
        for (int q = 0; q < AR / 4; q++)
            *reinterpret_cast<v4f *>(shares + ((wave_k * BM + wave_m * MT + lrow) * RP + wave_n * MT + 4 * MP * q + 4 * h)) =
                v4f{acc[0][0][4 * q], acc[0][0][4 * q + 1], acc[0][0][4 * q + 2], acc[0][0][4 * q + 3]};
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int p = i * NT + tid, r = p / QPR, n = n_base + p % QPR * 4;
            if (BM * QPR % NT != 0 && p >= BM * QPR) break;
            const float *at = shares + r * RP + p % QPR * 4;
            v4f own = *reinterpret_cast<const v4f *>(at);
#pragma unroll
            for (int k = 1; k < WK; k++) own += *reinterpret_cast<const v4f *>(at + k * BM * RP);
            uint32_t v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float sum = own[e];
                if (g.bias != nullptr) sum += Elem<TO>::get(bias_bits[0][e]);  // uniform (-0 + 0 would lose its sign)
                v[e] = Elem<TO>::put(sum, false);
            }
            if constexpr (CONV) {
                const bool nan = __builtin_isunordered(own[0], own[1]) || __builtin_isunordered(own[2], own[3]);
                if (__builtin_expect(g.border && nan, 0)) {
                    const FArgs &late = *late_args();
#pragma clang loop unroll(disable)
                    for (int e = 0; e < 4; e++) {
                        const uint32_t bits = e == 0 ? v[0] : (e == 1 ? v[1] : (e == 2 ? v[2] : v[3]));
                        float sum = Elem<TO>::get(bits);
                        if (sum == sum || m_base + r >= late.M || n + e >= late.N || !sum_inside<T, TO>(late, m_base + r, n + e, sum)) continue;
                        const uint32_t again = Elem<TO>::put(sum, false);
#pragma unroll
                        for (int k = 0; k < 4; k++) v[k] = k == e ? again : v[k];
                    }
                }
            }
            put_piece(SO == 2 ? make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), 0, 0) : make_uint4(v[0], v[1], v[2], v[3]), res[i], off[i], n);
        }
        return;
    }

    // ---- bias and rounding, then through shared memory (the same lanes' layout); the stores below write whole runs of a row
    bool nan = false;
#pragma unroll
    for (int u = 0; u < NQ; u++) {
        const int i = u / (AR / 4 * TN);
        const acc_t &t = acc[i][u / (AR / 4) % TN];
        const v4f own = v4f{t[u % (AR / 4) * 4], t[u % (AR / 4) * 4 + 1], t[u % (AR / 4) * 4 + 2], t[u % (AR / 4) * 4 + 3]};
        char *row = smem + ((wave_m * TM + i) * MT + lrow) * OP + quad_col(u) * SO;
        uint32_t v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float sum = own[e];
            if (g.bias != nullptr) sum += Elem<TO>::get(bias_bits[u % NB][e]);  // uniform
            v[e] = Elem<TO>::put(sum, false);
        }
        if constexpr (SO == 2) *reinterpret_cast<uint2 *>(row) = make_uint2(v[0] | (v[1] << 16), v[2] | (v[3] << 16));
        else *reinterpret_cast<uint4 *>(row) = make_uint4(v[0], v[1], v[2], v[3]);
        if constexpr (CONV) nan |= __builtin_isunordered(own[0], own[1]) || __builtin_isunordered(own[2], own[3]);
    }
    if constexpr (CONV) {
        if (__builtin_expect(g.border && nan, 0)) {
            const FArgs &late = *late_args();
#pragma clang loop unroll(disable)
            for (int q = 0; q < 4 * NQ; q++) {
                const int u = q / 4, r = (wave_m * TM + u / (AR / 4 * TN)) * MT + lrow, c = quad_col(u) + q % 4;
                char *at = smem + r * OP + c * SO;
                uint32_t v = 0;
                __builtin_memcpy(&v, at, SO);
                float sum = Elem<TO>::get(v);
                if (sum == sum || m_base + r >= late.M || n_base + c >= late.N || !sum_inside<T, TO>(late, m_base + r, n_base + c, sum)) continue;
                v = Elem<TO>::put(sum, false);
                __builtin_memcpy(at, &v, SO);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int p = i * NT + tid;
        if (BM * OPPR % NT != 0 && p >= BM * OPPR) break;
        put_piece(*reinterpret_cast<const uint4 *>(smem + (p / OPPR) * OP + (p % OPPR) * 16), res[i], off[i], n_base + (p % OPPR) * EO);
    }
}

// A convolution whose K is a few pieces in all (F_RUNS, up to 16 of them: the three channels of an image): a wavefront has 32
// positions and 32 NJ channels, its operands come from memory as matrix operands, each lane its own pieces, without
// stages or barriers.  The staged form spends its time on one or two stages' conditions (660 vector instructions per
// wavefront and 32 x 32 results, here half of that per 32 x 64); what is left is the trip of the operands and the results' way out.
template <typename T, int NJ, int STEPS>
__global__ void __launch_bounds__(256) conv_runs_float_kernel(const FArgs g) {
    constexpr int E = 16 / Elem<T>::size, SZ = Elem<T>::size, OP = NJ * 32 * SZ + 16, OPPR = NJ * 32 * SZ / 16;
    __shared__ __align__(16) char smem[4 * 32 * OP];
    asm volatile("" ::"s"(g.chunk), "s"(g.total_tiles), "s"(g.div_ohw.m), "s"(g.div_ohw.s), "s"(g.div_ow.m), "s"(g.div_ow.s),
                 "s"(g.div_ppr.m), "s"(g.div_ppr.s), "s"(g.x), "s"(g.w), "s"(g.bias), "s"(g.res), "s"(g.out), "s"(g.M), "s"(g.N), "s"(g.IC),
                 "s"(g.KW), "s"(g.KH), "s"(g.H), "s"(g.W), "s"(g.sy), "s"(g.sx), "s"(g.pt), "s"(g.pl), "s"(g.dy), "s"(g.OHW), "s"(g.OW),
                 "s"(g.x_img), "s"(g.x_row), "s"(g.x_pix), "s"(g.x_bytes), "s"(g.ldw), "s"(g.w_bytes), "s"(g.ldo), "s"(g.o_bytes),
                 "s"(g.bias_len), "s"(g.border), "s"(g.has_clamp));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int block = (int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u), m0 = (block * 4 + wave) * 32, n0 = (int)blockIdx.y * (32 * NJ);
    if (block >= g.total_tiles || m0 >= g.M) return;
    const int h = lane >> 5, lrow = lane & 31, m = min(m0 + lrow, g.M - 1);
    const int img = div_magic(m, g.div_ohw), pos = m - img * g.OHW, oy = div_magic(pos, g.div_ow), ox = pos - oy * g.OW;
    const int iy0 = oy * g.sy - g.pt, ix0 = ox * g.sx - g.pl;
    const int xb = (int)((uint32_t)img * g.x_img + (uint32_t)iy0 * g.x_row + (uint32_t)ix0 * g.x_pix);
    const int run = g.KW * g.IC, ppr = (run + E - 1) / E, pieces = g.KH * ppr;
    const bool inside = iy0 >= 0 && ix0 >= 0 && iy0 + (g.KH - 1) * g.dy < g.H && ix0 + g.KW <= g.W;

    // every piece is asked for at its place or, where it would reach beyond the operand, as its last 16 bytes
    uint4 x[STEPS], w[STEPS][NJ];
    int x_off[STEPS], part[STEPS];  // part: elements of this half's piece that belong to its run
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
        const int p = 2 * s + h, y = div_magic(p, g.div_ppr), e0 = (p - y * ppr) * E;
        part[s] = p < pieces ? run - e0 : 0;
        x_off[s] = (int)((uint32_t)xb + (uint32_t)(y * g.dy) * g.x_row + (uint32_t)(e0 * SZ));
        const uint32_t at = (uint32_t)min(max(p < pieces ? x_off[s] : 0, 0), (int)g.x_bytes - 16);
        __builtin_memcpy(&x[s], g.x + at, 16);
        const uint32_t w_at = p < pieces ? (uint32_t)((y * run + e0) * SZ) : 0u;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const uint32_t off = (uint32_t)min(n0 + j * 32 + lrow, g.N - 1) * g.ldw + w_at;
            __builtin_memcpy(&w[s][j], g.w + min(off, g.w_bytes - 16), 16);
        }
    }
    // four columns' bias at a time (N is a multiple of four: whole pieces of the result)
    uint4 bias[NJ][4];
    if (g.bias_len != 1) {  // uniform
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                __builtin_memcpy(&bias[j][q], g.bias + (uint32_t)(min(n0 + j * 32 + 8 * q + 4 * h, g.N - 4) * SZ), 4 * SZ);
    } else {
        uint32_t v = 0;
        __builtin_memcpy(&v, g.bias, SZ);
        if constexpr (SZ == 2) v *= 0x10001u;
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) bias[j][q] = make_uint4(v, v, v, v);
    }

    v16f acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[j][r] = 0.f;
    const bool all_inside = __all(inside);
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
        const int p = 2 * s + h, y = div_magic(p, g.div_ppr), e0 = (p - y * ppr) * E;
        const int beyond = x_off[s] - ((int)g.x_bytes - 16);
        if (__any(p < pieces && beyond > 0)) x[s] = move_elems<SZ>(x[s], min(max(beyond, 0) / SZ, E));  // (E: nothing is kept of it)
        const uint4 mask = first_elems<SZ>(part[s]);
        if (all_inside) {  // uniform
            x[s] = both(x[s], mask);
        } else {
            const int lo = min(max(-ix0, 0), g.KW) * g.IC - e0;
            const int hi = p < pieces && (uint32_t)(iy0 + y * g.dy) < (uint32_t)g.H ? min(g.W - ix0, g.KW) * g.IC - e0 : 0;
            if (__any(x_off[s] < 0 && lo < hi)) {  // in front of the operand: element by element
                const __amdgpu_buffer_rsrc_t xres = rsrc(g.x, g.x_bytes);
                uint32_t v[E];
#pragma unroll
                for (int e = 0; e < E; e++) v[e] = load_elem<SZ>(xres, e >= lo && e < hi ? (uint32_t)(x_off[s] + e * SZ) : kOob);
                if constexpr (SZ == 2) x[s] = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
                else x[s] = make_uint4(v[0], v[1], v[2], v[3]);
            }
            x[s] = keep_elems<SZ>(x[s], lo, hi);
        }
        const uint32_t w_at = p < pieces ? (uint32_t)((y * run + e0) * SZ) : 0u;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int over = (int)((uint32_t)min(n0 + j * 32 + lrow, g.N - 1) * g.ldw + w_at) - ((int)g.w_bytes - 16);
            if (__any(over > 0)) w[s][j] = move_elems<SZ>(w[s][j], max(over, 0) / SZ);
            acc[j] = multiply<T>(both(w[s][j], mask), x[s], acc[j]);
        }
    }

    // bias and rounding; the results through this wavefront's rows of shared memory, so that they leave as runs of a row
    char *rows = smem + wave * (32 * OP);
    bool nan = false;
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            char *at = rows + lrow * OP + (j * 32 + 8 * q + 4 * h) * SZ;
            uint32_t v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t *bw = &bias[j][q].x;
                v[e] = Elem<T>::put(acc[j][4 * q + e] + Elem<T>::get(SZ == 2 ? (bw[e / 2] >> (16 * (e & 1))) & 0xffffu : bw[e]), false);
            }
            if constexpr (SZ == 2) *reinterpret_cast<uint2 *>(at) = make_uint2(v[0] | (v[1] << 16), v[2] | (v[3] << 16));
            else *reinterpret_cast<uint4 *>(at) = make_uint4(v[0], v[1], v[2], v[3]);
            nan |= __builtin_isunordered(acc[j][4 * q], acc[j][4 * q + 1]) || __builtin_isunordered(acc[j][4 * q + 2], acc[j][4 * q + 3]);
        }
    if (__builtin_expect(g.border && nan, 0)) {  // taps outside the image, as above
#pragma clang loop unroll(disable)
        for (int q = 0; q < 16 * NJ; q++) {
            const int c = q / 16 * 32 + q % 16 / 4 * 8 + 4 * h + q % 4;
            char *at = rows + lrow * OP + c * SZ;
            uint32_t v = 0;
            __builtin_memcpy(&v, at, SZ);
            float sum = Elem<T>::get(v);
            if (sum == sum || m0 + lrow >= g.M || n0 + c >= g.N || !sum_inside<T, T>(g, m0 + lrow, n0 + c, sum)) continue;
            v = Elem<T>::put(sum, false);
            __builtin_memcpy(at, &v, SZ);
        }
    }
    __builtin_amdgcn_wave_barrier();  // a wavefront's own rows: its shared-memory accesses complete in order
    const __amdgpu_buffer_rsrc_t ores = rsrc(g.out, g.o_bytes);
#pragma unroll
    for (int i = 0; i < OPPR / 2; i++) {
        const int p = i * 64 + lane, r = p / OPPR, n = n0 + p % OPPR * E;
        uint4 v = *reinterpret_cast<const uint4 *>(rows + r * OP + p % OPPR * 16);
        if (g.has_clamp) v = finish_words<T, 4>(g, v, v);  // uniform
        store_piece<16>(ores, m0 + r < g.M && n < g.N ? (uint32_t)(m0 + r) * g.ldo + (uint32_t)(n * SZ) : kOob, v);
    }
}

template <typename T, int NJ>
int launch_runs(FArgs &g, int steps, hipStream_t s) {
    g.total_tiles = (g.M + 127) / 128;
    g.chunk = (g.total_tiles + 7) / 8;
    const dim3 grid((unsigned)(g.chunk * 8), (unsigned)((g.N + 32 * NJ - 1) / (32 * NJ)));
    if (steps <= 3) conv_runs_float_kernel<T, NJ, 3><<<grid, dim3(256), 0, s>>>(g);
    else if (steps <= 5) conv_runs_float_kernel<T, NJ, 5><<<grid, dim3(256), 0, s>>>(g);
    else conv_runs_float_kernel<T, NJ, 8><<<grid, dim3(256), 0, s>>>(g);
    MLEL_TRY(check_launch("floating-point convolution of few taps"));
    return 1;
}

template <typename T, typename TO, int BM, int BN, int WM, int WN, int WK, int BKB, int S, bool DIRECT, int XF, int WF>
int launch_tile(FArgs &g, int64_t batches, hipStream_t s) {
    constexpr int SO = Elem<TO>::size;
    constexpr size_t operands = (size_t)(DIRECT ? S : 2) * stage_bytes(BM, BN, BKB, Elem<T>::size, WF == F_KMAJOR), result = (size_t)BM * (BN * SO + 16);
    constexpr size_t shares = WK > 1 ? (size_t)WK * BM * (BN + 4) * 4 : 0;
    constexpr size_t sm = std::max(operands, std::max(result, shares));
    static_assert(sm <= 160 * 1024, "shared memory of a compute unit");
    const int64_t tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
    const int64_t total = tiles_m * tiles_n * batches;
    MLEL_REQUIRE(total < (int64_t(1) << 30), MLEL_ERR_LIMIT, "contraction: %lld tiles", (long long)total);
    g.total_tiles = (int)total;
    g.chunk = (int)((total + 7) / 8);
    // (the rows of a convolution's tile meet the same pixels tap after tap)
    g.order = make_tile_order(tiles_m, tiles_n, g.chunk, (int64_t)BM * g.IC * g.sy * g.sx, (int64_t)BN * g.K);
    g.div_ppr = make_div_magic((uint32_t)((g.KW * (int64_t)g.IC * Elem<T>::size + 15) / 16));
    auto kernel = contract_float_kernel<T, TO, BM, BN, WM, WN, WK, BKB, S, DIRECT, XF, WF>;
    static const bool raised = sm <= 48 * 1024 || hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm) == hipSuccess;
    (void)raised;
    kernel<<<dim3((unsigned)(g.chunk * 8)), dim3(64 * WM * WN * WK), sm, s>>>(g);
    MLEL_TRY(check_launch("floating-point contraction"));
    return 1;
}

// Tile choice.  128 x 128 from two tiles per compute unit on; 64 x 64 from half a tile per compute unit on; below that
// 32 x 32 with the wavefronts sharing K, and 16 x 16 where even those leave half of the machine idle: the time is then the
// chain of one block's products, four times shorter (fp32 convolutions, 7 x 13 x 96: 11.2 -> 5 us; a network of them, one image
// of 112 x 208: 99 -> 74 us).  The ring needs no more than three stages: eight, for the blocks that have a compute unit to
// themselves, changed nothing.
template <typename T, typename TO, bool DIRECT, int XF, int WF>
int launch_shape(mlel_ctx *ctx, FArgs &g, int64_t batches, hipStream_t s) {
    const int64_t cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
    auto tiles = [&](int bm, int bn) { return (int64_t)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn) * batches; };
    if constexpr (DIRECT) {
        // the taps as bits where the loop is long: against the comparisons, over some 600 convolutions and products, fp32 took
        // 1.02-1.06 of the time up to K = 128, 1.00 at 512, 0.94-0.98 to 1024, 0.92 to 2048, 0.85 beyond 4096 (K = 11760, 16 channels over
        // four of 2 x 189: 36.7 -> 30.5 us); the halves 1.03-1.14 up to 4096, 0.96-0.98 beyond (K = 21168, 47 channels over five of
        // 37 x 16: 41.9 -> 35.8)
        if constexpr (XF == F_PIECES)
            if (g.K > (Elem<T>::size == 4 ? 512 : 4096)) return launch_shape<T, TO, DIRECT, F_TAPS, WF>(ctx, g, batches, s);
        if (tiles(128, 128) >= 2 * cus && g.N > 64) return launch_tile<T, TO, 128, 128, 2, 4, 1, 64, 4, DIRECT, XF, WF>(g, batches, s);
        if (tiles(64, 64) * 2 >= cus) return launch_tile<T, TO, 64, 64, 2, 2, 2, 128, 3, DIRECT, XF, WF>(g, batches, s);
        if (tiles(32, 32) * 2 <= cus) return launch_tile<T, TO, 16, 16, 1, 1, 4, 256, 3, DIRECT, XF, WF>(g, batches, s);
        return launch_tile<T, TO, 32, 32, 1, 1, 4, 256, 3, DIRECT, XF, WF>(g, batches, s);
    }
    if constexpr (!DIRECT) {
        // K-major W: 128 x 128 tiles from one per compute unit on, unless most of one would be padding; products take eight wavefronts on
        // the smaller tiles where K is long: a wavefront that has a SIMD to itself issues an instruction every 7 clocks, two
        // share the work of a stage (7 x 4000 x 900 fp32: 32.6 -> 25.3 us, 4 x 2274 x 3609 x 32 fp16: 25.2 -> 19.6 us)
        if constexpr (WF == F_KMAJOR)
            if (g.M > 64 && g.N > 64 && tiles(128, 128) >= cus) return launch_tile<T, TO, 128, 128, 2, 4, 1, 64, 2, DIRECT, XF, WF>(g, batches, s);
        constexpr int W2 = XF == F_ROWS ? 2 : 1;
        if (tiles(64, 64) * 2 >= cus) {
            if constexpr (W2 == 2)
                if (!g.in_order && g.K * (int64_t)Elem<T>::size >= 1024) return launch_tile<T, TO, 64, 64, 2, 2, W2, 128, 2, DIRECT, XF, WF>(g, batches, s);
            return launch_tile<T, TO, 64, 64, 2, 2, 1, 128, 2, DIRECT, XF, WF>(g, batches, s);
        }
        return launch_tile<T, TO, 32, 32, 1, 1, 4 * W2, 256, 2, DIRECT, XF, WF>(g, batches, s);
    }
    return 0;
}

// quotients of one multiplication: exact for k IC < 2^32 and up to 1024 taps
void set_tap_magics(FArgs &g) {
    g.ic_magic = (uint32_t)((uint64_t(1) << 32) / (uint32_t)g.IC + 1);
    g.kw_magic = 65536u / (uint32_t)g.KW + 1;
}

// `direct`: both operands in aligned 16-byte pieces along K
template <typename T>
int launch_conv(mlel_ctx *ctx, FArgs &g, bool direct, hipStream_t s) {
    if (direct) return launch_shape<T, T, true, F_PIECES, F_PIECES>(ctx, g, 1, s);
    // A K of a few pieces: without stages from 700 sub-tiles of 32 x 32 on (3 -> 64, stride 2, 224 x 224: fp32 5.9 -> 4.2 us, fp16 4.3 -> 3.9,
    // 784 of them; fp32 3 -> 24 at 112 x 208, 182: 3.8 -> 4.1), unless 64 channels leave the wavefronts between one and four to a SIMD
    // (four such images in fp16, 3136: 5.8 -> 6.0; 3 -> 40 over six of 256 x 256, 6144: 9.2 -> 7.2; 4 -> 32 over eight of 224 x 224: 24.7 -> 10.4)
    constexpr int E = 16 / Elem<T>::size;
    const int64_t cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
    const int64_t ppr = (g.KW * (int64_t)g.IC + E - 1) / E, pieces = g.KH * ppr, tiles = (int64_t)((g.M + 31) / 32) * ((g.N + 31) / 32);
    // More than six pieces, against the stages over 2500 calls.  Halves: the seven or eight that fill a stage, and rows that are no
    // whole words or three pieces and more, lost up to 1.9 of the time (3 x 3 x 7 -> 232 over 43344 fp16: 19.2 us staged, 30.3 without;
    // 4 x 4 x 6 -> 16 over 22876 bf16: 5.2, 6.1); nine or ten of an even number of channels take 0.55-0.97, most that leave more than
    // 2048 sub-tiles to 32 channels 0.48-0.98.  Without a border the masks are one and more is won: 32 channels 0.48-1.05, rows of
    // two pieces 0.57-1.05.  fp32 lost beyond ten pieces of more than 32 channels with a border (0.85-1.26; the others 0.37-1.13).
    const int64_t steps = (pieces + 1) / 2;
    const bool narrow = g.N <= 32, words = g.IC % 2 == 0;
    bool taken;
    if (Elem<T>::size == 4) taken = steps <= 5 || narrow || !g.border;
    else if (steps <= 3 || (narrow && tiles > 8 * cus && (words || steps <= 5))) taken = true;
    else if (g.border) taken = steps == 5 && (words || (ppr <= 2 && narrow));
    else if (narrow) taken = words || ppr <= 2 || tiles <= 4 * cus;
    else taken = words ? steps == 5 || steps >= 7 : ppr <= 2;
    if (g.dx == 1 && pieces <= 16 && taken && g.wide_out && g.res == nullptr && g.x_bytes >= 16 && g.w_bytes >= 16 && 4 * tiles >= 11 * cus &&
        (g.N <= 32 || tiles <= 4 * cus || tiles >= 16 * cus)) {
        g.div_ppr = make_div_magic((uint32_t)ppr);
        return g.N > 32 && tiles > 4 * cus ? launch_runs<T, 2>(g, (int)steps, s) : launch_runs<T, 1>(g, (int)steps, s);
    }
    return g.dx == 1 ? launch_shape<T, T, false, F_RUNS, F_RUNS>(ctx, g, 1, s) : launch_shape<T, T, false, F_ELEMS, F_ELEMS>(ctx, g, 1, s);
}
template <typename T>
int launch_product(mlel_ctx *ctx, FArgs &g, int64_t batches, bool x_pieces, bool w_pieces, bool w_kmajor, hipStream_t s) {
    if (x_pieces && w_pieces) return launch_shape<T, float, true, F_PIECES, F_PIECES>(ctx, g, batches, s);
    if (!w_kmajor) return launch_shape<T, float, false, F_ROWS, F_ROWS>(ctx, g, batches, s);
    return launch_shape<T, float, false, F_ROWS, F_KMAJOR>(ctx, g, batches, s);
}

bool aligned16(const void *p, std::initializer_list<int64_t> strides) {
    if (((uintptr_t)p % 16) != 0) return false;
    for (int64_t v : strides)
        if (v % 16 != 0) return false;
    return true;
}
constexpr int64_t kLim = (int64_t(1) << 31) - 4096;

}  // namespace

// CONV2D with an fp32 accumulator, optionally followed by the ADD of a residual of the output's shape and by a CLAMP
// (each computed as the stand-alone operator would).  Returns 1 when launched (`probe`: when types and extents are covered;
// pointers are not looked at), 0 to decline.
int try_conv2d_float(mlel_ctx *ctx, hipStream_t s, const mlel_tensor *out, const mlel_tensor *in, const mlel_tensor *w,
                     const mlel_tensor *bias, const mlel_conv2d_attr *a, const mlel_tensor *residual,
                     const mlel_clamp_attr *clamp, bool probe) {
    const int dt = in->dtype;
    if ((dt != MLEL_F16 && dt != MLEL_BF16 && dt != MLEL_F32) || w->dtype != dt || out->dtype != dt ||
        a->acc_type != MLEL_ACC_F32 || a->input_zp != 0 || a->weight_zp != 0)
        return 0;
    if (!is_packed(in) || !is_packed(w) || !is_packed(out) || !is_packed(bias)) return 0;
    const int64_t sz = dt_size(dt), N = in->dims[0], H = in->dims[1], W = in->dims[2], IC = in->dims[3];
    const int64_t OC = w->dims[0], KH = w->dims[1], KW = w->dims[2], OH = out->dims[1], OW = out->dims[2];
    if (w->dims[3] != IC || out->dims[0] != N || out->dims[3] != OC) return 0;
    if (N <= 0 || H <= 0 || W <= 0 || IC <= 0 || OC <= 0 || KH <= 0 || KW <= 0 || OH <= 0 || OW <= 0) return 0;
    if (bias->dims[0] != 1 && bias->dims[0] < OC) return 0;
    if (a->stride[0] <= 0 || a->stride[1] <= 0 || a->dilation[0] <= 0 || a->dilation[1] <= 0) return 0;
    const int64_t K = KH * KW * IC, M = N * OH * OW, small = 1 << 20;
    if (N * H * W * IC * sz >= kLim || OC * K * sz >= kLim || M * OC * sz >= kLim || K >= (1 << 24) || M >= (1 << 30)) return 0;
    // coordinates and taps stay far inside 31 bits
    if (H >= small || W >= small || OH >= small || OW >= small || KH >= 4096 || KW >= 4096 || a->stride[0] >= 1024 ||
        a->stride[1] >= 1024 || a->dilation[0] >= 1024 || a->dilation[1] >= 1024)
        return 0;
    for (int i = 0; i < 4; i++)
        if (a->pad[i] < -small || a->pad[i] > small) return 0;
    if (residual != nullptr && (residual->dtype != dt || !is_packed(residual) || !same_shape(residual, out))) return 0;
    if (probe) return 1;
    FArgs g{};
    g.x = static_cast<const char *>(in->ptr), g.w = static_cast<const char *>(w->ptr);
    g.bias = static_cast<const char *>(bias->ptr), g.out = static_cast<char *>(out->ptr);
    g.res = residual != nullptr ? static_cast<const char *>(residual->ptr) : nullptr;
    g.M = (int)M, g.N = (int)OC, g.K = (int)K;
    g.IC = (int)IC, g.KW = (int)KW, g.KH = (int)KH, g.H = (int)H, g.W = (int)W;
    g.sy = a->stride[0], g.sx = a->stride[1], g.pt = a->pad[0], g.pl = a->pad[2], g.dy = a->dilation[0], g.dx = a->dilation[1];
    g.OHW = (int)(OH * OW), g.OW = (int)OW;
    g.div_ohw = make_div_magic((uint32_t)g.OHW), g.div_ow = make_div_magic((uint32_t)g.OW);
    g.x_pix = (uint32_t)(IC * sz), g.x_row = (uint32_t)(W * IC * sz), g.x_img = (uint32_t)(H * W * IC * sz);
    g.x_bytes = (uint32_t)(N * H * W * IC * sz), g.w_bytes = (uint32_t)(OC * K * sz), g.ldw = (uint32_t)(K * sz);
    g.ldo = (uint32_t)(OC * sz), g.o_bytes = (uint32_t)(M * OC * sz);
    g.bias_len = bias->dims[0] == 1 ? 1 : (int)OC;
    g.border = a->pad[0] > 0 || a->pad[2] > 0 || (OH - 1) * g.sy - a->pad[0] + (KH - 1) * g.dy >= H || (OW - 1) * g.sx - a->pad[2] + (KW - 1) * g.dx >= W;
    const bool pieces = aligned16(in->ptr, {IC * sz}) && aligned16(w->ptr, {IC * sz});
    // the DIRECT form's taps are bits of a word and its divisions single multiplications
    const bool direct = pieces && KH <= 32 && KW <= 32 && (K + 1024) * IC < (int64_t(1) << 32) &&
                        g.dy * (int64_t)g.x_row < (1 << 24) && g.dx * (int64_t)g.x_pix < (1 << 24);
    set_tap_magics(g);
    g.wide_out = aligned16(out->ptr, {OC * sz}) && (residual == nullptr || aligned16(residual->ptr, {}));
    if (clamp != nullptr) {
        g.has_clamp = 1, g.clamp_nan_ignore = clamp->nan_mode == MLEL_NAN_IGNORE;
        g.clamp_lo = (float)clamp->min_val, g.clamp_hi = (float)clamp->max_val;
        if (dt == MLEL_F16) g.clamp_lo = (float)(_Float16)g.clamp_lo, g.clamp_hi = (float)(_Float16)g.clamp_hi;
    }
    if (dt == MLEL_F16) return launch_conv<_Float16>(ctx, g, direct, s);
    if (dt == MLEL_BF16) return launch_conv<BF16>(ctx, g, direct, s);
    return launch_conv<float>(ctx, g, direct, s);
}

// MATMUL over fp16, bf16 or fp32 operands with an fp32 result, optionally followed by the ADD of an fp32 row (one or N values).
// Returns 1 when launched (`probe`: when types, extents and strides are covered; pointers are not looked at), 0 to decline.
// `in_order`: the wavefronts of a tile don't share K (a K-major W of at least half a tile of 64 x 64 per compute unit), so that the
// result is that of gemm_f16.hip to the bit.
int try_matmul_float(mlel_ctx *ctx, hipStream_t s, const mlel_tensor *out, const mlel_tensor *a, const mlel_tensor *b,
                     const mlel_matmul_attr *attr, const mlel_tensor *bias, bool probe, bool in_order) {
    const int dt = a->dtype;
    if ((dt != MLEL_F16 && dt != MLEL_BF16 && dt != MLEL_F32) || b->dtype != dt || out->dtype != MLEL_F32 || attr->a_zp != 0 ||
        attr->b_zp != 0)
        return 0;
    const int64_t sz = dt_size(dt), NB = out->dims[0], M = out->dims[1], N = out->dims[2], K = a->dims[2];
    // (a contraction shorter than one matrix instruction is mostly padding there)
    if (NB <= 0 || M <= 0 || N <= 0 || K < 16) return 0;
    if (a->dims[0] < NB || b->dims[0] < NB || a->dims[1] < M || b->dims[1] < K || b->dims[2] < N) return 0;
    if (a->strides[2] != sz || out->strides[2] != 4 || a->strides[1] < K * sz || out->strides[1] < N * 4) return 0;
    const bool rows = K > 1 && b->strides[1] == sz && b->strides[2] >= b->dims[1] * sz;
    if (!rows && (b->strides[2] != sz || b->strides[1] < N * sz)) return 0;
    for (const mlel_tensor *t : {out, a, b})
        for (int i = 0; i < 3; i++)
            if (t->strides[i] < 0 || t->strides[i] % dt_size(t->dtype) != 0) return 0;
    const int64_t ldw = rows ? b->strides[2] : b->strides[1];
    if (M * a->strides[1] >= kLim || (rows ? N : K) * ldw >= kLim || M * out->strides[1] >= kLim || K >= (1 << 24) ||
        M >= (1 << 30) || N >= (1 << 30))
        return 0;
    if (bias != nullptr && (bias->dtype != MLEL_F32 || bias->rank != 3 || !is_packed(bias) || bias->dims[0] != 1 || bias->dims[1] != 1 ||
                            (bias->dims[2] != 1 && bias->dims[2] != N)))
        return 0;
    if (probe) return 1;
    FArgs g{};
    g.in_order = in_order;
    if (bias != nullptr) g.bias = static_cast<const char *>(bias->ptr), g.bias_len = (int)bias->dims[2];
    g.x = static_cast<const char *>(a->ptr), g.w = static_cast<const char *>(b->ptr), g.out = static_cast<char *>(out->ptr);
    g.M = (int)M, g.N = (int)N, g.K = (int)K;
    g.IC = (int)K, g.KW = g.KH = 1, g.H = 1, g.W = (int)M, g.sy = g.sx = g.dy = g.dx = 1;
    g.OHW = g.OW = (int)M;
    g.div_ohw = make_div_magic((uint32_t)g.OHW), g.div_ow = make_div_magic((uint32_t)g.OW);
    g.x_pix = (uint32_t)a->strides[1];
    g.x_bytes = (uint32_t)((M - 1) * a->strides[1] + K * sz);
    g.ldw = (uint32_t)ldw;
    g.w_bytes = (uint32_t)(((rows ? N : K) - 1) * ldw + (rows ? K : N) * sz);
    g.ldo = (uint32_t)out->strides[1], g.o_bytes = (uint32_t)((M - 1) * out->strides[1] + N * 4);
    g.x_batch = a->strides[0], g.w_batch = b->strides[0], g.o_batch = out->strides[0];
    set_tap_magics(g);
    // (the DIRECT form's division by K is one multiplication)
    const bool xp = aligned16(a->ptr, {a->strides[0], a->strides[1], K * sz}) && (K + 1024) * K < (int64_t(1) << 32);
    const bool wp = rows && aligned16(b->ptr, {b->strides[0], ldw, K * sz});
    g.wide_out = aligned16(out->ptr, {out->strides[0], out->strides[1], N * 4});
    if (dt == MLEL_F16) return launch_product<_Float16>(ctx, g, NB, xp, wp, !rows, s);
    if (dt == MLEL_BF16) return launch_product<BF16>(ctx, g, NB, xp, wp, !rows, s);
    return launch_product<float>(ctx, g, NB, xp, wp, !rows, s);
}

}  // namespace mlel
