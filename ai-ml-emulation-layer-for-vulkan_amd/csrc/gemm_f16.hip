// fp16 x fp16 -> fp32 MATMUL on the gfx950 matrix cores (reference arithmetic: matmul.comp:30-73 with an fp32
// accumulator: out[b][m][n] = sum_k A[b][m][k] * B[b][k][n]; the order of the fp32 additions differs from the
// shader's sequential loop, which is why floating-point graphs are compared within a tolerance).
//
// Kernel shape.  256 threads = 4 wavefronts; a block owns a BM x BN tile of one batch and walks K in steps of 32
// halfs through two LDS buffers, with the global loads of the next step in flight while the current one is
// multiplied (v_mfma_f32_32x32x16_f16).  As in the int8 kernel the B matrix supplies the MFMA row operand and A the
// column operand, so a lane ends up with four consecutive output columns of one output row per register quad and
// stores them as one 128-bit word.
//   A tile: [BM][32 halfs], 80-byte pitch, operands read with ds_read_b128 (8 consecutive k of one row);
//   B tile: kept K-major as in memory, [32][BN halfs]; operands are gathered with ds_read_b64_tr_b16, which hands
//           lane L of a 16-lane group the four k values of column L out of a 4(k) x 16(n) block whose rows are
//           addressed by the group's lanes (lane s points at row s / 4, columns 4 * (s % 4) ..).
// All global loads are buffer loads: an offset at or beyond the extent returns 0, which pads M, N and K tails.
#include <algorithm>

#include "common.hpp"
#include "dispatch.hpp"
#include "float_programs.hpp"

namespace mlel {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v4s lds_v4s;

constexpr uint32_t kOob = 0x80000000u;

struct HGemmArgs {
    const char *a, *b;
    char *out;
    int32_t M, N, K, batches;
    int32_t b_rows;                     // B is laid down row-wise, [N][K]: ldb is then the pitch of a row of K
    int64_t a_batch, b_batch, o_batch;  // bytes
    uint32_t lda, ldb, ldo;             // bytes per row
    uint32_t a_bytes, b_bytes, o_bytes; // per-batch extents (all below 2^31)
    int32_t total_tiles, chunk;
    // set at the launch from the fields above and tiles_n_group
    TileOrder order;
    DivMagic div_group;
    // fused epilogue (EPI = 1): out = fp16(acc + bias[n]) with the addition in fp32; bias may be null
    const float *bias;
    int32_t bias_len;  // 1 (broadcast) or N
    // fp16 tensor of the output's shape added to the rounded result (the ADD of a residual connection), or null
    const char *res;
    int64_t r_batch;
    uint32_t ldr, r_bytes;
    // fp16 result written through a six-dimensional view [NB1, NB2, M1, M2, N1, N2] of other strides (a head split
    // or merge behind the product): batch = nb1 * NB2 + nb2, row = m1 * M2 + m2, column = n1 * N2 + n2 with eight
    // consecutive n2 contiguous.  view == 0: the plain [batch][row][column] layout above.
    // view == 2: the same with eight consecutive m2 contiguous instead (the innermost extent of the product ends up
    // somewhere else: a transposing view) and n2 at a stride of vs_n2 bytes
    int32_t view, v_nb2, v_m2, v_n2;
    int64_t vs_nb1, vs_nb2;
    uint32_t vs_m1, vs_m2, vs_n1, vs_n2;
    // Several products of the same A in one launch (the Q, K and V projections): tile columns [k * tiles_n_group,
    // (k + 1) * tiles_n_group) belong to product k, which has a B, a bias and an output of its own; product 0 uses
    // the fields above.  All products have the same extents and operand strides.
    // the tanh form of GELU applied to the rounded result (GeluTanhProgram with the result as its value 0): the
    // program's four single-element fp16 inputs, or null
    const uint16_t *act[4];
    int32_t groups, tiles_n_group;
    struct Extra {
        const char *b;
        const float *bias;
        char *out;
        int64_t o_batch;
        uint32_t ldo, o_bytes;
        int32_t view, v_nb2, v_m2, v_n2;
        int64_t vs_nb1, vs_nb2;
        uint32_t vs_m1, vs_m2, vs_n1, vs_n2;
    } extra[2];
};
// what a block needs of its product: filled from HGemmArgs or from one of its Extra entries
struct HProduct {
    const char *b;
    const float *bias;
    char *out;
    int64_t o_batch;
    uint32_t ldo, o_bytes;
    int32_t view, v_nb2, v_m2, v_n2;
    int64_t vs_nb1, vs_nb2;
    uint32_t vs_m1, vs_m2, vs_n1, vs_n2;
};

__device__ __forceinline__ uint4 load16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const v4i v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
    return make_uint4((uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w);
}


// Division of the row and column indices of a view by its inner extents, once per 16-byte piece: the extents are the
// same for every piece, so the quotient is one multiplication by floor((2^32 - 1) / d) + 1 (exact while x * d < 2^32,
// which `usable` says for the tile's largest index; otherwise, and for d == 1, the plain division).
struct ViewDiv {
    uint32_t d, magic;
    bool usable;
    __device__ __forceinline__ ViewDiv(int32_t divisor, int32_t largest) {
        d = (uint32_t)divisor;
        usable = d > 1 && (uint64_t)(uint32_t)largest * d < (uint64_t(1) << 32);
        magic = usable ? 0xffffffffu / d + 1u : 0u;
    }
    __device__ __forceinline__ uint32_t quotient(uint32_t x) const { return usable ? __umulhi(x, magic) : (d == 1 ? x : x / d); }
};

// BKH: halfs of K per step (32, or 64 for long contractions: half as many barriers and LDS round trips per K)
// BROWS: B is given row-wise, [N][K] (a weight matrix laid down transposed once, ahead of time): both operands are
// then rows of K, and the main loop is the direct-to-LDS pipeline of the int8 kernel (gemm_i8_kernel.hpp): 64 or 128 bytes of
// K per step, `buffer_load ... lds` into a ring of four unpadded stages whose 16-byte pieces are XOR-swizzled (piece p
// of row r in slot p ^ ((r >> 2) & 3), or p ^ ((r >> 1) & 7)), 128-bit operand reads without bank conflicts and without the
// transposing reads of the K-major tile, one barrier per step, reads of the next 16 halfs issued before the multiplies of these.
// The ring is four stages deep, eight short ones for the 64 x 64 tile: it is taken where a compute unit gets one or two blocks,
// and the stages in flight are then all that hides the trip to memory.  A width that is no whole number of requests per thread
// (192 columns over eight wavefronts) is rounded up in shared memory, the rows beyond the tile fetched as zeros.
constexpr int ring_stages(int bm, int bn, int bkh) { return bm * bn <= 64 * 64 && bkh == 32 ? 8 : 4; }
constexpr int ring_w_pieces(int bn, int nt, int bkh) { return (bn * bkh / 8 + nt - 1) / nt; }  // of a thread
template <int BM, int BN, int WAVES_M, int WAVES_N, int EPI, int BKH, bool BROWS = false>
__global__ void __launch_bounds__(64 * WAVES_M * WAVES_N) gemm_f16_kernel(const HGemmArgs g) {
    constexpr int NT = 64 * WAVES_M * WAVES_N;  // four or eight wavefronts
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
    constexpr int TM = WM / 32, TN = WN / 32;
    constexpr int XPITCH = BKH * 2 + 16;      // bytes per A row in LDS
    constexpr int XP16 = BKH / 8;             // 16-byte pieces per A row
    constexpr int XPASS = NT / XP16;          // A rows covered by one pass of the block
    constexpr int XROWS = BM / XPASS;         // 16-byte pieces of A per thread and step
    constexpr int WPITCH = 2 * BN + 32;       // bytes per K row of the B tile: 4 rows x 32 B land on distinct banks
    constexpr int WROW16 = BN / 8;            // 16-byte pieces per K row
    constexpr int WCHUNKS = (BKH * WROW16) / NT;
    static_assert((WAVES_M * WAVES_N == 4 || WAVES_M * WAVES_N == 8) && BM % XPASS == 0 && WM % 32 == 0 && WN % 32 == 0 && (BROWS || (BKH * WROW16) % NT == 0), "tile shape");
    constexpr int XBUF = BM * XPITCH, WBUF = BKH * WPITCH;
    extern __shared__ __align__(16) char smem[];
    char *xs = smem;             // [2][BM][XPITCH]
    char *ws = smem + 2 * XBUF;  // [2][BKH][WPITCH]

    // Every argument that the tile assignment and the first operand requests depend on is asked for here, in one
    // batch (every dword of the wide loads that bring them named: a register nobody waits for is given away at once,
    // and whoever gets it waits for the load first).  Left alone the compiler loads arguments where they are first
    // used, behind the early exit, behind three divisions and behind each other: five to nine trips to memory in a
    // row before a wavefront's first address.
    asm volatile("" ::"s"(g.chunk), "s"(g.total_tiles), "s"(g.order.tiles_m), "s"(g.order.tiles_n), "s"(g.order.rows), "s"(g.order.m_batch),
                 "s"(g.order.m_band), "s"(g.order.m_rows), "s"(g.order.m_last), "s"(g.order.shifts),
                 "s"(g.div_group.m), "s"(g.div_group.s),
                 "s"(g.groups), "s"(g.tiles_n_group), "s"(g.a), "s"(g.b), "s"(g.extra[0].b), "s"(g.extra[1].b), "s"(g.out),
                 "s"(g.M), "s"(g.N), "s"(g.K), "s"(g.batches), "s"(g.b_rows), "s"(g.a_batch), "s"(g.b_batch), "s"(g.o_batch),
                 "s"(g.lda), "s"(g.ldb), "s"(g.ldo), "s"(g.a_bytes), "s"(g.b_bytes), "s"(g.o_bytes),
                 // the pointers of the epilogue, which the compiler follows up here already (the activation's scalars)
                 "s"(g.bias), "s"(g.bias_len), "s"(g.res), "s"(g.act[0]), "s"(g.act[1]), "s"(g.act[2]), "s"(g.act[3]));
    // consecutive tiles (sharing operand panels) go to the same XCD; blocks are dealt to XCDs round-robin
    const int lin = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u));
    if (lin >= g.total_tiles) return;
    int batch, tile_m, tile_n;
    g.order.tile(lin, batch, tile_m, tile_n);
    HProduct o{g.b, g.bias, g.out, g.o_batch, g.ldo, g.o_bytes, g.view, g.v_nb2, g.v_m2, g.v_n2, g.vs_nb1, g.vs_nb2,
               g.vs_m1, g.vs_m2, g.vs_n1, g.vs_n2};
    if (g.groups > 1) {  // uniform
        const int product = div_magic(tile_n, g.div_group);
        tile_n -= product * g.tiles_n_group;
        if (product > 0) {
            const HGemmArgs::Extra &e = product == 1 ? g.extra[0] : g.extra[1];
            o = HProduct{e.b, e.bias, e.out, e.o_batch, e.ldo, e.o_bytes, e.view, e.v_nb2, e.v_m2, e.v_n2, e.vs_nb1, e.vs_nb2,
                         e.vs_m1, e.vs_m2, e.vs_n1, e.vs_n2};
        }
        // the operand pointer is on the way to the first request: picked from registers that are already there
        o.b = product == 0 ? g.b : (product == 1 ? g.extra[0].b : g.extra[1].b);
    }
    const int m_base = tile_m * BM, n_base = tile_n * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wave_m = wave / WAVES_N, wave_n = wave % WAVES_N;

    const __amdgpu_buffer_rsrc_t ares = rsrc(g.a + (int64_t)batch * g.a_batch, g.a_bytes);
    const __amdgpu_buffer_rsrc_t bres = rsrc(o.b + (int64_t)batch * g.b_batch, g.b_bytes);

    v16f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    // the bias of this lane's columns (fused form): lane holds, per register quad q, columns 8q + 4 * (lane / 32) ...
    // (where to fetch it: behind the first stages of the direct-to-LDS loop when that costs 16 registers; the wide tile's
    // 32 cost its GELU epilogue more than the trip to memory they hide, 35.5 -> 36.0 us)
    constexpr bool BIAS_AHEAD = BROWS && TN == 1;
    float bias_r[TN][4][4];
    auto fetch_bias = [&]() {
        // through a buffer resource of the bias's extent: a column beyond N (or no bias at all) reads as zero without a test
        const __amdgpu_buffer_rsrc_t bias_res =
            rsrc(o.bias, o.bias != nullptr ? (g.bias_len == 1 ? 4u : (uint32_t)g.N * 4u) : 0u);
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int n0 = n_base + wave_n * WN + j * 32 + 8 * q + 4 * (lane >> 5);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    bias_r[j][q][e] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(bias_res, g.bias_len == 1 ? 0 : (n0 + e) * 4, 0, 0));
            }
    };
    if constexpr (BROWS) {
        // ---- direct-to-LDS main loop (K % 32 == 0: whole 64-byte steps)
        constexpr int BK = BKH * 2, PP = BK / 16, SH = BK == 64 ? 2 : 1, KKN = BK / 32;
        constexpr int XI = BM * PP / NT, WI = ring_w_pieces(BN, NT, BKH);  // 16-byte pieces per thread and stage
        constexpr int DL_S = ring_stages(BM, BN, BKH), DL_STAGE = (BM + WI * NT / PP) * BK;
        // (request counts above 15 need the upper bits of the vmcnt field, a path no instance has exercised)
        static_assert((BM * PP) % NT == 0 && (DL_S - 1) * (XI + WI) < 16, "whole pieces per thread");
        const int wave_u = __builtin_amdgcn_readfirstlane(wave);
        uint32_t xo[XI], wo[WI];
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const int q = i * NT + tid, r = q / PP, p = (q % PP) ^ ((r >> SH) & (PP - 1));
            const int m = m_base + r;
            xo[i] = m < g.M ? (uint32_t)m * g.lda + (uint32_t)(p * 16) : kOob;
        }
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int q = i * NT + tid, r = q / PP, p = (q % PP) ^ ((r >> SH) & (PP - 1));
            const int n = n_base + r;
            wo[i] = n < g.N && r < BN ? (uint32_t)n * g.ldb + (uint32_t)(p * 16) : kOob;  // (beyond the tile: zeros)
        }
        const v4i xres4 = rsrc_words(g.a + (int64_t)batch * g.a_batch, g.a_bytes);
        const v4i wres4 = rsrc_words(o.b + (int64_t)batch * g.b_batch, g.b_bytes);
        const uint32_t lds0 = (uint32_t) reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem) +
                              (uint32_t)(wave_u * 1024);
        // operand addresses inside a stage: row lane % 32 of a 32-row group, the lane half's eight halfs of K half kk
        const int h = lane >> 5, swz = (lane >> SH) & (PP - 1);
        const char *x_base[KKN], *w_base[KKN];
#pragma unroll
        for (int kk = 0; kk < KKN; kk++) {
            const int slot = ((kk * 2 + h) ^ swz) * 16;
            x_base[kk] = smem + (wave_m * WM + (lane & 31)) * BK + slot;
            w_base[kk] = smem + BM * BK + (wave_n * WN + (lane & 31)) * BK + slot;
        }
        // The loop, as in the int8 kernel's direct-to-LDS form: a wavefront issues in order, so a K half is one
        // straight line -- a matrix instruction, then a share of the next half's operand reads and of the requests,
        // which issue while the matrix core works, then the next matrix instruction.  Stage s lives in buffer
        // s % DL_S; a stage's requests ride in the last 16 halfs of a step, behind the step's barrier, which frees the
        // buffer (spread over both halves of a step they arrive a step later, which the long contractions whose
        // operands come from memory rather than from the L2 pay for: 4096 x 3072 x 768 ran 5 % slower).  Beyond the last step they go through an
        // empty resource and fetch nothing, so every step has the same requests in flight and the waits count exactly:
        // at most DL_S - 3 stages outstanding at the barrier of step s means this thread's part of stage s + 1 has
        // landed; the barrier extends that to every thread's part and says that every wavefront has received its
        // reads of stage s - 1, whose buffer the step's requests overwrite.
        const int nk = g.K / BKH;
        const v4i null4 = v4i{xres4[0], xres4[1], 0, xres4[3]};
        constexpr int NLA = XI + WI;
        auto half = [&](auto lp_t, const v8h(&xc)[TM], const v8h(&wc)[TN], v8h(&xn)[TM], v8h(&wn)[TN], int rbuf, int rkk,
                        int ibuf, int istep) {
            constexpr int LP = decltype(lp_t)::value;  // 1: the stage's requests ride in this half, 0: none
            constexpr int NM = TM * TN, NR = TM + TN;
            constexpr int L0 = 0, L1 = LP == 1 ? NLA : 0, NL = L1 - L0, LPER = (NL + NM - 1) / NM;
            const bool live = istep < nk;
            const v4i xr = live ? xres4 : null4, wr = live ? wres4 : null4;
            const uint32_t xd = lds0 + (uint32_t)(ibuf * DL_STAGE), wd = xd + BM * BK;
            const uint32_t kb = (uint32_t)istep * BK;
            // (two wavefronts share a SIMD here and fill each other's gaps: the reads go first, so that their data
            // is there when the next half starts; only the requests are dealt out behind the matrix instructions)
#pragma unroll
            for (int r = 0; r < NR; r++) {
                if (r < TM) xn[r] = *reinterpret_cast<const v8h *>(x_base[rkk] + rbuf * DL_STAGE + r * 32 * BK);
                else wn[r - TM] = *reinterpret_cast<const v8h *>(w_base[rkk] + rbuf * DL_STAGE + (r - TM) * 32 * BK);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < NM; t++) {
                const int i = t / TN, j = t % TN;
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wc[j], xc[i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < LPER; u++) {
                    const int l = L0 + t * LPER + u;
                    if (l < L1) {
                        if (l < XI) load16_to_lds(xr, xd + l * NT * 16, xo[l], kb);
                        else load16_to_lds(wr, wd + (l - XI) * NT * 16, wo[l - XI], kb);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        v8h xf0[TM], wf0[TN], xf1[TM], wf1[TN];
#pragma unroll
        for (int d = 0; d < DL_S - 1; d++) {
            const v4i xr = d < nk ? xres4 : null4, wr = d < nk ? wres4 : null4;
            const uint32_t xd = lds0 + (uint32_t)(d * DL_STAGE), wd = xd + BM * BK;
#pragma unroll
            for (int l = 0; l < NLA; l++) {
                if (l < XI) load16_to_lds(xr, xd + l * NT * 16, xo[l], (uint32_t)d * BK);
                else load16_to_lds(wr, wd + (l - XI) * NT * 16, wo[l - XI], (uint32_t)d * BK);
            }
        }
        // The bias is asked for behind the first stages and used behind the loop (asked for there, its trip to memory
        // was waited out by every wavefront in front of the first store).  These loads are younger than the first
        // stages and older than every later request, so the counted waits hold with them in flight: the first ones
        // only wait for a few requests more.
        if (EPI == 1 && BIAS_AHEAD) fetch_bias();
        wait_vmcnt<(DL_S - 2) * NLA>();  // stage 0 has landed: what was requested behind it may be in flight
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < TM; i++) xf0[i] = *reinterpret_cast<const v8h *>(x_base[0] + i * 32 * BK);
#pragma unroll
        for (int j = 0; j < TN; j++) wf0[j] = *reinterpret_cast<const v8h *>(w_base[0] + j * 32 * BK);
        for (int step = 0; step < nk; step += DL_S) {
#pragma unroll
            for (int d = 0; d < DL_S; d++) {
                if (step + d < nk) {  // uniform
                    half(std::integral_constant<int, 0>{}, xf0, wf0, xf1, wf1, d, 1, 0, 0);
#pragma unroll
                    for (int kk = 1; kk + 1 < KKN; kk += 2) {
                        half(std::integral_constant<int, 0>{}, xf1, wf1, xf0, wf0, d, kk + 1, 0, 0);
                        half(std::integral_constant<int, 0>{}, xf0, wf0, xf1, wf1, d, kk + 2, 0, 0);
                    }
                    wait_vmcnt<(DL_S - 3) * NLA>();
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    half(std::integral_constant<int, 1>{}, xf1, wf1, xf0, wf0, (d + 1) % DL_S, 0, (d + DL_S - 1) % DL_S,
                         step + d + DL_S - 1);
                }
            }
        }
        wait_vmcnt<0>();  // the requests beyond the last step write (zeros) into the ring, which the epilogue reuses
        __syncthreads();
    } else {
    uint32_t xoff[XROWS], woff[WCHUNKS];
#pragma unroll
    for (int i = 0; i < XROWS; i++) {
        const int m = m_base + tid / XP16 + XPASS * i;
        xoff[i] = m < g.M ? (uint32_t)m * g.lda + (tid % XP16) * 16 : kOob;
    }
#pragma unroll
    for (int i = 0; i < WCHUNKS; i++) {
        const int c = tid + NT * i;
        const int n = n_base + (c % WROW16) * 8;
        woff[i] = n < g.N ? (uint32_t)(c / WROW16) * g.ldb + (uint32_t)n * 2 : kOob;
    }
    auto prefetch = [&](int k0, uint4 (&xr)[XROWS], uint4 (&wr)[WCHUNKS]) {
        const bool kin = k0 + (tid % XP16) * 8 < g.K;  // K % 8 == 0: a piece lies wholly inside or outside
#pragma unroll
        for (int i = 0; i < XROWS; i++) xr[i] = load16(ares, (kin && xoff[i] != kOob) ? xoff[i] + (uint32_t)k0 * 2 : kOob);
#pragma unroll
        for (int i = 0; i < WCHUNKS; i++) {
            const int row = (tid + NT * i) / WROW16;
            wr[i] = load16(bres, (k0 + row < g.K && woff[i] != kOob) ? woff[i] + (uint32_t)k0 * g.ldb : kOob);
        }
    };
    auto stage = [&](int buf, const uint4 (&xr)[XROWS], const uint4 (&wr)[WCHUNKS]) {
#pragma unroll
        for (int i = 0; i < XROWS; i++)
            *reinterpret_cast<uint4 *>(xs + buf * XBUF + (tid / XP16 + XPASS * i) * XPITCH + (tid % XP16) * 16) = xr[i];
#pragma unroll
        for (int i = 0; i < WCHUNKS; i++) {
            const int c = tid + NT * i;
            *reinterpret_cast<uint4 *>(ws + buf * WBUF + (c / WROW16) * WPITCH + (c % WROW16) * 16) = wr[i];
        }
    };

    // operand addresses inside a tile: A row = lane % 32, k group = lane / 32 (8 halfs each);
    // B: 16-lane group q = lane / 16 covers columns 16 * (q & 1) .., k group q / 2; lane s = lane % 16 points at
    // row s / 4, columns 4 * (s % 4) of the 4 x 16 block
    const int a_row = lane & 31, a_kg = lane >> 5;
    const int s16 = lane & 15, q16 = lane >> 4;
    const int b_row = 8 * (q16 >> 1) + (s16 >> 2), b_col = 16 * (q16 & 1) + 4 * (s16 & 3);
    auto compute = [&](int buf) {
        const char *xt = xs + buf * XBUF;
        const char *wt = ws + buf * WBUF;
#pragma unroll
        for (int kk = 0; kk < BKH / 16; kk++) {
            v8h af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; i++)
                af[i] = *reinterpret_cast<const v8h *>(xt + (wave_m * WM + i * 32 + a_row) * XPITCH + kk * 32 + a_kg * 16);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const char *p = wt + (kk * 16 + b_row) * WPITCH + (wave_n * WN + j * 32 + b_col) * 2;
                const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)p);
                const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(p + 4 * WPITCH));
                union {
                    v4s s[2];
                    v8h h;
                } u;
                u.s[0] = lo;
                u.s[1] = hi;
                bf[j] = u.h;
            }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[j], af[i], acc[i][j], 0, 0, 0);
        }
    };

    // ring of DEPTH register sets: DEPTH - 1 steps of global loads in flight while one step is multiplied
    constexpr int DEPTH = BKH == 32 ? 4 : 3;
    const int nk = (g.K + BKH - 1) / BKH;
    uint4 xr[DEPTH][XROWS], wr[DEPTH][WCHUNKS];
#pragma unroll
    for (int d = 0; d < DEPTH; d++) prefetch(d * BKH, xr[d], wr[d]);
    stage(0, xr[0], wr[0]);
    __syncthreads();
    for (int step = 0; step < nk; step += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) {
            if (step + d < nk) {  // uniform
                const int cur = (step + d) & 1;  // LDS buffer of this step
                prefetch((step + d + DEPTH) * BKH, xr[d], wr[d]);
                compute(cur);
                stage(cur ^ 1, xr[(d + 1) % DEPTH], wr[(d + 1) % DEPTH]);
                __syncthreads();
            }
        }
    }
    }

    // ---- store: lane holds row m = lane % 32 of each sub-tile and, per register quad q, columns 8q + 4 * (lane / 32)
    const int64_t o_base = o.view ? (int64_t)(batch / o.v_nb2) * o.vs_nb1 + (int64_t)(batch % o.v_nb2) * o.vs_nb2
                                  : (int64_t)batch * o.o_batch;
    const __amdgpu_buffer_rsrc_t ores = rsrc(o.out + o_base, o.o_bytes);
    // otherwise fetched here, in one batch before any store (a load after a store would have to wait for it: the
    // compiler cannot tell that the two do not alias)
    if (EPI == 1 && !BIAS_AHEAD) fetch_bias();
    if (EPI == 1) {
        // fp16 result: a lane's four values are only eight bytes of a row, and a store instruction would touch 32 rows.
        // The tile goes through shared memory instead (the operand buffers are free: the loop ended with a barrier)
        // and leaves in 16-byte pieces, consecutive lanes along a row, so that every instruction writes whole lines.
        constexpr int OPITCH = BN * 2 + 16;
        constexpr int TPITCH = BM * 2 + 16;  // a column of the tile, for transposing views
        // the launch sizes shared memory for the larger of the operand buffers and the result tile
#pragma unroll
        for (int i = 0; i < TM; i++) {
            char *orow = smem + (wave_m * WM + i * 32 + (lane & 31)) * OPITCH;
#pragma unroll
            for (int j = 0; j < TN; j++) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    // ADD in fp32 (one rounding), then CAST to fp16 (round to nearest even): the two operators that
                    // follow the MATMUL in the unfused graph
                    _Float16 h[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float sum = o.bias != nullptr ? acc[i][j][4 * q + e] + bias_r[j][q][e] : acc[i][j][4 * q + e];
                        h[e] = (_Float16)sum;
                    }
                    const int col = wave_n * WN + j * 32 + 8 * q + 4 * (lane >> 5);
                    if (o.view == 2) {  // uniform; transposing view: the tile is laid down column by column
                        const int trow = wave_m * WM + i * 32 + (lane & 31);
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            *reinterpret_cast<_Float16 *>(smem + (col + e) * TPITCH + trow * 2) = h[e];
                        continue;
                    }
                    uint2 v;
                    v.x = (uint32_t)__builtin_bit_cast(unsigned short, h[0]) | ((uint32_t)__builtin_bit_cast(unsigned short, h[1]) << 16);
                    v.y = (uint32_t)__builtin_bit_cast(unsigned short, h[2]) | ((uint32_t)__builtin_bit_cast(unsigned short, h[3]) << 16);
                    *reinterpret_cast<uint2 *>(orow + col * 2) = v;
                }
            }
        }
        const __amdgpu_buffer_rsrc_t rres = rsrc(g.res != nullptr ? g.res + (int64_t)batch * g.r_batch : o.out, g.res != nullptr ? g.r_bytes : 0);
        // the residual's pieces of this thread, requested before the barrier and before any store (a load behind a
        // store waits for it, and one fetch per piece in the store loop would expose its latency four times over)
        constexpr int PIECES = BM * (BN / 8) / NT;
        constexpr bool RES_AHEAD = PIECES <= 4;
        uint4 res_r[RES_AHEAD ? PIECES : 1];
        if (RES_AHEAD && g.res != nullptr && o.view != 2) {  // uniform
#pragma unroll
            for (int i = 0; i < (RES_AHEAD ? PIECES : 1); i++) {
                const int p = i * NT + tid, r = p / (BN / 8), c = p % (BN / 8);
                const int m = m_base + r, n = n_base + c * 8;
                res_r[i] = load16(rres, (m < g.M && n < g.N) ? (uint32_t)m * g.ldr + (uint32_t)n * 2 : kOob);
            }
        }
        __syncthreads();
        const ViewDiv by_m2(o.view ? o.v_m2 : 1, g.M), by_n2(o.view ? o.v_n2 : 1, g.N);
        if (o.view == 2) {
            // transposing view: a piece is eight consecutive rows of one column (tile rows start at multiples of
            // eight and M2 is one, so a piece never straddles two m1)
            for (int p = tid; p < BN * (BM / 8); p += NT) {
                const int c = p / (BM / 8), r8 = p - c * (BM / 8);
                const int m = m_base + r8 * 8, n = n_base + c;
                if (m >= g.M || n >= g.N) continue;
                const uint4 piece = *reinterpret_cast<const uint4 *>(smem + c * TPITCH + r8 * 16);
                const uint32_t w[4] = {piece.x, piece.y, piece.z, piece.w};
                const uint32_t m1 = by_m2.quotient((uint32_t)m), n1 = by_n2.quotient((uint32_t)n);
                const uint32_t off = m1 * o.vs_m1 + ((uint32_t)m - m1 * (uint32_t)o.v_m2) * 2 + n1 * o.vs_n1 +
                                     ((uint32_t)n - n1 * (uint32_t)o.v_n2) * o.vs_n2;
                v4i v;
                v.x = (int)w[0], v.y = (int)w[1], v.z = (int)w[2], v.w = (int)w[3];
                __builtin_amdgcn_raw_buffer_store_b128(v, ores, (int)off, 0, kOutAux);
            }
            return;
        }
        constexpr int PPR = BN / 8;  // 16-byte pieces per row of the tile
        uint32_t act_c[4] = {0, 0, 0, 0};
        if (g.act[0] != nullptr) {  // uniform
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t bits = *g.act[k];
                act_c[k] = bits | (bits << 16);
            }
        }
#pragma unroll
        for (int p0 = 0; p0 < BM * PPR; p0 += NT) {
            const int p = p0 + tid, r = p / PPR, c = p % PPR;
            const int m = m_base + r, n = n_base + c * 8;
            uint4 piece = *reinterpret_cast<const uint4 *>(smem + r * OPITCH + c * 16);
            const bool inside = m < g.M && n < g.N;
            uint32_t off = inside ? (uint32_t)m * o.ldo + (uint32_t)n * 2 : kOob;
            if (o.view && inside) {  // uniform
                const uint32_t m1 = by_m2.quotient((uint32_t)m), n1 = by_n2.quotient((uint32_t)n);
                off = m1 * o.vs_m1 + ((uint32_t)m - m1 * (uint32_t)o.v_m2) * o.vs_m2 + n1 * o.vs_n1 +
                      ((uint32_t)n - n1 * (uint32_t)o.v_n2) * 2;
            }
            if (g.act[0] != nullptr) piece = gelu_tanh_piece(piece, act_c);  // uniform
            if (g.res != nullptr) {  // uniform; ADD of two fp16 tensors: one rounding of the exact sum
                const uint4 other = RES_AHEAD ? res_r[RES_AHEAD ? p0 / NT : 0]
                                              : load16(rres, inside ? (uint32_t)m * g.ldr + (uint32_t)n * 2 : kOob);
                typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
                h2_t *ph = reinterpret_cast<h2_t *>(&piece);
                const h2_t *oh = reinterpret_cast<const h2_t *>(&other);
#pragma unroll
                for (int e = 0; e < 4; e++) ph[e] = ph[e] + oh[e];
            }
            v4i v;
            v.x = (int)piece.x, v.y = (int)piece.y, v.z = (int)piece.z, v.w = (int)piece.w;
            __builtin_amdgcn_raw_buffer_store_b128(v, ores, (int)off, 0, kOutAux);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = m_base + wave_m * WM + i * 32 + (lane & 31);
        const uint32_t row_off = m < g.M ? (uint32_t)m * o.ldo : kOob;
#pragma unroll
        for (int j = 0; j < TN; j++) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int n0 = n_base + wave_n * WN + j * 32 + 8 * q + 4 * (lane >> 5);
                const uint32_t off = (row_off != kOob && n0 < g.N) ? row_off + (uint32_t)n0 * 4 : kOob;
                v4i v;
                v.x = __float_as_int(acc[i][j][4 * q + 0]);
                v.y = __float_as_int(acc[i][j][4 * q + 1]);
                v.z = __float_as_int(acc[i][j][4 * q + 2]);
                v.w = __float_as_int(acc[i][j][4 * q + 3]);
                __builtin_amdgcn_raw_buffer_store_b128(v, ores, (int)off, 0, kOutAux);
            }
        }
    }
}

// The same product for few tiles.  A 64 x 64 tile of a long contraction is bound by the bytes its compute unit takes from the
// L2 (41 per clock at best: 393 KB, 4.6 us, for K = 1536) while most of the other units idle; four times as many tiles of
// 32 x 32 need half of that each.  One wavefront multiplies -- eight products per stage of 256 bytes of K take it 256 clocks,
// less than the stage's 16 KB take to arrive -- so that K is added in the one order that every form of the product has, and
// four request stages, straight into shared memory, in a ring of three: a wavefront that does both issues the instructions of both, one
// every seven clocks.  X: [32][256 bytes], piece p of row r in slot p ^ (r & 15); W the same, or (KM) the 128 rows of K of
// 32 columns as they lie in memory, transposed by the reads.  The tile is finished and stored by all of the other wavefronts, a
// thread per four columns of a row (four rows of a column for a transposing view).
// PART: products whose operands are read while as many are multiplied -- a whole stage where every tile has a compute unit to
// itself (197 x 1536 x 384: 5.5 us without, 5.2 with four, 4.4 with eight); half of one where two tiles share one, whose
// registers eight would not leave (504 tiles, 197 x 1536 x 2304: 6.3, 6.2, 7.3).
constexpr int kFewStages = 3;
template <int PART, int EPI, bool KM>
__global__ void __launch_bounds__(320) gemm_f16_few_kernel(const HGemmArgs g) {
    constexpr int BT = 32, NT = 256, PPR = 16, BK = 256, XI = BT * PPR / NT, STAGE = 2 * BT * BK, KKN = 8, S = kFewStages;
    constexpr int RP = BT + 4, QPR = BT / 4;
    static_assert((S - 1) * 2 * XI < 16, "request counts above 15 need the upper bits of the vmcnt field");
    extern __shared__ __align__(16) char smem[];

    // (the arguments in one batch, as above)
    asm volatile("" ::"s"(g.chunk), "s"(g.total_tiles), "s"(g.order.tiles_m), "s"(g.order.tiles_n), "s"(g.order.rows), "s"(g.order.m_batch),
                 "s"(g.order.m_band), "s"(g.order.m_rows), "s"(g.order.m_last), "s"(g.order.shifts),
                 "s"(g.div_group.m), "s"(g.div_group.s),
                 "s"(g.groups), "s"(g.tiles_n_group), "s"(g.a), "s"(g.b), "s"(g.extra[0].b), "s"(g.extra[1].b), "s"(g.out),
                 "s"(g.M), "s"(g.N), "s"(g.K), "s"(g.batches), "s"(g.a_batch), "s"(g.b_batch), "s"(g.o_batch),
                 "s"(g.lda), "s"(g.ldb), "s"(g.ldo), "s"(g.a_bytes), "s"(g.b_bytes), "s"(g.o_bytes),
                 "s"(g.bias), "s"(g.bias_len), "s"(g.res), "s"(g.act[0]), "s"(g.act[1]), "s"(g.act[2]), "s"(g.act[3]));
    const int lin = __builtin_amdgcn_readfirstlane((int)(blockIdx.x % 8u) * g.chunk + (int)(blockIdx.x / 8u));
    if (lin >= g.total_tiles) return;
    int batch, tile_m, tile_n;
    g.order.tile(lin, batch, tile_m, tile_n);
    HProduct o{g.b, g.bias, g.out, g.o_batch, g.ldo, g.o_bytes, g.view, g.v_nb2, g.v_m2, g.v_n2, g.vs_nb1, g.vs_nb2,
               g.vs_m1, g.vs_m2, g.vs_n1, g.vs_n2};
    if (g.groups > 1) {  // uniform
        const int product = div_magic(tile_n, g.div_group);
        tile_n -= product * g.tiles_n_group;
        if (product > 0) {
            const HGemmArgs::Extra &e = product == 1 ? g.extra[0] : g.extra[1];
            o = HProduct{e.b, e.bias, e.out, e.o_batch, e.ldo, e.o_bytes, e.view, e.v_nb2, e.v_m2, e.v_n2, e.vs_nb1, e.vs_nb2,
                         e.vs_m1, e.vs_m2, e.vs_n1, e.vs_n2};
        }
        o.b = product == 0 ? g.b : (product == 1 ? g.extra[0].b : g.extra[1].b);
    }
    const int m_base = tile_m * BT, n_base = tile_n * BT;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // ---- requests: the same piece of rows r0 + i NT / PPR of both operands; KM: row q / 4 of K, columns 8 (q % 4) ..
    const bool loads = wave < 4;  // uniform
    const int r0 = tid / PPR, p0 = (tid % PPR) ^ (r0 & 15);
    const v4i xres = rsrc_words(g.a + (int64_t)batch * g.a_batch, g.a_bytes), wres = rsrc_words(o.b + (int64_t)batch * g.b_batch, g.b_bytes);
    uint32_t xo[XI], wo[XI];
#pragma unroll
    for (int i = 0; i < XI; i++) {
        const int m = m_base + r0 + i * (NT / PPR), q = i * NT + tid, n = KM ? n_base + q % 4 * 8 : n_base + r0 + i * (NT / PPR);
        xo[i] = m < g.M ? (uint32_t)m * g.lda + (uint32_t)(p0 * 16) : kOob;
        wo[i] = n >= g.N ? kOob : (KM ? (uint32_t)(q / 4) * g.ldb + (uint32_t)n * 2 : (uint32_t)n * g.ldb + (uint32_t)(p0 * 16));
    }
    const uint32_t lds0 = (uint32_t) reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem) + (uint32_t)(wave * 1024);
    const int nk = (g.K + 127) / 128;
    auto request = [&](int step, int buf) {
        const uint32_t d = lds0 + (uint32_t)(buf * STAGE), kb = (uint32_t)step * BK, wb = KM ? (uint32_t)step * 128 * g.ldb : kb;
        if ((step + 1) * 128 > g.K) {  // uniform: the stage that ends beyond K, whose pieces there are zeros
            const bool in = step * 128 + p0 * 8 < g.K;
#pragma unroll
            for (int i = 0; i < XI; i++) load16_to_lds(xres, d + i * NT * 16, in ? xo[i] : kOob, kb);
#pragma unroll
            for (int i = 0; i < XI; i++)
                load16_to_lds(wres, d + BT * BK + i * NT * 16, (KM ? step * 128 + (i * NT + tid) / 4 < g.K : in) ? wo[i] : kOob, wb);
        } else {
#pragma unroll
            for (int i = 0; i < XI; i++) load16_to_lds(xres, d + i * NT * 16, xo[i], kb);
#pragma unroll
            for (int i = 0; i < XI; i++) load16_to_lds(wres, d + BT * BK + i * NT * 16, wo[i], wb);
        }
    };
    const bool across = o.view == 2;  // uniform: a transposing view, four rows of a column
    const int qm = across ? tid % QPR * 4 : tid / QPR, qn = across ? tid / QPR : tid % QPR * 4;  // this thread's first element within the tile
    float bias_r[4] = {0.f, 0.f, 0.f, 0.f};
    v2i res_r = v2i{0, 0};
    uint32_t act_c[4] = {0, 0, 0, 0};
    auto meet = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    float *tile = reinterpret_cast<float *>(smem);  // [32][RP], when the stages have been read
    // barrier s: stage s has landed, and stage s - 1 has been read, whose buffer the next request overwrites
    if (loads) {
#pragma unroll
        for (int d = 0; d < S - 1; d++)
            if (d < nk) request(d, d);  // uniform
        if constexpr (EPI == 1) {
            // what the epilogue needs: younger than the first stages and older than every later request, so the counted waits hold
            const __amdgpu_buffer_rsrc_t bias_res = rsrc(o.bias, o.bias != nullptr ? (g.bias_len == 1 ? 4u : (uint32_t)g.N * 4u) : 0u);
            const __amdgpu_buffer_rsrc_t rres = rsrc(g.res + (int64_t)batch * g.r_batch, g.res != nullptr ? g.r_bytes : 0u);
#pragma unroll
            for (int e = 0; e < 4; e++)
                bias_r[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                          bias_res, g.bias_len == 1 ? 0 : (n_base + qn + (across ? 0 : e)) * 4, 0, 0));
            const uint32_t at = (uint32_t)(m_base + qm) * g.ldr + (uint32_t)(n_base + qn) * 2;
            res_r = __builtin_amdgcn_raw_buffer_load_b64(rres, m_base + qm < g.M && n_base + qn < g.N ? (int)at : (int)kOob, 0, 0);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const __amdgpu_buffer_rsrc_t ares = rsrc(g.act[k], g.act[k] != nullptr ? 2u : 0u);
                const uint32_t bits = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(ares, 0, 0, 0);
                act_c[k] = bits | (bits << 16);
            }
        }
        int step = 0;
        for (; step + S - 1 < nk; step++) {
            wait_vmcnt<(S - 2) * 2 * XI>();
            meet();
            request(step + S - 1, (step + S - 1) % S);
        }
        auto drain = [&](auto self, auto left) {  // the last S - 1 stages: nothing is left to request
            constexpr int R = decltype(left)::value;
            if constexpr (R > 0) {
                if (nk - step >= R) {  // uniform
                    wait_vmcnt<(R - 1) * 2 * XI>();
                    meet();
                    step++;
                }
                self(self, std::integral_constant<int, R - 1>{});
            }
        };
        drain(drain, std::integral_constant<int, S - 1>{});
        meet();  // (the last stage is being read)
    } else {
        v16f acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.f;
        const int h = lane >> 5, lrow = lane & 31;
        const int s16 = lane & 15, q16 = lane >> 4;  // KM: as in the K-major loop above
        const char *x_row = smem + lrow * BK, *w_row = KM ? smem + BT * BK + (8 * (q16 >> 1) + (s16 >> 2)) * 64 + (16 * (q16 & 1) + 4 * (s16 & 3)) * 2
                                                          : smem + BT * BK + lrow * BK;
        const int flip = (lrow & 15) * 16;
        struct Operands {
            v8h x[PART], w[PART];
        };
        int buf = 0;
        auto read = [&](Operands &f, int k0) {
#pragma unroll
            for (int k = 0; k < PART; k++) {
                const int slot = ((2 * (k0 + k) + h) * 16) ^ flip;
                f.x[k] = *reinterpret_cast<const v8h *>(x_row + buf + slot);
                if constexpr (KM) {
                    union {
                        v4s s[2];
                        v8h h;
                    } u;
                    u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(w_row + buf + (k0 + k) * 16 * 64));
                    u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(w_row + buf + (k0 + k) * 16 * 64 + 4 * 64));
                    f.w[k] = u.h;
                } else {
                    f.w[k] = *reinterpret_cast<const v8h *>(w_row + buf + slot);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto multiply = [&](const Operands &f) {
#pragma unroll
            for (int k = 0; k < PART; k++) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.w[k], f.x[k], acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto next_stage = [&]() {
            __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the stage has been read before the barrier that gives its buffer away
            buf = buf == (S - 1) * STAGE ? 0 : buf + STAGE;
            meet();
        };
        Operands f0, f1;
        meet();
        read(f0, 0);
        if constexpr (PART == KKN) {
            int left = nk - 1;
            for (; left >= 2; left -= 2) {
                next_stage();
                read(f1, 0);
                multiply(f0);
                next_stage();
                read(f0, 0);
                multiply(f1);
            }
            if (left == 1) {  // uniform
                next_stage();
                read(f1, 0);
                multiply(f0);
                multiply(f1);
            } else {
                multiply(f0);
            }
        } else {
            for (int left = nk; left > 1; left--) {
                read(f1, PART);
                multiply(f0);
                next_stage();
                read(f0, 0);
                multiply(f1);
            }
            read(f1, PART);
            multiply(f0);
            multiply(f1);
        }
        meet();
        // lane holds row lane % 32 and, per register quad q, columns 8 q + 4 (lane / 32) ..
#pragma unroll
        for (int q = 0; q < 4; q++)
            *reinterpret_cast<v4f *>(tile + lrow * RP + 8 * q + 4 * h) = v4f{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    }
    __syncthreads();
    if (!loads) return;
    const int64_t o_base = o.view ? (int64_t)(batch / o.v_nb2) * o.vs_nb1 + (int64_t)(batch % o.v_nb2) * o.vs_nb2
                                  : (int64_t)batch * o.o_batch;
    const __amdgpu_buffer_rsrc_t ores = rsrc(o.out + o_base, o.o_bytes);
    const ViewDiv by_m2(o.view ? o.v_m2 : 1, g.M), by_n2(o.view ? o.v_n2 : 1, g.N);
    const int m = m_base + qm, n = n_base + qn;
    const float *at = tile + qm * RP + qn;
    const v4f sum = across ? v4f{at[0], at[RP], at[2 * RP], at[3 * RP]} : *reinterpret_cast<const v4f *>(at);
    const bool inside = m < g.M && n < g.N;
    if constexpr (EPI == 0) {
        const v4i v = v4i{__float_as_int(sum[0]), __float_as_int(sum[1]), __float_as_int(sum[2]), __float_as_int(sum[3])};
        __builtin_amdgcn_raw_buffer_store_b128(v, ores, inside ? (int)((uint32_t)m * o.ldo + (uint32_t)n * 4) : (int)kOob, 0, kOutAux);
        return;
    }
    // ADD of the bias in fp32 (one rounding), CAST to fp16, the activation, the ADD of the residual: as above
    uint32_t b[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float v = o.bias != nullptr ? sum[e] + bias_r[e] : sum[e];
        b[e] = __builtin_bit_cast(unsigned short, (_Float16)v);
    }
    uint4 piece = make_uint4(b[0] | (b[1] << 16), b[2] | (b[3] << 16), 0, 0);
    uint32_t off = inside ? (uint32_t)m * o.ldo + (uint32_t)n * 2 : kOob;
    if (o.view && inside) {  // uniform
        const uint32_t m1 = by_m2.quotient((uint32_t)m), n1 = by_n2.quotient((uint32_t)n);
        off = m1 * o.vs_m1 + ((uint32_t)m - m1 * (uint32_t)o.v_m2) * (across ? 2u : o.vs_m2) + n1 * o.vs_n1 +
              ((uint32_t)n - n1 * (uint32_t)o.v_n2) * (across ? o.vs_n2 : 2u);
    }
    if (g.act[0] != nullptr && !across) piece = gelu_tanh_piece(piece, act_c);  // uniform
    if (g.res != nullptr && !across) {  // uniform
        typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
        piece.x = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, piece.x) + __builtin_bit_cast(h2_t, (uint32_t)res_r.x));
        piece.y = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, piece.y) + __builtin_bit_cast(h2_t, (uint32_t)res_r.y));
    }
    __builtin_amdgcn_raw_buffer_store_b64(v2i{(int)piece.x, (int)piece.y}, ores, (int)off, 0, kOutAux);
}

template <bool KM>
void launch_few(const HGemmArgs &args, int cus, bool cast_epilogue, hipStream_t s) {
    HGemmArgs g = args;
    g.tiles_n_group = (g.N + 31) / 32;
    const int tiles_m = (g.M + 31) / 32, tiles_n = g.tiles_n_group * g.groups;
    g.total_tiles = tiles_m * tiles_n * g.batches;
    g.chunk = (g.total_tiles + 7) / 8;
    g.order = make_tile_order(tiles_m, tiles_n, g.chunk, 32, 32);
    g.div_group = make_div_magic((uint32_t)g.tiles_n_group);
    constexpr size_t sm = (size_t)kFewStages * 2 * 32 * 256;
    static_assert(sm <= 64 * 1024, "the default limit of dynamic shared memory");
    auto kernel = g.total_tiles <= cus ? (cast_epilogue ? gemm_f16_few_kernel<8, 1, KM> : gemm_f16_few_kernel<8, 0, KM>)
                                       : (cast_epilogue ? gemm_f16_few_kernel<4, 1, KM> : gemm_f16_few_kernel<4, 0, KM>);
    kernel<<<dim3((unsigned)(g.chunk * 8)), dim3(320), sm, s>>>(g);
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int BKH, bool BROWS = false>
void launch_k(const HGemmArgs &args, bool cast_epilogue, dim3 grid, hipStream_t s) {
    HGemmArgs g = args;
    // (the largest tiles, one to a compute unit, want larger savings: 4096^3, 67 %, 131 us row by row, 140 in bands;
    // 2048 x 4096 x 4096, 47 %, 97 and 93)
    g.order = make_tile_order((g.M + BM - 1) / BM, (int64_t)g.tiles_n_group * g.groups, g.chunk, BM, BN, BM * BN >= 256 * 192 ? 60 : 70);
    g.div_group = make_div_magic((uint32_t)(g.tiles_n_group > 0 ? g.tiles_n_group : 1));
    constexpr int NT = 64 * WAVES_M * WAVES_N;
    constexpr size_t operands = BROWS ? (size_t)ring_stages(BM, BN, BKH) * (BM + ring_w_pieces(BN, NT, BKH) * NT * 8 / BKH) * BKH * 2
                                      : (size_t)2 * BM * (BKH * 2 + 16) + (size_t)2 * BKH * (2 * BN + 32);
    constexpr size_t result = std::max((size_t)BM * (BN * 2 + 16), (size_t)BN * (BM * 2 + 16));
    constexpr size_t sm = std::max(operands, result);
    static_assert(sm <= 160 * 1024, "shared memory of a compute unit");
    // above the default dynamic shared-memory limit the limit is raised once per kernel (thread-safe static)
    if (cast_epilogue) {
        auto kernel = gemm_f16_kernel<BM, BN, WAVES_M, WAVES_N, 1, BKH, BROWS>;
        static const bool raised = sm <= 48 * 1024 || hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm) == hipSuccess;
        (void)raised;
        kernel<<<grid, dim3(64 * WAVES_M * WAVES_N), sm, s>>>(g);
    } else {
        auto kernel = gemm_f16_kernel<BM, BN, WAVES_M, WAVES_N, 0, BKH, BROWS>;
        static const bool raised = sm <= 48 * 1024 || hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm) == hipSuccess;
        (void)raised;
        kernel<<<grid, dim3(64 * WAVES_M * WAVES_N), sm, s>>>(g);
    }
}

template <int BM, int BN, int WAVES_M, int WAVES_N>
void launch(const HGemmArgs &g, bool cast_epilogue, dim3 grid, hipStream_t s) {
    if (g.K >= 256)
        launch_k<BM, BN, WAVES_M, WAVES_N, 64>(g, cast_epilogue, grid, s);
    else
        launch_k<BM, BN, WAVES_M, WAVES_N, 32>(g, cast_epilogue, grid, s);
}

bool dense_rows(const mlel_tensor *t) { return t->strides[2] == 2 && t->strides[1] >= t->dims[2] * 2; }

// Checks one product against what the kernel's indexing assumes and describes it.  1: described, 0: not a case for
// this kernel, 2: nothing to compute.
int fill_args(const mlel_tensor *out, const mlel_tensor *a, const mlel_tensor *b, const mlel_matmul_attr *attr,
              bool bias_cast, const mlel_tensor *bias, const mlel_tensor *residual, HGemmArgs *filled,
              const mlel_tensor *const *act = nullptr) {
    if (act != nullptr) {
        if (!bias_cast || residual != nullptr || out->rank != 3) return 0;
        for (int k = 0; k < 4; k++)
            if (act[k] == nullptr || act[k]->dtype != MLEL_F16 || numel(act[k]) != 1 || ((uintptr_t)act[k]->ptr % 2) != 0) return 0;
    }
    if (residual != nullptr) {
        if (!bias_cast || residual->dtype != MLEL_F16 || residual->rank != 3 || !same_shape(residual, out)) return 0;
        if (residual->strides[2] != 2 || ((uintptr_t)residual->ptr % 16) != 0 || residual->strides[0] % 16 != 0 ||
            residual->strides[1] % 16 != 0)
            return 0;
        const int64_t rb = residual->dims[1] * residual->strides[1];
        if (rb >= (int64_t(1) << 31) - 64 || residual->strides[1] < residual->dims[2] * 2) return 0;
    }
    if (a->dtype != MLEL_F16 || b->dtype != MLEL_F16 || out->dtype != (bias_cast ? MLEL_F16 : MLEL_F32)) return 0;
    // a six-dimensional output is a strided view [NB1, NB2, M1, M2, N1, N2] of the product (fused fp16 form only)
    mlel_tensor plain_out;
    const mlel_tensor *view = nullptr;
    if (out->rank == 6) {
        if (!bias_cast || residual != nullptr) return 0;
        view = out;
        plain_out = *out;
        plain_out.rank = 3;
        plain_out.dims[0] = out->dims[0] * out->dims[1];
        plain_out.dims[1] = out->dims[2] * out->dims[3];
        plain_out.dims[2] = out->dims[4] * out->dims[5];
        plain_out.strides[2] = 2;
        plain_out.strides[1] = plain_out.dims[2] * 2;
        plain_out.strides[0] = plain_out.dims[1] * plain_out.strides[1];
        out = &plain_out;  // extents for the checks below; the addresses come from the view
        // eight contiguous elements along n2 (strides[5] == 2) or, transposing, along m2 (strides[3] == 2)
        const int inner = view->strides[5] == 2 ? 5 : 3;
        if (view->strides[inner] != 2 || view->dims[inner] % 8 != 0) return 0;
        int64_t span = 16;
        for (int i = 0; i < 6; i++) {
            if (i != inner && (view->strides[i] % 16 != 0 || view->strides[i] < 0)) return 0;
            if (i >= 2) span += (view->dims[i] - 1) * view->strides[i];
        }
        if (span >= (int64_t(1) << 31) - 64) return 0;
    }
    const int osize = bias_cast ? 2 : 4;
    if (bias_cast && bias != nullptr) {
        const int64_t n = numel(bias);
        const bool last_axis = bias->dims[bias->rank - 1] == n && bias->strides[bias->rank - 1] == 4;
        if (bias->dtype != MLEL_F32 || !last_axis || (n != 1 && n != out->dims[2]) || ((uintptr_t)bias->ptr % 4) != 0)
            return 0;
    }
    if (attr->a_zp != 0 || attr->b_zp != 0) return 0;
    const int64_t NB = out->dims[0], M = out->dims[1], N = out->dims[2], K = a->dims[2];
    // what the kernel's indexing assumes: element-contiguous rows, 16-byte aligned rows and bases, K and N in
    // multiples of 8, per-batch extents below 2^31, operands at least as large as the output implies
    if (a->dims[0] < NB || b->dims[0] < NB || a->dims[1] < M || b->dims[1] < K || b->dims[2] < N) return 0;
    // B row-wise: element (k, n) at n * pitch + 2 k, i.e. a [K][N] view of a matrix stored as [N][K] (K > 1, so the
    // two layouts cannot be confused); the direct-to-LDS loop then wants whole 64-byte steps of K
    const bool b_rows = K > 1 && b->strides[1] == 2 && b->strides[2] >= b->dims[1] * 2;
    if (!dense_rows(a) || !(b_rows || dense_rows(b)) || out->strides[2] != osize) return 0;
    if (K % 8 != 0 || N % 8 != 0 || K <= 0 || (b_rows && K % 32 != 0)) return 0;
    auto aligned = [](const mlel_tensor *t) {
        return ((uintptr_t)t->ptr % 16) == 0 && t->strides[0] % 16 == 0 && t->strides[1] % 16 == 0;
    };
    if (!aligned(a) || !aligned(out) || (b_rows ? ((uintptr_t)b->ptr % 16) != 0 || b->strides[0] % 16 != 0 || b->strides[2] % 16 != 0
                                                : !aligned(b)))
        return 0;
    const int64_t lim = (int64_t(1) << 31) - 64;
    const int64_t b_pitch = b_rows ? b->strides[2] : b->strides[1];
    const int64_t ab = a->dims[1] * a->strides[1], bb = (b_rows ? b->dims[2] : b->dims[1]) * b_pitch, ob = M * out->strides[1];
    if (ab >= lim || bb >= lim || ob >= lim || a->strides[1] >= lim || b_pitch >= lim) return 0;
    if (M >= (1 << 24) || N >= (1 << 24) || K >= (1 << 24)) return 0;
    if (NB <= 0 || M <= 0 || N <= 0) return 2;

    HGemmArgs g{};
    g.a = static_cast<const char *>(a->ptr);
    g.b = static_cast<const char *>(b->ptr);
    g.out = static_cast<char *>(out->ptr);
    g.M = (int)M;
    g.N = (int)N;
    g.K = (int)K;
    g.batches = (int)NB;
    g.a_batch = a->strides[0];
    g.b_batch = b->strides[0];
    g.o_batch = out->strides[0];
    g.lda = (uint32_t)a->strides[1];
    g.ldb = (uint32_t)b_pitch;
    g.b_rows = b_rows ? 1 : 0;
    g.ldo = (uint32_t)out->strides[1];
    g.a_bytes = (uint32_t)ab;
    g.b_bytes = (uint32_t)bb;
    g.o_bytes = (uint32_t)ob;
    g.bias = bias_cast && bias != nullptr ? static_cast<const float *>(bias->ptr) : nullptr;
    g.bias_len = bias_cast && bias != nullptr ? (int)numel(bias) : 0;
    if (view != nullptr) {
        g.view = 1;
        g.v_nb2 = (int32_t)view->dims[1];
        g.v_m2 = (int32_t)view->dims[3];
        g.v_n2 = (int32_t)view->dims[5];
        g.vs_nb1 = view->strides[0];
        g.vs_nb2 = view->strides[1];
        g.vs_m1 = (uint32_t)view->strides[2];
        g.vs_m2 = (uint32_t)view->strides[3];
        g.vs_n1 = (uint32_t)view->strides[4];
        g.vs_n2 = (uint32_t)view->strides[5];
        if (view->strides[5] != 2) g.view = 2;
        int64_t span = 16;
        for (int i = 2; i < 6; i++) span += (view->dims[i] - 1) * view->strides[i];
        g.o_bytes = (uint32_t)span;
    }
    if (residual != nullptr) {
        g.res = static_cast<const char *>(residual->ptr);
        g.r_batch = residual->strides[0];
        g.ldr = (uint32_t)residual->strides[1];
        g.r_bytes = (uint32_t)(residual->dims[1] * residual->strides[1]);
    }
    if (act != nullptr)
        for (int k = 0; k < 4; k++) g.act[k] = static_cast<const uint16_t *>(act[k]->ptr);
    g.groups = 1;
    *filled = g;
    return 1;
}

// Tile choice and launch of a described product (or group of products).
int launch_args(mlel_ctx *ctx, hipStream_t s, HGemmArgs &g, bool bias_cast) {
    const int64_t M = g.M, N = g.N, K = g.K, NB = g.batches;
    // tile choice: the width with the least padding of N; the tall tile when it still gives every compute unit two
    // blocks and the contraction is long enough to matter (a K of a few steps is bound by the stores, which the
    // short tile spreads over more blocks), otherwise the short one
    const int BN = ((N + 127) / 128) * 128 <= ((N + 63) / 64) * 64 ? 128 : 64;
    const int cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
    g.tiles_n_group = (int)((N + BN - 1) / BN);
    const int64_t tiles_n = (int64_t)g.tiles_n_group * g.groups;
    const bool tall = K > 128 && ((M + 127) / 128) * tiles_n * NB >= 2 * (int64_t)cus;
    const int BM = tall ? 128 : 64;
    const int64_t total = (M + BM - 1) / BM * tiles_n * NB;
    MLEL_REQUIRE(total < (int64_t(1) << 30), MLEL_ERR_LIMIT, "matmul: %lld tiles", (long long)total);
    g.total_tiles = (int)total;
    g.chunk = (int)((total + 7) / 8);
    const dim3 grid((unsigned)(g.chunk * 8));
    // Eight wavefronts on the 128 x 128 tile when a compute unit gets at most three tiles: with so few blocks
    // resident nothing else hides the per-step barrier and LDS round trip (4096 x 768 x 3072: 36.4 -> 33.3 us); with
    // more tiles the four-wavefront blocks overlap each other and the larger wavefront tile wins.
    // A contraction of some length over few tiles (4096 x 3072 x 768 and 4096 x 768 x 768: 192 tiles of 128 x 128):
    // the eight-wavefront tile even when it leaves a quarter of the compute units idle, 43.1 -> 38.4 us and
    // 15.5 -> 13.7 us against 384 short tiles
    const int64_t tiles128 = ((M + 127) / 128) * tiles_n * NB;
    // The 256 x 256 tile of eight wavefronts (128 x 64 each: a third fewer operand reads from shared memory per
    // multiply) when it still occupies three quarters of the compute units: 4096 x 768 x 3072 in 192 tiles,
    // 37.7 -> 34.7 us.  With fewer tiles the idle compute units cost more than the reads (144 tiles: no gain;
    // 48 tiles: twice the time).  With the K-major loop an activation in the epilogue loses too, its arithmetic
    // running on three quarters of the machine (the same product with the tanh GELU: 40.9 -> 44.1 us); with the
    // direct-to-LDS loop it gains a little (38.4 -> 37.3 us inside the encoder block), so that path takes the large
    // tile with or without one.
    const int64_t tiles256 = ((M + 255) / 256) * ((N + 255) / 256) * NB;
    if (g.b_rows) {
        // Row-wise B: the direct-to-LDS loop, whatever the extents (rows beyond M or N are fetched as zeros).
        const auto tiles_of = [&](int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn) * g.groups * NB; };
        const auto go = [&](auto bm, auto bn, auto wm, auto wn, auto bkh) {
            constexpr int BM = decltype(bm)::value, BN = decltype(bn)::value;
            g.tiles_n_group = (int)((N + BN - 1) / BN);
            const int64_t t = tiles_of(BM, BN);
            g.total_tiles = (int)t;
            g.chunk = (int)((t + 7) / 8);
            launch_k<BM, BN, decltype(wm)::value, decltype(wn)::value, decltype(bkh)::value, true>(g, bias_cast, dim3((unsigned)(g.chunk * 8)), s);
        };
        MLEL_REQUIRE(tiles_of(64, 64) < (int64_t(1) << 30), MLEL_ERR_LIMIT, "matmul: %lld tiles", (long long)tiles_of(64, 64));
        constexpr std::integral_constant<int, 2> two;
        constexpr std::integral_constant<int, 4> four;
        constexpr std::integral_constant<int, 32> k32;
        constexpr std::integral_constant<int, 64> k64, t64;
        constexpr std::integral_constant<int, 128> t128;
        constexpr std::integral_constant<int, 192> t192;
        constexpr std::integral_constant<int, 256> t256;
        const bool whole64 = K % 64 == 0;
        const auto fills = [&](int64_t tiles, int64_t most) { return tiles * 4 >= 3 * (int64_t)cus && tiles <= most; };
        // - Up to two tiles of 32 x 32 per compute unit: gemm_f16_few_kernel.  us, 64 x 64 / there: 16 x 192 x 192 3.0 / 2.7,
        //   64 x 768 x 2304 (144 tiles) 5.3 / 3.4, 197 x 1536 x 384 (84) 7.0 / 4.4, 197 x 1536 x 2304 (504) 7.3 / 6.2, 512 x 768 x 1536
        //   (768) 5.6 / 6.6.
        // - One or two tiles of 64 x 64 per compute unit: 64 x 64 over four wavefronts.  An encoder block of 8 x 197 rows, 768
        //   columns: 107.7 -> 100.7 us with the line at two tiles per unit, 105.7 at four.
        // - 256 rows where three quarters of the compute units get a tile: a third fewer operand reads from shared memory per
        //   multiply.  256 x 192 where that is one round: the wider tile would then be one round too, of a
        //   third more work per unit (4096 x 768 x 3072 with the GELU, 256 tiles against 192: an encoder block 137 -> 132 us), or
        //   leave units idle (4096 x 768 x 2304, 192 tiles: 27.2 -> 23.4 us against 576 of 128 x 128).
        // - 128 x 128 over eight wavefronts otherwise.
        // Steps of 64 halfs, half as many of them at twice the shared memory: for the tiles that have a compute unit to themselves
        // anyway (4096 x 3072 x 768: 30.2 -> 25.1 us, 878 x 896 x 3584: 14.0 -> 12.1, even at K = 768 and below), and for the
        // 64 x 64 tile, of which two still fit (1576 x 3072 x 768: 25.0 -> 19.9).
        if (tiles_of(32, 32) <= 2 * (int64_t)cus) {
            launch_few<false>(g, cus, bias_cast, s);
        } else if (tiles_of(64, 64) <= 2 * (int64_t)cus) {
            if (whole64) go(t64, t64, two, two, k64);
            else go(t64, t64, two, two, k32);
        } else if (K >= 256 && fills(tiles_of(256, 192), cus)) {
            go(t256, t192, four, two, k32);
        } else if (g.groups == 1 && K >= 256 && fills(tiles_of(256, 256), 2 * (int64_t)cus)) {
            go(t256, t256, two, four, k32);
        } else if (whole64 && K > 768 && tiles_of(128, 128) <= cus) {
            go(t128, t128, two, four, k64);
        } else {
            go(t128, t128, two, four, k32);
        }
        MLEL_TRY(check_launch("matmul fp16, row-wise B"));
        return 1;
    }
    // K-major B, few tiles: up to two of 32 x 32 per compute unit, three for longer contractions over whole tiles of 128 columns.  us,
    // before / there: 256 x 1024 x 1024 11.7 / 4.6, 64 x 2048 x 4096 19.5 / 6.8, 128^3 4.8 / 2.9, 800 x 768 x 768 (600 tiles) 9.9 / 7.8,
    // 512 x 64 x 2048 (1024) 4.5 / 6.4, 1024^3 (1024) 11.9 / 11.5; other columns, whose tiles of 64 x 64 are not half empty, 705 x 264 x 1032
    // (759) 5.5 / 7.1 (162 such products 10 % slower there, 195 over whole tiles 17 % faster)
    const int64_t tiles32 = ((M + 31) / 32) * ((N + 31) / 32) * g.groups * NB;
    if (tiles32 <= (K >= 256 && BN == 128 ? 3 : 2) * (int64_t)cus) launch_few<true>(g, cus, bias_cast, s);
    else if (BN == 128 && g.groups == 1 && g.act[0] == nullptr && g.K >= 256 && tiles256 * 4 >= 3 * (int64_t)cus && tiles256 <= 2 * (int64_t)cus) {
        g.tiles_n_group = (int)((N + 255) / 256);
        g.total_tiles = (int)tiles256;
        g.chunk = (int)((tiles256 + 7) / 8);
        launch_k<256, 256, 2, 4, 32>(g, bias_cast, dim3((unsigned)(g.chunk * 8)), s);
    } else if (BN == 128 && !tall && g.K >= 512 && tiles128 * 5 >= 3 * (int64_t)cus) {
        g.total_tiles = (int)tiles128;
        g.chunk = (int)((tiles128 + 7) / 8);
        launch_k<128, 128, 2, 4, 64>(g, bias_cast, dim3((unsigned)(g.chunk * 8)), s);
    } else if (BN == 128 && tall && g.K >= 256 && total <= 3 * (int64_t)cus)
        launch_k<128, 128, 2, 4, 64>(g, bias_cast, grid, s);
    else if (BN == 128 && tall)
        launch<128, 128, 2, 2>(g, bias_cast, grid, s);
    else if (BN == 128)
        launch<64, 128, 1, 4>(g, bias_cast, grid, s);
    else if (tall)
        launch<128, 64, 2, 2>(g, bias_cast, grid, s);
    else
        launch<64, 64, 2, 2>(g, bias_cast, grid, s);
    MLEL_TRY(check_launch("matmul fp16"));
    return 1;
}

}  // namespace

// `bias_cast` set: the fused form out(fp16) = CAST(MATMUL + bias) with an fp32 bias of length 1 or N (or none)
int try_matmul_f16_mfma(mlel_ctx *ctx, hipStream_t s, const mlel_tensor *out, const mlel_tensor *a,
                        const mlel_tensor *b, const mlel_matmul_attr *attr, bool bias_cast, const mlel_tensor *bias,
                        const mlel_tensor *residual, const mlel_tensor *const *gelu_inputs) {
    HGemmArgs g{};
    const int rc = fill_args(out, a, b, attr, bias_cast, bias, residual, &g, gelu_inputs);
    if (rc != 1) return rc == 2 ? 1 : 0;
    // A K-major B with an fp32 result, more than two tiles of 32 x 32 per compute unit: contract_float.hip's loop is faster, told to
    // add K in this file's order, unless the 256 x 256 tile has a long contraction or a narrow result with a short one is all
    // stores.  us, here / there: 500 x 2048 x 2048 20.1 / 12.6, 1024^3 12.1 / 8.0, 2048^3 30.0 / 25.5, 4096 x 768 x 3072 39.9 / 34.4,
    // 4096 x 1024 x 4096 57.5 / 56.2, 4096 x 2048 x 4096 88 / 100, 4096 x 3072 x 3072 104 / 103, 4096^3 139 / 171, 2048 x 8192 x
    // 2048 (64 tiles of 256) 93 / 84; 8192 x 32 x 64 3.2 / 3.5, 8192 x 128 x 64 3.8 / 3.9, 4096 x 64 x 64 3.3 / 3.2.
    // Of 4000 such products the kernels here are faster for (mean time there, of here)
    // - at most 32 rows, K below 512, up to two tiles of 64 x 64 per unit, eight for K up to 128, or 32 columns, 24 for K up to 72, up to
    //   five tiles: 1.2 (9 x 2 x 72 x 2416 3.5 us here, 4.9 there, 23 x 2576 x 88 x 8 4.5, 8.3)
    // - N whose last 64 columns a tile of 128 would leave empty and a K of no whole steps, up to a tile of 64 x 64 per unit, or one and a
    //   half beyond K = 72: 1.06 (705 x 264 x 1032 5.2, 6.9)
    // - other N, less than a round of tiles of 128 x 128 on five eighths of the units or more from K = 768 on, four fifths from 400: 1.15
    //   (3356 x 1928 x 1112 30.1, 43.4)
    // - up to an eighth more tiles of 128 x 128 than units, beyond a short K: 1.04 (22 x 183 x 56 x 672 6.9, 9.0)
    // and the others, on average, slower: 0.88
    if (!bias_cast && !g.b_rows) {
        const int64_t cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
        const auto tiles = [&](int64_t t) { return ((g.M + t - 1) / t) * ((g.N + t - 1) / t) * g.batches; };
        const bool large = tiles(256) * 2 >= cus && g.K * std::min(tiles(256), cus) >= 2048 * cus;
        const bool wide = (g.N + 127) / 128 * 128 <= (g.N + 63) / 64 * 64;  // (launch_args' condition for 128 columns)
        const bool thin = g.M <= 32 ? g.K < 512 && tiles(64) <= (g.K <= 128 ? 8 : 2) * cus : g.N <= (g.K > 72 ? 32 : 24) && tiles(64) <= 5 * cus;
        const bool narrow = !wide && g.K % 64 != 0 && tiles(64) * 2 <= (g.K > 72 ? 3 : 2) * cus;
        const bool round = wide && g.M > 64 && tiles(128) * 8 >= 5 * cus && tiles(128) < cus && g.K >= (tiles(128) * 5 >= 4 * cus ? 400 : 768);
        const bool second = g.K > (wide ? 128 : 32) && g.M > 64 && g.N > 64 && tiles(128) > cus && tiles(128) * 8 <= 9 * cus;
        const bool here = large || thin || narrow || round || second || (g.N <= 64 && g.K <= 128 && g.M >= 8192);
        if (tiles(32) > 2 * cus && !here) {
            const int there = try_matmul_float(ctx, s, out, a, b, attr, nullptr, false, true);
            if (there != 0) return there;
        }
    }
    return launch_args(ctx, s, g, bias_cast);
}

// Whether a product with a row added behind it is better off here, the ADD a pass of its own over the result, than in the kernel
// that adds in its epilogue (contract_float.hip): where this file's 256 x 256 tile applies and K is long enough for its faster
// loop to pay for the pass.  us, apart / there -- K-major B: 4096 x 2048 x 4096 110 / 105, 4096 x 3072 x 4096 141 / 146, 4096^3
// 167 / 189, 3072 x 4096 x 4096 (192 tiles) 143 / 141, 4096 x 2048 x 8192 214 / 210, 4096 x 4096 x 8192 337 / 379; row-wise B:
// 4096 x 1024 x 4096 74 / 61, 4096 x 2048 x 4096 101 / 102, 4096 x 3072 x 4096 128 / 146, 3072 x 4096 x 4096 124 / 141.
bool matmul_f16_then_add(mlel_ctx *ctx, const mlel_tensor *out, const mlel_tensor *a, const mlel_tensor *b, const mlel_matmul_attr *attr) {
    HGemmArgs g{};
    if (a->dtype != MLEL_F16 || fill_args(out, a, b, attr, false, nullptr, nullptr, &g) != 1) return false;
    const int64_t cus = ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
    const int64_t tiles = ((int64_t)(g.M + 255) / 256) * ((g.N + 255) / 256) * g.batches;
    const bool wide = g.b_rows || (g.N + 127) / 128 * 128 <= (g.N + 63) / 64 * 64;  // (launch_args' condition for that tile)
    return wide && tiles * 4 >= 3 * cus && tiles <= 2 * cus && g.K * std::min(tiles, cus) >= (g.b_rows ? 2048 : 3072) * cus;
}

// Up to three fused products of one A in a single launch; 0 unless every product is a case for the kernel and they
// agree in everything but their B, bias and output.
int try_matmul_f16_group(mlel_ctx *ctx, hipStream_t s, int n, const mlel_tensor *const *outs, const mlel_tensor *a,
                         const mlel_tensor *const *bs, const mlel_tensor *const *biases, const mlel_matmul_attr *attr) {
    if (n < 2 || n > 3) return 0;
    HGemmArgs g[3];
    for (int i = 0; i < n; i++) {
        if (fill_args(outs[i], a, bs[i], attr, true, biases[i], nullptr, &g[i]) != 1) return 0;
        const HGemmArgs &x = g[i], &y = g[0];
        if (x.M != y.M || x.N != y.N || x.K != y.K || x.batches != y.batches || x.ldb != y.ldb || x.b_rows != y.b_rows || x.b_bytes != y.b_bytes ||
            (x.batches > 1 && x.b_batch != y.b_batch) || x.bias_len != y.bias_len || (x.bias == nullptr) != (y.bias == nullptr))
            return 0;
    }
    for (int i = 1; i < n; i++) {
        const HGemmArgs &x = g[i];
        g[0].extra[i - 1] = HGemmArgs::Extra{x.b, x.bias, x.out, x.o_batch, x.ldo, x.o_bytes, x.view, x.v_nb2, x.v_m2, x.v_n2,
                                             x.vs_nb1, x.vs_nb2, x.vs_m1, x.vs_m2, x.vs_n1, x.vs_n2};
    }
    g[0].groups = n;
    return launch_args(ctx, s, g[0], true);
}

}  // namespace mlel
