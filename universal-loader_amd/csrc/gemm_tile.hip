// gemm_tile.hip -- the dequant-GEMM for many rows (prompts, batches): a tile of
// Y per workgroup on 32x32x16 fp16 MFMAs, X staged through LDS, the weights
// dequantized in registers.
//
// Workgroup: 8 waves over ROWS staged rows x 256 columns; wave w owns columns
// 32 w .. 32 w + 31 and all the rows, so every weight is loaded and
// dequantized once per workgroup and never passes through LDS.  K advances in
// stages of 256 elements (a super-block, or two 128-element chunks):
//   - X of stage s + 1 goes to the other LDS buffer by direct buffer->LDS
//     copies, and the raw weights of s + 1 to registers, while stage s is
//     multiplied; one barrier per stage.
//   - Waves 0-3 dequantize stage s + 1 at the end of stage s, waves 4-7 at the
//     start of stage s + 1: a SIMD's two waves are in opposite phases, one on
//     the vector unit while the other feeds the matrix cores.
// The products are the exact fp16 ones of the other kernels (Q4_K q * sc with
// the mins against sub-block sums of X, Q6_K (q - 32) sc, Q4_0 / Q8_0 per
// block), scaled by the block's d as fp32 on the way into the accumulator, in
// K order.
//
// Operands of a 32x32x16 MFMA: lane l supplies row (A) or column (B) l & 31
// and 8 K values of half kg = l >> 5, and holds C rows 8 (i / 4) + 4 kg + i % 4
// of column l & 31.  Column l & 31 is row l & 15 of weight tile (l >> 4) & 1
// of the wave's two; the half kg takes the weight layout's lane groups kg
// and kg + 2 in two steps.
//
// X in LDS: [4 segments of 64 K][ROWS][8 units of 16 B], unit u of row r at
// position u ^ ((r / 2) & 7): the copies read whole 128-byte lines, and the 16
// rows of an operand read land in 16 distinct 16-byte bank groups.
//
// Measured against the 64-row launches of the split-K kernel it replaces (which
// reads and dequantizes the whole weight once per 64 rows), at 2048 x 11008 x
// 4096: Q4_K 869 -> 202 us (0.92 PFLOP/s), Q4_0 240, Q8_0 266 (a block's scale
// per 32 K: twice the accumulator updates of the super-block types), Q6_K 217,
// F16 214 us; 333 x 4096 x 4096 Q8_0 79.9 -> 32.3 us.  Bound by the vector unit
// beside the matrix cores: dequantization, and the scaling of every product.
#include "gemm_dev.h"

#include <algorithm>
#include <utility>

using namespace ulspec;

namespace {

constexpr int kTileWaves = 8;
constexpr int kTileCols = 32 * kTileWaves;  // columns of a workgroup
constexpr int kTileXcds = 8;

struct TileArgs {
    GemmArgs a;
    const uint4* xsum;  // Q4_K: sub-block sums of X (tile_sums_kernel), [K / 256][xsum_rows][2]
    int xsum_rows;
    int n_stages;       // ceil(K / 256)
    int tm, tn;         // row and column blocks
    // Blocks 0 .. n_full - 1 take a workgroup each, the n_part others a.ks_count
    // workgroups: slices of st_q or st_q + 1 stages (n_stages = st_q ks_count +
    // st_r), left as fp32 parts for tile_fixup_kernel.
    int n_full, n_part;
    int st_q, st_r;
    float* part;        // [n_part][ks_count][rows of a block][kTileCols]
};

// Row and column block i: 8 row blocks before the next column block, so the ~32
// resident workgroups of an XCD share 8 X blocks and a few weight blocks in its L2.
__device__ __forceinline__ void block_at(const TileArgs& ta, int i, int& mb, int& nb)
{
    constexpr int GM = 8;
    const int grp = i / (GM * ta.tn), first = grp * GM, in = i - grp * GM * ta.tn;
    const int gm = min(GM, ta.tm - first);
    mb = first + in % gm;
    nb = in / gm;
}

// One stage of a wave's weights as loaded: the chunk pieces of lane groups kg
// and kg + 2.
template <int TYPE>
struct TileRaw;
template <>
struct TileRaw<ULSPEC_GGML_Q4_K> {
    uint4 w[2][2], hd;
};
template <>
struct TileRaw<ULSPEC_GGML_Q6_K> {
    uint4 w[2][2], hb[2];
    uint32_t sc[2], d;
};
template <>
struct TileRaw<ULSPEC_GGML_Q4_0> {
    uint4 w[2][2];  // [chunk][s]
    uint2 sc[2];
};
template <>
struct TileRaw<ULSPEC_GGML_Q8_0> {
    uint4 w[2][2][2];  // [chunk][s][half]
    uint2 sc[2];
};
template <>
struct TileRaw<ULSPEC_GGML_F16> {};  // loaded as B operands (tile_load_f16)

// The same, dequantized: B operands f = 8 s + j (super-block types) or 8 c +
// 2 j + s (128-element chunks c of blocks j), and what scales their products.
template <int TYPE>
struct TileW {
    half8_t f[16];
    float d[kSuperBlock<TYPE> ? 2 : 8];  // Q4_K: d, -dmin; Q6_K: d; per block otherwise
    half8_t mins;                        // Q4_K
};

template <int TYPE>
constexpr int kChunkBytes = TYPE == ULSPEC_GGML_Q4_K   ? kQ4KChunk
                            : TYPE == ULSPEC_GGML_Q6_K ? kQ6KChunk
                            : TYPE == ULSPEC_GGML_Q4_0 ? kQ40Chunk
                            : TYPE == ULSPEC_GGML_Q8_0 ? kQ80Chunk
                                                       : kF16Chunk;

__device__ __forceinline__ uint4 load16_at(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff)
{
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
}

// Chunk pieces of stage st (K from 256 st) for this lane.  base: offset of the
// first chunk of this lane's tile, or kOOB past the last tile (kOOB plus any
// offset in a chunk row is out of range too).
template <int TYPE>
__device__ __forceinline__ void tile_load(const GemmArgs& a, __amdgpu_buffer_rsrc_t wr, uint32_t base, int st,
                                          TileRaw<TYPE>& w)
{
    const int lane = threadIdx.x & 63, r = lane & 15, kg = lane >> 5;
    const uint32_t pl = base + (uint32_t)(r + 16 * kg) * 16u;  // lane group kg; kg + 2 is 512 bytes on
    if constexpr (kSuperBlock<TYPE>) {
        const uint32_t so = (uint32_t)st * kChunkBytes<TYPE>;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int p = 0; p < 2; ++p) w.w[s][p] = load16_at(wr, pl + 512 * s + 1024 * p, so);
        if constexpr (TYPE == ULSPEC_GGML_Q4_K) {
            w.hd = load16_at(wr, base + r * 16 + 2048, so);
        } else {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                w.hb[s] = load16_at(wr, pl + 2048 + 512 * s, so);
                w.sc[s] = __builtin_amdgcn_raw_buffer_load_b32(wr, base + r * 16 + kg * 4 + 3072 + 8 * s, so, 0);
            }
            w.d = __builtin_amdgcn_raw_buffer_load_b16(wr, base + r * 2 + 3328, so, 0);
        }
    } else {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const bool ok = 2 * st + c < a.n_chunks;  // uniform: an odd chunk count's last stage holds one
            const uint32_t so = (uint32_t)(2 * st + c) * kChunkBytes<TYPE>;
            const uint32_t o = ok ? pl : kOOB;
            constexpr int NP = TYPE == ULSPEC_GGML_Q8_0 ? 2 : 1;
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    const uint4 v = load16_at(wr, o + 512 * s + 1024 * p, so);
                    if constexpr (TYPE == ULSPEC_GGML_Q8_0) w.w[c][s][p] = v;
                    else w.w[c][s] = v;
                }
            w.sc[c] = __builtin_bit_cast(
                uint2, __builtin_amdgcn_raw_buffer_load_b64(wr, (ok ? base + r * 8 : kOOB) + 1024 * NP, so, 0));
        }
    }
}

// F16: the B operands of chunk c of stage st.
__device__ __forceinline__ void tile_load_f16(const GemmArgs& a, __amdgpu_buffer_rsrc_t wr, uint32_t base, int st, int c,
                                              half8_t (&f)[16])
{
    const int lane = threadIdx.x & 63;
    const uint32_t o = 2 * st + c < a.n_chunks ? base + (uint32_t)((lane & 15) + 16 * (lane >> 5)) * 16u : kOOB;
    const uint32_t so = (uint32_t)(2 * st + c) * kF16Chunk;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int s = 0; s < 2; ++s)
            f[8 * c + 2 * j + s] = __builtin_bit_cast(half8_t, load16_at(wr, o + 1024 * j + 512 * s, so));
}

__device__ __forceinline__ uint32_t word_of(const uint4& v, int j)
{
    return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
}

__device__ __forceinline__ float half_of(const uint2& v, int j)
{
    return half_bits_to_float(((j < 2 ? v.x : v.y) >> (16 * (j & 1))) & 0xffffu);
}

template <int TYPE>
__device__ __forceinline__ void tile_dequant(const TileRaw<TYPE>& w, const NibbleConsts& nk, TileW<TYPE>& o)
{
    const int kg = (threadIdx.x & 63) >> 5;
    if constexpr (TYPE == ULSPEC_GGML_Q4_K) {
        o.d[0] = half_bits_to_float(w.hd.x & 0xffffu);
        o.d[1] = -half_bits_to_float(w.hd.x >> 16);
        // group g's 24 bits at 24 g of y, z, w: g = kg at bit 24 kg of z:y, g = kg + 2 at 16 + 24 kg of w:z
        const uint32_t b0 = (uint32_t)(((uint64_t)w.hd.z << 32 | w.hd.y) >> (24 * kg));
        const uint32_t b1 = (uint32_t)(((uint64_t)w.hd.w << 32 | w.hd.z) >> (16 + 24 * kg));
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const uint32_t bits = s ? b1 : b0;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const _Float16 hs = (_Float16)(uint16_t)((bits >> (6 * e)) & 63u);  // exact, as are the products below
                SubScale ss;
                ss.sc = half2_t{hs, hs};
                ss.nsc1024 = ss.sc * splat2(-1024.0f);
                ss.sc16 = ss.sc * splat2(0.0625f);
                ss.nsc64 = ss.sc * splat2(-64.0f);
#pragma unroll
                for (int j = 0; j < 4; ++j) o.f[8 * s + 4 * e + j] = dequant_q4_k(word_of(w.w[s][e], j), ss, nk);
                const _Float16 hm = (_Float16)(uint16_t)((bits >> (12 + 6 * e)) & 63u);
                o.mins[4 * s + 2 * e] = hm * (_Float16)32.0f;
                o.mins[4 * s + 2 * e + 1] = hm * (_Float16)0.015625f;
            }
        }
    } else if constexpr (TYPE == ULSPEC_GGML_Q6_K) {
        const Q6Consts k6 = q6_consts();
        o.d[0] = half_bits_to_float(w.d & 0xffffu);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const Q6Scale sc = q6_scale((int)(int8_t)(w.sc[s] >> (8 * (j >> 1))));
                const uint32_t hw = word_of(w.hb[s], j >> 1);
                o.f[8 * s + j] = dequant_q6_k(word_of(w.w[s][j >> 2], j & 3), (j & 1) ? hw >> 2 : hw, sc, nk, k6);
            }
    } else {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                o.d[4 * c + j] = half_of(w.sc[c], j);
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    half8_t& f = o.f[8 * c + 2 * j + s];
                    if constexpr (TYPE == ULSPEC_GGML_Q8_0)
                        f = dequant_q8_0(word_of(w.w[c][s][j >> 1], 2 * (j & 1)),
                                         word_of(w.w[c][s][j >> 1], 2 * (j & 1) + 1));
                    else f = dequant_q4_0(word_of(w.w[c][s], j), nk);
                }
            }
    }
}

// f(integral_constant 0) .. f(integral_constant N - 1): a loop whose indexes are
// constants before any optimisation, so register arrays stay in registers.
template <class F, int... I>
__device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, F f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void unrolled(F f)
{
    unrolled(std::make_integer_sequence<int, N>{}, f);
}

// Keeps the accumulator's update here, and the instructions of one item (see
// the main loop) from moving into another.
__device__ __forceinline__ void pin(float16_t& v)
{
    asm volatile("" : "+v"(v));
    __builtin_amdgcn_sched_barrier(0);
}

constexpr size_t tile_lds_bytes(int rows) { return (size_t)2 * rows * 512 + (size_t)2 * rows * 32; }

// MT: 32-row operand tiles of staged rows.  HL: tiles 0 .. MT / 2 - 1 are high
// parts of rows m0 .., tiles MT / 2 .. the low parts of the same rows.
template <int TYPE, int MT, bool HL>
__global__ __launch_bounds__(kTileWaves * 64, 2) void gemm_tile_kernel(TileArgs ta)
{
    static_assert(!HL || MT % 2 == 0, "high and low tiles");
    constexpr bool kSums = TYPE == ULSPEC_GGML_Q4_K, kF16 = TYPE == ULSPEC_GGML_F16;
    constexpr int ROWS = 32 * MT;                // staged rows
    constexpr int RB = HL ? ROWS / 2 : ROWS;     // rows of Y
    constexpr int SEG = ROWS * 128, BUF = 4 * SEG, SBUF = ROWS * 32;
    constexpr int RBLK = ROWS / 8;               // 8-row blocks of a segment, one 1 KB copy each
    constexpr int NCOPY = 4 * RBLK / kTileWaves; // X copies of a wave per stage
    constexpr int NR = RBLK > kTileWaves ? RBLK / kTileWaves : 1;  // row blocks a wave copies
    extern __shared__ uint4 tile_lds[];
    char* const lds = (char*)tile_lds;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)tile_lds;
    const GemmArgs& a = ta.a;

    // Workgroups of one XCD (blockIdx.x % 8) are consecutive blocks, or slices of
    // blocks, of the order of block_at.
    const bool sliced = (int)blockIdx.x >= ta.n_full;
    const int count = sliced ? ta.n_part * a.ks_count : ta.n_full, bid = (int)blockIdx.x - (sliced ? ta.n_full : 0);
    const int per = count / kTileXcds, extra = count % kTileXcds, xcd = bid % kTileXcds;
    const int id = xcd * per + min(xcd, extra) + bid / kTileXcds;
    const int ks = sliced ? id / ta.n_part : 0, u = id - ks * ta.n_part;
    int mb, nb;
    block_at(ta, sliced ? ta.n_full + u : id, mb, nb);

    const int lane = threadIdx.x & 63, kg = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool late = wave >= kTileWaves / 2;
    const int m0 = mb * RB;
    const int t = (nb * kTileCols + 32 * wave) / 16 + ((lane >> 4) & 1);
    const int n = nb * kTileCols + 32 * wave + (lane & 31);
    const uint32_t wbase = t < a.n_tiles ? (uint32_t)t * (uint32_t)a.n_chunks * kChunkBytes<TYPE> : kOOB;
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.w, a.w_bytes);
    const rsrc_words xr = make_words(a.x, x_bytes(a));
    const NibbleConsts nk = nibble_consts();

    // X row behind staged row rho, or -1 past M
    auto xrow = [&](int rho) {
        const int m = m0 + (HL && rho >= RB ? rho - RB : rho);
        return m < a.M ? (HL && rho >= RB ? a.lo_rows + m : m) : -1;
    };
    // this lane's source in each of its row blocks: row byte offset, and its unit
    uint32_t roff[NR];
    int unit[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const int rb = (wave + kTileWaves * i) % RBLK;
        const int row = xrow(rb * 8 + (lane >> 3));
        unit[i] = (lane & 7) ^ (((rb & 1) << 2) | (lane >> 4));
        roff[i] = row < 0 ? kOOB : (uint32_t)row * (uint32_t)a.K * 2u + (uint32_t)unit[i] * 16u;
    }
    const int srow = wave * 32 + (lane >> 1);  // staged row of the sums' copy
    const uint32_t soff = kSums && srow < ROWS && xrow(srow) >= 0 ? (uint32_t)(xrow(srow) * 2 + (lane & 1)) * 16u : kOOB;
    const rsrc_words sr =
        make_words(ta.xsum, kSums ? (uint32_t)ta.xsum_rows * (uint32_t)ta.n_stages * 32u : 0u);
    auto copy = [&](int st, int buf) {
#pragma unroll
        for (int i = 0; i < NCOPY; ++i) {
            const int q = wave + kTileWaves * i, rb = q % RBLK, seg = q / RBLK;
            const int k0 = 256 * st + 64 * seg;
            copy_lds(xr, lds0 + (uint32_t)(buf * BUF + seg * SEG + rb * 1024),
                     k0 + 8 * unit[i % NR] < a.K ? roff[i % NR] : kOOB, (uint32_t)k0 * 2u);
        }
        if constexpr (kSums) {
            if (wave < ROWS / 32)
                copy_lds(sr, lds0 + (uint32_t)(2 * BUF + buf * SBUF + wave * 1024),
                         soff, (uint32_t)st * (uint32_t)ta.xsum_rows * 32u);
        }
    };

    // A operands: staged row 32 mt + (lane & 31), units 8 (kg + 2 s) + j of the
    // super-block types, 16 c + 4 j + 2 s + kg otherwise
    const int ar = lane & 31, afr = (ar >> 1) & 7;
    constexpr int NA = kSuperBlock<TYPE> ? 8 : 4;
    int aoff[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i)
        aoff[i] = kSuperBlock<TYPE> ? kg * SEG + ar * 128 + ((i ^ afr) << 4)
                                    : ar * 128 + (((4 * (i >> 1) + 2 * (i & 1) + kg) ^ afr) << 4);
    auto a_op = [&](int buf, int mt, int f) {
        const int o = kSuperBlock<TYPE> ? aoff[(f & 7) % NA] + (f >> 3) * 2 * SEG
                                        : aoff[f & 3] + (2 * (f >> 3) + ((f >> 2) & 1)) * SEG;
        return *(const half8_t*)(lds + buf * BUF + o + mt * 4096);
    };

    const int lo = sliced ? ks * ta.st_q + min(ks, ta.st_r) : 0;
    const int hi = sliced ? lo + ta.st_q + (ks < ta.st_r ? 1 : 0) : ta.n_stages;
    float16_t acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = zero16();
    TileRaw<TYPE> raw;
    TileW<TYPE> w;
    copy(lo, 0);
    if constexpr (kF16) {
        tile_load_f16(a, wr, wbase, lo, 0, w.f);
        tile_load_f16(a, wr, wbase, lo, 1, w.f);
    } else {
        tile_load<TYPE>(a, wr, wbase, lo, raw);
        if (!late) tile_dequant<TYPE>(raw, nk, w);
    }
    for (int st = lo, buf = 0; st < hi; ++st, buf ^= 1) {
        vm_wait<0>();  // this wave's copies of stage st
        lds_barrier();
        if constexpr (!kF16) {
            if (late) tile_dequant<TYPE>(raw, nk, w);
        }
        if (st + 1 < hi) {
            copy(st + 1, buf ^ 1);
            if constexpr (!kF16) tile_load<TYPE>(a, wr, wbase, st + 1, raw);
        }
        // Items of two B operands (64 matrix-core cycles) of one row tile: the A
        // operands are read two items ahead, and the products of the last
        // group (a row tile, or a block of one) are folded into the
        // accumulators behind the next group's first MFMAs.  pin() keeps that
        // order (and the live products at two groups).
        // F16 runs through all row tiles for each chunk, so that the next
        // stage's chunk 0 loads behind the MFMAs of chunk 1 and the reverse.
        constexpr bool kBlocks = !kSuperBlock<TYPE> && !kF16;
        constexpr int NI = 8 * MT, AD = TYPE == ULSPEC_GGML_Q4_K || TYPE == ULSPEC_GGML_Q8_0 ? 2 : 3;
        // item i: row tile and first B operand
        constexpr auto mt_of = [](int i) { return kBlocks ? i % MT : kF16 ? i / 4 % MT : i / 8; };
        constexpr auto f_of = [](int i) { return kBlocks ? 2 * (i / MT) : kF16 ? 8 * (i / (4 * MT)) + 2 * (i % 4) : 2 * (i % 8); };
        half8_t A[AD][2];
        float16_t P[2], P2;
        unrolled<AD - 1>([&](auto i) {
            A[i][0] = a_op(buf, mt_of(i), f_of(i));
            A[i][1] = a_op(buf, mt_of(i), f_of(i) + 1);
        });
        unrolled<NI>([&](auto ic) {
            constexpr int i = decltype(ic)::value, mt = mt_of(i), f = f_of(i);
            if constexpr (i + AD - 1 < NI) {
                constexpr int q = i + AD - 1;
                A[q % AD][0] = a_op(buf, mt_of(q), f_of(q));
                A[q % AD][1] = a_op(buf, mt_of(q), f_of(q) + 1);
            }
            if constexpr (kBlocks) {
                P[i & 1] = mfma32x32x16(A[i % AD][0], w.f[f], zero16());
                P[i & 1] = mfma32x32x16(A[i % AD][1], w.f[f + 1], P[i & 1]);
                if constexpr (i > 0) {
                    constexpr int pm = mt_of(i - 1);
                    acc[pm] = __builtin_elementwise_fma((float16_t)w.d[f_of(i - 1) / 2], P[(i - 1) & 1], acc[pm]);
                    pin(acc[pm]);
                }
            } else if constexpr (kF16) {
                if constexpr (i == NI / 2) {
                    if (st + 1 < hi) tile_load_f16(a, wr, wbase, st + 1, 0, w.f);
                }
                acc[mt] = mfma32x32x16(A[i % AD][0], w.f[f], acc[mt]);
                acc[mt] = mfma32x32x16(A[i % AD][1], w.f[f + 1], acc[mt]);
                pin(acc[mt]);
            } else {
                P[mt & 1] = mfma32x32x16(A[i % AD][0], w.f[f], f == 0 ? zero16() : P[mt & 1]);
                P[mt & 1] = mfma32x32x16(A[i % AD][1], w.f[f + 1], P[mt & 1]);
                if constexpr (kSums && f == 0) {
                    const half8_t s8 = *(const half8_t*)(lds + 2 * BUF + buf * SBUF + (32 * mt + ar) * 32 + kg * 16);
                    P2 = mfma32x32x16(s8, w.mins, zero16());
                }
                if constexpr (kSums && f == 4) acc[mt] = __builtin_elementwise_fma((float16_t)w.d[1], P2, acc[mt]);
                if constexpr (mt > 0 && f == 2)
                    acc[mt - 1] = __builtin_elementwise_fma((float16_t)w.d[0], P[(mt - 1) & 1], acc[mt - 1]);
                if constexpr (mt > 0 && f == 2) pin(acc[mt - 1]);
                else pin(acc[mt]);
            }
        });
        if constexpr (kBlocks)
            acc[MT - 1] = __builtin_elementwise_fma((float16_t)w.d[7], P[(NI - 1) & 1], acc[MT - 1]);
        else if constexpr (!kF16)
            acc[MT - 1] = __builtin_elementwise_fma((float16_t)w.d[0], P[(MT - 1) & 1], acc[MT - 1]);
        if constexpr (kF16) {
            if (st + 1 < hi) tile_load_f16(a, wr, wbase, st + 1, 1, w.f);
        } else {
            if (!late && st + 1 < hi) tile_dequant<TYPE>(raw, nk, w);
        }
    }

    // accumulator i of tile mt: row 32 mt + 8 (i / 4) + 4 kg + i % 4
    constexpr int MO = HL ? MT / 2 : MT;
    if constexpr (HL) unrolled<MO>([&](auto mt) { acc[mt] = acc[mt] + acc[MO + mt] * kLoUnscale; });
    if (sliced) {
        // (Parts as [slice][M][N] instead: rows a power of two apart when N is; 4096 x
        // 4096 Q4_K at 128 rows 23.6 -> 28.2 us, level elsewhere.)
        float* out = ta.part + ((size_t)u * a.ks_count + ks) * RB * kTileCols + 32 * wave + (lane & 31);
        unrolled<MO>([&](auto mt) {
            unrolled<16>([&](auto i) {
                const int r = 32 * mt + 8 * (i >> 2) + 4 * kg + (i & 3);
                if (m0 + r < a.M) out[r * kTileCols] = acc[mt][(int)i];
            });
        });
        return;
    }
    if constexpr (!HL) {  // fp16 X has no epilogue
        unrolled<MO>([&](auto mt) {
            unrolled<16>([&](auto i) {
                const int m = m0 + 32 * mt + 8 * (i >> 2) + 4 * kg + (i & 3);
                if (m < a.M && n < a.N) a.out[(size_t)m * a.N + n] = acc[mt][(int)i];
            });
        });
    }
    if constexpr (HL) {
        float* rs = (float*)lds;
        if (a.f.rs_pss) {
            lds_barrier();  // every wave is past its reads of X
            for (int r = wave; r < RB; r += kTileWaves)
                if (m0 + r < a.M) {
                    const float v = rs_reduce(a, rs_load(a, m0 + r));
                    if (lane == 0) rs[r] = v;
                }
            lds_barrier();
        }
        const EpiPos pos0 = epi_pos0(a);
        unrolled<4 * MO>([&](auto q) {
            constexpr int mt = decltype(q)::value >> 2, i4 = decltype(q)::value & 3;
            const int r0 = 32 * mt + 8 * i4 + 4 * kg;
            float2 pre[4];
            unrolled<4>([&](auto i) { pre[i] = epi_load(a, m0 + r0 + i, n, pos0); });
            unrolled<4>([&](auto i) {
                float s = acc[mt][4 * i4 + i];
                if (a.f.rs_pss) s *= rs[r0 + i];
                epilogue(a, s, m0 + r0 + i, n, n >> 4, lane, pre[i], pos0);
            });
        });
    }
}

// The sliced blocks: their slices summed in K order, then the row scale and
// epilogue.  Grid (n_part, rows of a block / RPT), a thread per column; SU >=
// ks_count reads a row are issued before the first add.
template <int SU, int RPT>
__global__ __launch_bounds__(kTileCols) void tile_fixup_kernel(TileArgs ta, int rb)
{
    static_assert(RPT <= kTileCols / 64, "one wave per row scale");
    __shared__ float rs[RPT];
    const GemmArgs& a = ta.a;
    // the parts are read whatever M and N are (they hold whole blocks), ahead of the block's place
    const int r0 = (int)blockIdx.y * RPT;
    const size_t slice = (size_t)rb * kTileCols;
    const float* p = ta.part + (size_t)blockIdx.x * a.ks_count * slice + (size_t)r0 * kTileCols + threadIdx.x;
    float v[RPT][SU];
#pragma unroll
    for (int j = 0; j < RPT; ++j)
#pragma unroll
        for (int k = 0; k < SU; ++k) v[j][k] = k < a.ks_count ? p[k * slice + j * kTileCols] : 0.0f;
    int mb, nb;
    block_at(ta, ta.n_full + (int)blockIdx.x, mb, nb);
    const int m0 = mb * rb + r0;
    if (m0 >= a.M) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = nb * kTileCols + (int)threadIdx.x;
    const EpiPos pos0 = epi_pos0(a);
    float2 pre[RPT];
#pragma unroll
    for (int j = 0; j < RPT; ++j) pre[j] = epi_load(a, m0 + j, n, pos0);
    if (a.f.rs_pss) {
        if (wave < RPT && m0 + wave < a.M) {  // wave-uniform
            const float r = rs_reduce(a, rs_load(a, m0 + wave));
            if (lane == 0) rs[wave] = r;
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        float s = v[j][0];
#pragma unroll
        for (int k = 1; k < SU; ++k) s = k < a.ks_count ? s + v[j][k] : s;
        if (a.f.rs_pss) s *= rs[j];
        if (m0 + j < a.M) epilogue(a, s, m0 + j, n, n >> 4, lane, pre[j], pos0);
    }
}

// Sub-block sums of fp16 X [R][K] (K a multiple of 256) for the Q4_K mins:
// out[super-block][row][2 units]: unit kg holds sub-blocks 2 kg, 2 kg + 1, 2
// kg + 4, 2 kg + 5 as (hi, lo) fp16 pairs of s / 32 (lo scaled by 2^11), s the
// fp32 sum.  A quad of lanes takes one sub-block.
__global__ __launch_bounds__(256) void tile_sums_kernel(const uint4* __restrict__ x, uint32_t R, uint32_t K,
                                                        half2_t* __restrict__ out)
{
    const uint32_t u = blockIdx.x * 256 + threadIdx.x, row = blockIdx.y;  // 16-byte unit of the row
    const bool ok = u < K / 8;
    const uint4 v4 = ok ? x[(size_t)row * (K / 8) + u] : uint4{0, 0, 0, 0};
    const half2_t one2 = {(_Float16)1.0f, (_Float16)1.0f};
    float v = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, v4.x), one2, 0.0f, false);
    v = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, v4.y), one2, v, false);
    v = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, v4.z), one2, v, false);
    v = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, v4.w), one2, v, false);
    v += xor_lane<1>(v);
    v += xor_lane<2>(v);
    if (ok && (u & 3) == 0) {
        v *= 0.03125f;
        const _Float16 hi = (_Float16)v;
        const _Float16 lo = (_Float16)((v - (float)hi) * 2048.0f);
        const uint32_t sub = (u >> 2) & 7, kg = (sub >> 1) & 1, slot = (sub & 1) + 2 * (sub >> 2);
        out[((size_t)(u >> 5) * R + row) * 8 + 4 * kg + slot] = half2_t{hi, lo};
    }
}

template <int TYPE, int MT, bool HL>
void tile_launch(const TileArgs& ta, hipStream_t st)
{
    const int grid = ta.n_full + ta.n_part * ta.a.ks_count;
    hipLaunchKernelGGL((gemm_tile_kernel<TYPE, MT, HL>), dim3(grid), dim3(kTileWaves * 64), tile_lds_bytes(32 * MT), st,
                       ta);
}

template <int TYPE>
void tile_launch_t(const TileArgs& ta, int mt, hipStream_t st)
{
    if (ta.a.hl) {
        tile_launch<TYPE, 4, true>(ta, st);
        return;
    }
    if (mt <= 1) tile_launch<TYPE, 1, false>(ta, st);
    else if (mt <= 2) tile_launch<TYPE, 2, false>(ta, st);
    else tile_launch<TYPE, 4, false>(ta, st);
}

template <int TYPE>
ulspec_status tile_attrs(ulspec_ctx* ctx)
{
    const struct {
        const void* fn;
        int rows;
    } fns[] = {{(const void*)gemm_tile_kernel<TYPE, 1, false>, 32},
               {(const void*)gemm_tile_kernel<TYPE, 2, false>, 64},
               {(const void*)gemm_tile_kernel<TYPE, 4, false>, 128},
               {(const void*)gemm_tile_kernel<TYPE, 4, true>, 128}};
    for (const auto& f : fns) {
        const hipError_t e =
            hipFuncSetAttribute(f.fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)tile_lds_bytes(f.rows));
        if (e != hipSuccess) return hip_fail(ctx, e, "hipFuncSetAttribute(tile GEMM LDS)");
    }
    return ULSPEC_OK;
}

}  // namespace

namespace ulspec {

ulspec_status gemm_tile_init(ulspec_ctx* ctx)
{
    ulspec_status s = tile_attrs<ULSPEC_GGML_Q4_0>(ctx);
    if (s == ULSPEC_OK) s = tile_attrs<ULSPEC_GGML_Q4_K>(ctx);
    if (s == ULSPEC_OK) s = tile_attrs<ULSPEC_GGML_Q6_K>(ctx);
    if (s == ULSPEC_OK) s = tile_attrs<ULSPEC_GGML_Q8_0>(ctx);
    if (s == ULSPEC_OK) s = tile_attrs<ULSPEC_GGML_F16>(ctx);
    return s;
}

namespace {

// 32-row operand tiles of a workgroup for M rows of fp16 X.
int tile_mt(uint32_t M) { return M <= 32 ? 1 : M <= 64 ? 2 : 4; }

// Slices of the rem blocks that do not fill a round of the CUs (a workgroup holds
// a CU's LDS): those that minimise the rounds' length in stages of about 4 us, a
// workgroup's start about one, plus the fix-up (its launch about three, and each
// part's way through memory: rb rows of 1 KB twice, at about 20 MB a stage).  1:
// no slices.  Slicing the last round only, against every block in n_cu / blocks
// slices or none: split X of 1500 rows through the 7B layer (1152, 384, 2064 and
// 384 blocks) 7.6 -> 7.1 ms per 4 layers, 12288 x 4096 Q4_K at 1500 rows 195 -> 177
// us, 4096 x 4096 Q4_K at 128 27.3 -> 23.6, 6000 x 1024 F16 at 300 23.9 -> 16.9.
// (The last round's stages dealt out evenly, as a loop over parts of two blocks:
// 2048 x 11008 x 4096 Q4_K 202 -> 236 us, its parts being 56 MB.)
constexpr float kTileStart = 1.0f, kTileFixup = 3.0f;
constexpr int kTileMaxSlices = 32;
int tile_slices(int rem, int stages, int rb, int n_cu)
{
    int best = 1;
    float best_cost = (float)stages + kTileStart;
    for (int ks = 2; ks <= std::min(stages / 2, kTileMaxSlices) && rem * ks <= 4 * n_cu; ++ks) {
        const int rounds = (rem * ks + n_cu - 1) / n_cu;
        const float cost = (float)rounds * ((float)((stages + ks - 1) / ks) + kTileStart) + kTileFixup +
                           (float)rem * (float)ks * (float)rb * 1e-4f;
        if (cost < best_cost) {
            best = ks;
            best_cost = cost;
        }
    }
    return best;
}

template <int SU>
void fixup_launch(const TileArgs& ta, int rb, int n_cu, hipStream_t st)
{
    const int rows = std::min(rb, ta.a.M), four = (rows + 3) / 4;
    if (ta.n_part * four >= 2 * n_cu)
        hipLaunchKernelGGL((tile_fixup_kernel<SU, 4>), dim3(ta.n_part, four), dim3(kTileCols), 0, st, ta, rb);
    else
        hipLaunchKernelGGL((tile_fixup_kernel<SU, 1>), dim3(ta.n_part, rows), dim3(kTileCols), 0, st, ta, rb);
}

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

size_t tile_sum_bytes(const Weight& w, uint32_t rows)
{
    return w.type == ULSPEC_GGML_Q4_K ? align256((size_t)rows * (w.k / 8)) : 0;
}

}  // namespace

// Whether fp16 X of M rows runs here rather than on the whole-X / split-K
// kernels.  Past 64 rows those take further launches over the whole weight
// (4096 x 11008 Q4_K at M = 128: 43.2 -> 31.4 us; a narrow weight at two launches
// is still ahead there: 512 x 2048 Q4_0 at 65 11.9 against 14.7 us, at 200 29.7
// -> 15.4).  From 17 to 64 rows both read it once; this kernel's blocks are 256 columns wide, so it wins where there are
// enough of them (22016 x 4096 Q4_K at M = 17 / 48 / 64: 23.3 / 35.8 / 42.3 ->
// 21.2 / 28.3 / 30.0 us; 32000 x 4096 Q6_K at 64: 50.0 -> 44.9; 11008 x 4096
// Q4_0 at 48: 25.7 -> 22.0) and loses on narrower ones (4096 x 4096 Q4_K at 48:
// 11.5 against 14.9 us).  Up to 16 rows the others are ahead (22016 x 4096 Q4_K
// at 16: 20.4 against 21.0 us).
bool gemm_tile_wins(const Weight& w, uint32_t M)
{
    return M > 128 || (M > 64 && w.n > 2048) || (M > 16 && w.n > 8192);
}

// Workspace of the tile GEMM: parts for one round of slices (gemm_tile takes
// fewer where more would not fit), the sums those of kTileRowsH16 rows.
size_t gemm_tile_workspace_bytes(const Weight& w, int n_cu)
{
    return tile_sum_bytes(w, kTileRowsH16) + (size_t)std::max(1, n_cu) * 128 * kTileCols * sizeof(float);
}

size_t gemm_tile_split_bytes(uint32_t M, uint32_t K, int n_cu)
{
    return align256((size_t)2 * M * (K / 8)) + (size_t)std::max(1, n_cu) * 64 * kTileCols * sizeof(float);
}

ulspec_status gemm_tile(ulspec_ctx* ctx, const Weight& w, const GemmFuse& f, const uint16_t* x, uint32_t M, bool hl,
                        uint32_t lo_rows, float* y, void* ws, size_t ws_bytes)
{
    TileArgs ta;
    GemmArgs& a = ta.a;
    a.w = w.dev;
    a.w_bytes = (uint32_t)w.bytes;
    a.x = reinterpret_cast<const _Float16*>(x);
    a.M = (int)M;
    a.N = (int)w.n;
    a.K = (int)w.k;
    a.n_tiles = (int)w.n_tiles;
    a.n_chunks = (int)w.n_chunks;
    a.ks_q = a.ks_r = 0;
    a.hl = hl ? 1 : 0;
    a.lo_rows = hl ? (int)lo_rows : 0;
    a.xrows = hl ? 2 * (int)M : (int)M;
    a.f = f;
    const uint32_t xrows = hl ? lo_rows + M : M;
    if ((uint64_t)xrows * w.k * 2 >= kOOB || (uint64_t)M * w.n * 4 >= kOOB)
        return fail(ctx, ULSPEC_EINVAL, "tile gemm: %u rows past the 2 GiB operand limit", M);
    const int mt = hl ? 4 : tile_mt(M), rb = hl ? 64 : 32 * mt;
    ta.tm = ((int)M + rb - 1) / rb;
    ta.tn = ((int)w.n + kTileCols - 1) / kTileCols;
    ta.n_stages = (int)((w.k + 255) / 256);
    const size_t sums = tile_sum_bytes(w, xrows);
    if (sums > ws_bytes) return fail(ctx, ULSPEC_EINVAL, "tile gemm: %zu bytes of row sums, %zu available", sums, ws_bytes);
    const int n_cu = std::max(1, ctx->n_cu), blocks = ta.tm * ta.tn, rem = blocks % n_cu;
    int ks = rem ? tile_slices(rem, ta.n_stages, rb, n_cu) : 1;
    while (ks > 1 && sums + (size_t)rem * ks * rb * kTileCols * sizeof(float) > ws_bytes) --ks;
    ta.n_part = ks > 1 ? rem : 0;
    ta.n_full = blocks - ta.n_part;
    a.ks_count = ks;
    ta.st_q = ta.n_stages / ks;
    ta.st_r = ta.n_stages % ks;
    ta.xsum = (const uint4*)ws;
    ta.xsum_rows = (int)xrows;
    ta.part = (float*)((char*)ws + sums);
    a.out = y;
    if (w.type == ULSPEC_GGML_Q4_K)
        hipLaunchKernelGGL(tile_sums_kernel, dim3((w.k / 8 + 255) / 256, xrows), dim3(256), 0, ctx->stream,
                           (const uint4*)x, xrows, w.k, (half2_t*)ws);
    if (w.type == ULSPEC_GGML_Q4_0) tile_launch_t<ULSPEC_GGML_Q4_0>(ta, mt, ctx->stream);
    else if (w.type == ULSPEC_GGML_Q4_K) tile_launch_t<ULSPEC_GGML_Q4_K>(ta, mt, ctx->stream);
    else if (w.type == ULSPEC_GGML_Q6_K) tile_launch_t<ULSPEC_GGML_Q6_K>(ta, mt, ctx->stream);
    else if (w.type == ULSPEC_GGML_Q8_0) tile_launch_t<ULSPEC_GGML_Q8_0>(ta, mt, ctx->stream);
    else tile_launch_t<ULSPEC_GGML_F16>(ta, mt, ctx->stream);
    if (ks > 1) {
        if (ks <= 2) fixup_launch<2>(ta, rb, n_cu, ctx->stream);
        else if (ks <= 4) fixup_launch<4>(ta, rb, n_cu, ctx->stream);
        else if (ks <= 8) fixup_launch<8>(ta, rb, n_cu, ctx->stream);
        else if (ks <= 16) fixup_launch<16>(ta, rb, n_cu, ctx->stream);
        else fixup_launch<kTileMaxSlices>(ta, rb, n_cu, ctx->stream);
    }
    return ULSPEC_OK;
}

}  // namespace ulspec
