// gemm_dev.h -- device helpers shared by the dequant-GEMM kernels (q4_gemm.hip,
// gemm_tile.hip): the re-tiled weight chunks (layout at the top of
// q4_gemm.hip) and their dequantization, buffer loads, the X operand, the row
// scale and the fused epilogues.
#pragma once

#include "detmath.h"
#include "hip_common.h"
#include "ulspec_internal.h"

namespace ulspec {

// Arguments of the dequant-GEMM kernels (see the X operand below).
struct GemmArgs {
    const uint8_t* w;
    uint32_t w_bytes;
    const _Float16* x;
    float* out;  // Y, or the slice partials [ks_count][M][N] of the split-K kernel
    int M, N, K, n_tiles, n_chunks, ks_count;
    int ks_q, ks_r;  // n_chunks = ks_q * ks_count + ks_r; slice s starts at s * ks_q + min(s, ks_r)
    int hl;          // split X (see above)
    int lo_rows;     // split X: row of X holding the low part of row 0
    int xrows;       // rows of X staged: M, or 2M when split
    GemmFuse f;      // row scale and epilogue
};

namespace {

constexpr int kQ40Chunk = 1152;
// Q8_0: one 16-row tile x 4 blocks (128 K): lane l holds the 8 int8 values
// k = 32 j + 8 (l >> 4) .. +7 of row l & 15 for blocks j = 0, 1 at l * 16 and
// j = 2, 3 at 1024 + l * 16 (two 1 KB coalesced loads per wave), then the
// 16 rows' 4 fp16 block scales at 2048 + row * 8.  1.0625 B per weight, as
// in GGUF.
constexpr int kQ80Chunk = 2176;
constexpr int kQ4KChunk = 2304;
constexpr int kQ6KChunk = 3360;
// fp16 weights (GGUF F16, and Q6_K or mixed-type fused weights converted at
// upload): a chunk is
// one 16-row tile x 128 K, 4 KB; lane l reads 16 contiguous bytes at
// 1024 j + 16 l for MFMA j (rows l & 15, K 32 j + 8 (l >> 4) ..).
constexpr int kF16Chunk = 4096;
// Types whose chunk is one 256-element super-block (lane group g takes
// elements 64 g .. 64 g + 63 of it); the others take 128 K per chunk.
template <int TYPE>
constexpr bool kSuperBlock = TYPE == ULSPEC_GGML_Q4_K || TYPE == ULSPEC_GGML_Q6_K;
// 16-byte X units (8 halves) per weight chunk: 128 K for Q4_0, Q8_0 and F16,
// 256 for Q4_K and Q6_K
template <int TYPE>
constexpr int kUnitsPerChunk = kSuperBlock<TYPE> ? 32 : 16;

// Compiler-only barrier: loads issued before it stay before it (they are not
// sunk to their first use), so all of a batch's loads are in flight together.
// The hardware still overlaps them; s_waitcnt is placed at each first use.
__device__ __forceinline__ void pin_loads() { asm volatile("" ::: "memory"); }

#define ULSPEC_VM_CASE(n) \
    case n: vm_wait<n>(); break;
#define ULSPEC_VM_CASE8(n) \
    ULSPEC_VM_CASE(n) ULSPEC_VM_CASE(n + 1) ULSPEC_VM_CASE(n + 2) ULSPEC_VM_CASE(n + 3) \
    ULSPEC_VM_CASE(n + 4) ULSPEC_VM_CASE(n + 5) ULSPEC_VM_CASE(n + 6) ULSPEC_VM_CASE(n + 7)

// vm_wait with a wave-uniform count n known only at run time (a jump table);
// counts outside 0..63 wait for everything.
__device__ __forceinline__ void vm_wait_dyn(int n)
{
    switch (n) {
        ULSPEC_VM_CASE8(0) ULSPEC_VM_CASE8(8) ULSPEC_VM_CASE8(16) ULSPEC_VM_CASE8(24)
        ULSPEC_VM_CASE8(32) ULSPEC_VM_CASE8(40) ULSPEC_VM_CASE8(48) ULSPEC_VM_CASE8(56)
    default: vm_wait<0>();
    }
}
#undef ULSPEC_VM_CASE8
#undef ULSPEC_VM_CASE

// Raw buffer loads: 32-bit offsets from a base held in scalar registers, and
// the hardware returns 0 for offsets at or past num_records instead of
// faulting (such a load still occupies the texture unit like any other).  0x00020000 is the gfx9-family dword-3 of the resource.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ uint4 buf_load16(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// Weight loads are non-temporal: a weight is read once per call, and the
// step streams gigabytes of other weights and K / V before it comes back, so
// allocating it in the last-level cache only evicts the activations the next
// kernel reads.  (A plain streaming read of 2 GB: 5.47 TB/s plain, 5.78 TB/s
// non-temporal, and a 160 MB buffer read before it stays cache-resident; the
// 7B target's verify GEMMs as the step runs them 13.15 -> 12.90 us per call.)
constexpr int kWeightCache = 2;  // the nt bit of the buffer instructions' cache policy

__device__ __forceinline__ uint4 wt_load16(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kWeightCache));
}

__device__ __forceinline__ uint2 wt_load8(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kWeightCache));
}

__device__ __forceinline__ half8_t buf_load_h8(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    return __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// (v & mask) | magic as one v_and_or_b32 (gfx9 VOP3 takes no two literals,
// so the compiler would otherwise split it).
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t magic)
{
    uint32_t o;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(o) : "v"(v), "v"(mask), "v"(magic));
    return o;
}

// Masks and the fp16 exponent magic, kept in VGPRs.
struct NibbleConsts {
    uint32_t lo, hi, magic;
};

__device__ __forceinline__ NibbleConsts nibble_consts()
{
    NibbleConsts k;
    k.lo = 0x000F000Fu;
    k.hi = 0x00F000F0u;
    k.magic = 0x64006400u;
    // keep them in registers across the loop
    asm volatile("" : "+v"(k.lo), "+v"(k.hi), "+v"(k.magic));
    return k;
}

// 8 nibbles in the tiled order -> fp16 (1024+q, 1024+16q, 1024+q, 1024+16q) pairs
struct MagicPairs {
    half2_t a, b, c, d;  // (e0,e1) q, (e2,e3) 16q, (e4,e5) q, (e6,e7) 16q
};

__device__ __forceinline__ MagicPairs magic_pairs(uint32_t v, const NibbleConsts& k)
{
    const uint32_t v8 = v >> 8;
    MagicPairs m;
    m.a = as_half2(and_or(v, k.lo, k.magic));
    m.b = as_half2(and_or(v, k.hi, k.magic));
    m.c = as_half2(and_or(v8, k.lo, k.magic));
    m.d = as_half2(and_or(v8, k.hi, k.magic));
    return m;
}

// Q4_0: (q - 8) exactly, elements e0..e7.
__device__ __forceinline__ half8_t dequant_q4_0(uint32_t v, const NibbleConsts& k)
{
    MagicPairs m = magic_pairs(v, k);
    const half2_t c1032 = splat2(-1032.0f), s16 = splat2(0.0625f), c72 = splat2(-72.0f);
    half2_t a = m.a + c1032;
    half2_t b = __builtin_elementwise_fma(m.b, s16, c72);
    half2_t c = m.c + c1032;
    half2_t d = __builtin_elementwise_fma(m.d, s16, c72);
    return make_half8(a, b, c, d);
}

// Q4_K: q * sc exactly (q <= 15, sc <= 63 -> <= 945).
struct SubScale {
    half2_t sc, nsc1024, sc16, nsc64;
};

__device__ __forceinline__ half8_t dequant_q4_k(uint32_t v, const SubScale& s, const NibbleConsts& k)
{
    MagicPairs m = magic_pairs(v, k);
    half2_t a = __builtin_elementwise_fma(m.a, s.sc, s.nsc1024);
    half2_t b = __builtin_elementwise_fma(m.b, s.sc16, s.nsc64);
    half2_t c = __builtin_elementwise_fma(m.c, s.sc, s.nsc1024);
    half2_t d = __builtin_elementwise_fma(m.d, s.sc16, s.nsc64);
    return make_half8(a, b, c, d);
}


// ---- X operand and common pieces -------------------------------------------
// X is fp16 rows [M][K] (hl = 0), or split fp32 activations (hl = 1): the
// high parts (split_hl) of rows 0..M-1, and the low part of row m at row
// lo_rows + m.  In split mode an MFMA covers 8 output rows: A-operand slots
// 0-7 take the high parts of 8 rows, slots 8-15 the low parts of the same
// rows, and the two halves of the result are added in the epilogue (hi + lo *
// 2^-11), so M <= 8 per 16-column tile.
constexpr uint32_t kOOB = 0x80000000u;  // >= any buffer's num_records

// X row behind staged row rho (0 .. xrows-1).
__device__ __forceinline__ int x_row(const GemmArgs& a, int rho)
{
    return a.hl && rho >= a.M ? a.lo_rows + rho - a.M : rho;
}

// Bytes of X the kernels may read.
__device__ __forceinline__ uint32_t x_bytes(const GemmArgs& a)
{
    return (uint32_t)(a.hl ? a.lo_rows + a.M : a.M) * (uint32_t)a.K * 2u;
}

// Staged row that A-operand slot r (0..15) of column tile mt reads; slots past
// the last row repeat it (their outputs are never stored).
__device__ __forceinline__ int xslot_row(const GemmArgs& a, int mt, int r)
{
    if (!a.hl) return min(16 * mt + r, a.M - 1);
    const int m = min(8 * mt + (r & 7), a.M - 1);
    return r < 8 ? m : a.M + m;
}

// Output row of accumulator element i of lane `lane` in column tile mt, or
// -1 where the element is a low-part slot of split X.
__device__ __forceinline__ int acc_row(const GemmArgs& a, int mt, int lane, int i)
{
    if (!a.hl) return 16 * mt + 4 * (lane >> 4) + i;
    return lane < 32 ? 8 * mt + 4 * (lane >> 4) + i : -1;
}

__device__ __forceinline__ void slice_range(const GemmArgs& a, int ks, int& lo, int& hi)
{
    lo = ks * a.ks_q + min(ks, a.ks_r);
    hi = lo + a.ks_q + (ks < a.ks_r ? 1 : 0);
}

// Eight int8 values (two words) -> fp16, exactly: each biased byte b ^ 0x80
// under exponent 0x64 is 1024 + (b + 128); subtracting 1152 leaves b.
__device__ __forceinline__ half8_t dequant_q8_0(uint32_t lo, uint32_t hi)
{
    const uint32_t x0 = lo ^ 0x80808080u, x1 = hi ^ 0x80808080u;
    const uint4 u = {(x0 & 0xffu) | ((x0 & 0xff00u) << 8) | 0x64006400u,
                     ((x0 >> 16) & 0xffu) | ((x0 >> 8) & 0xff0000u) | 0x64006400u,
                     (x1 & 0xffu) | ((x1 & 0xff00u) << 8) | 0x64006400u,
                     ((x1 >> 16) & 0xffu) | ((x1 >> 8) & 0xff0000u) | 0x64006400u};
    return __builtin_bit_cast(half8_t, u) - (half8_t)(_Float16)1152.0f;
}

// Q6_K: 8 values -> fp16 (q - 32) * sc, q = low nibble | high pair << 4.  The
// magic 0x6400 pairs are 1024 + q (pairs a, c) or 1024 + 16 q (b, d), the
// high pairs ORed in under the magic first; subtracting 1056 / 1536 leaves
// q - 32 / 16 (q - 32) exactly, and one multiply by sc / sc/16 rounds only
// where |(q - 32) sc| > 2048 (2^-12 relative, as an fp16 copy of the
// weight).  hx: the step's high-bit word (shifted right by 2 for odd steps).
struct Q6Consts {
    uint32_t m30, m300;  // 0x00300030, 0x03000300
};

__device__ __forceinline__ Q6Consts q6_consts()
{
    Q6Consts k;
    k.m30 = 0x00300030u;
    k.m300 = 0x03000300u;
    asm volatile("" : "+v"(k.m30), "+v"(k.m300));
    return k;
}

struct Q6Scale {
    half2_t s1, s16;  // sc, sc / 16
};

__device__ __forceinline__ Q6Scale q6_scale(int sc)
{
    const float f = (float)sc;
    return Q6Scale{splat2(f), splat2(f * 0.0625f)};
}

__device__ __forceinline__ half8_t dequant_q6_k(uint32_t v, uint32_t hx, const Q6Scale& s, const NibbleConsts& k,
                                                const Q6Consts& k6)
{
    const uint32_t v8 = v >> 8;
    const uint32_t ta = and_or(hx, k6.m30, k.magic), tb = and_or(hx, k6.m300, k.magic);
    const uint32_t tc = and_or(hx >> 8, k6.m30, k.magic), td = and_or(hx << 8, k6.m300, k.magic);
    const half2_t c1056 = splat2(-1056.0f), c1536 = splat2(-1536.0f);
    const half2_t a = as_half2(and_or(v, k.lo, ta)) + c1056, b = as_half2(and_or(v, k.hi, tb)) + c1536;
    const half2_t c = as_half2(and_or(v8, k.lo, tc)) + c1056, d = as_half2(and_or(v8, k.hi, td)) + c1536;
    return make_half8(a * s.s1, b * s.s16, c * s.s1, d * s.s16);
}

// ---- row scale and epilogue --------------------------------------------------
// Row scale r_m = 1 / sqrt(sum_p pss[m][p] / K + eps) (RMSNorm,
// src/shaders/ffn/ffn_fused.glsl:23-33).  The GEMMs that follow a norm take X
// = split(h * w) from the producer of h and apply r_m to each output, which
// is x * W^T for x = (h * r) * w.  Lane l holds partials 4 l .. 4 l + 3 of the
// row (P <= 256); rs_reduce sums them ((a + b) + (c + d), then an xor tree).
constexpr int kMaxPartials = 256;

__device__ __forceinline__ float4 rs_load(const GemmArgs& a, int m)
{
    const GemmFuse& f = a.f;
    const __amdgpu_buffer_rsrc_t pr = make_rsrc(f.rs_pss, (uint32_t)a.M * (uint32_t)f.rs_P * 4u);
    const int p0 = 4 * (threadIdx.x & 63);
    return __builtin_bit_cast(float4, buf_load16(pr, m < a.M && p0 < f.rs_P ? (uint32_t)(m * f.rs_P + p0) * 4u : kOOB));
}

__device__ __forceinline__ float rs_reduce(const GemmArgs& a, float4 v)
{
    const int p0 = 4 * (threadIdx.x & 63), P = a.f.rs_P;
    float ss = ((p0 < P ? v.x : 0.0f) + (p0 + 1 < P ? v.y : 0.0f)) + ((p0 + 2 < P ? v.z : 0.0f) + (p0 + 3 < P ? v.w : 0.0f));
    ss += xor_lane<32>(ss);
    ss += xor_lane<16>(ss);
    ss += xor_lane<8>(ss);
    ss += xor_lane<4>(ss);
    ss += xor_lane<2>(ss);
    ss += xor_lane<1>(ss);
    return 1.0f / __builtin_sqrtf(ss / (float)a.K + a.f.rs_eps);
}

// First position of each sequence's rows for the RoPE epilogue: scalar
// loads through the constant address space (the values are fixed for the
// whole kernel), so they never wait behind the vector loads in flight.
// (Named fields, not an array: the positions stay in registers.)
static_assert(kMaxSeqs == 8, "EpiPos holds 8 sequences");
struct EpiPos {
    int p0, p1, p2, p3, p4, p5, p6, p7;
};

__device__ __forceinline__ EpiPos epi_pos0(const GemmArgs& a)
{
    EpiPos r{0, 0, 0, 0, 0, 0, 0, 0};
    if (a.f.epi != kEpiRope) return r;
    const __attribute__((address_space(4))) int32_t* p = (const __attribute__((address_space(4))) int32_t*)a.f.pos_dev;
    const int n = a.f.nseq, add = a.f.pos_add;
    r.p0 = p[0] + add;
    if (n > 1) {
        r.p1 = p[1] + add;
        r.p2 = n > 2 ? p[2] + add : 0;
        r.p3 = n > 3 ? p[3] + add : 0;
        r.p4 = n > 4 ? p[4] + add : 0;
        r.p5 = n > 5 ? p[5] + add : 0;
        r.p6 = n > 6 ? p[6] + add : 0;
        r.p7 = n > 7 ? p[7] + add : 0;
    }
    return r;
}

// Sequence of row m (rows are grouped by sequence, seq_rows each) and the
// row's index j within it.
__device__ __forceinline__ int row_seq(const GemmFuse& f, int m, int& j)
{
    const int b = f.nseq > 1 ? m / f.seq_rows : 0;
    j = m - b * f.seq_rows;
    return b;
}

__device__ __forceinline__ int seq_pos0(EpiPos ps, int b)
{
    int v = ps.p0;
    v = b == 1 ? ps.p1 : v;
    v = b == 2 ? ps.p2 : v;
    v = b == 3 ? ps.p3 : v;
    v = b == 4 ? ps.p4 : v;
    v = b == 5 ? ps.p5 : v;
    v = b == 6 ? ps.p6 : v;
    v = b == 7 ? ps.p7 : v;
    return v;
}

// RoPE position of row m: its sequence's first position plus j, or plus the
// row's tree depth.
__device__ __forceinline__ int rope_pos(const GemmFuse& f, EpiPos ps, int m)
{
    int j;
    const int b = row_seq(f, m, j);
    return seq_pos0(ps, b) + (f.tree ? (int)((f.row_depth >> (4 * (j & 15))) & 15u) : j);
}

// K / V cache row of row m: slot first position + j of its sequence's cache.
__device__ __forceinline__ size_t kv_row(const GemmFuse& f, EpiPos ps, int m)
{
    int j;
    const int b = row_seq(f, m, j);
    return (size_t)(f.seq0 + b) * f.seq_slots + (size_t)(seq_pos0(ps, b) + j);
}

// The memory operands of the epilogue of output (m, n), loaded ahead of it
// with the weights so that the epilogue reads no memory (vmcnt retires in
// issue order: a load issued in the epilogue would wait for every weight load
// in flight).  Two 4-byte loads for the resid and rope epilogues (out of range
// where a thread has no output), none otherwise:
//   resid: (h[m][n], xn_w[n])   rope: (cos, sin) of the pair at the row's
//                               RoPE position (rope_pos)
// Split in two: epi_addr (the buffer descriptors and the offsets, most of the
// address arithmetic) and epi_issue (the loads), so that a wave without an
// output slot skips the arithmetic while every wave still issues the same
// number of loads (the vmcnt waits count them).
struct EpiAddr {
    __amdgpu_buffer_rsrc_t r0, r1;
    uint32_t o0, o1;
};

// Descriptors of the epilogue's operands, offsets out of range (no output).
__device__ __forceinline__ EpiAddr epi_none(const GemmArgs& a)
{
    const GemmFuse& f = a.f;
    EpiAddr e;
    if (f.epi == kEpiResid) {
        e.r0 = make_rsrc(f.h, (uint32_t)a.M * (uint32_t)a.N * 4u);
        e.r1 = make_rsrc(f.xn_w, f.xn ? (uint32_t)a.N * 4u : 0u);
    } else if (f.epi == kEpiRope) {
        e.r0 = make_rsrc(f.rope, (uint32_t)min((uint64_t)f.rope_rows * (uint64_t)(f.hd / 2) * 8u, (uint64_t)0xffffffffu));
        e.r1 = e.r0;
    } else {
        e.r0 = e.r1 = make_rsrc(a.out, 0u);
    }
    e.o0 = e.o1 = kOOB;
    return e;
}

// The offsets of output (m, n)'s operands into e (out of range where the
// thread has no output).
__device__ __forceinline__ void epi_offsets(const GemmArgs& a, int m, int n, EpiPos pos0, EpiAddr& e)
{
    const GemmFuse& f = a.f;
    const bool ok = m < a.M && n < a.N;
    if (!ok) return;
    if (f.epi == kEpiResid) {
        e.o0 = (uint32_t)(m * a.N + n) * 4u;
        e.o1 = (uint32_t)n * 4u;
    } else if (f.epi == kEpiRope && n < f.qdim + f.kvdim) {
        const int nn = n < f.qdim ? n : n - f.qdim;
        e.o0 = (uint32_t)(rope_pos(f, pos0, m) * (f.hd / 2) + (nn % f.hd) / 2) * 8u;
        e.o1 = e.o0 + 4u;
    }
}

__device__ __forceinline__ float2 epi_issue(const GemmArgs& a, const EpiAddr& e)
{
    float2 v = {0.f, 0.f};
    if (a.f.epi == kEpiResid || a.f.epi == kEpiRope) {
        v.x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(e.r0, e.o0, 0, 0));
        v.y = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(e.r1, e.o1, 0, 0));
    }
    return v;
}

__device__ __forceinline__ float2 epi_load(const GemmArgs& a, int m, int n, EpiPos pos0)
{
    EpiAddr e = epi_none(a);
    epi_offsets(a, m, n, pos0, e);
    return epi_issue(a, e);
}

// epi_load for the threads of tile slot j (wave-uniform): slots past the
// iteration's tiles skip the address arithmetic and issue out-of-range loads.
__device__ __forceinline__ float2 epi_load_slot(const GemmArgs& a, int j, int tpi, int m, int n, EpiPos pos0)
{
    EpiAddr e = epi_none(a);
    if (__builtin_amdgcn_readfirstlane(j) < tpi) epi_offsets(a, m, n, pos0, e);
    return epi_issue(a, e);
}

// Vector loads epi_load issues (wave-uniform).
__device__ __forceinline__ int epi_nloads(const GemmArgs& a)
{
    return a.f.epi == kEpiResid || a.f.epi == kEpiRope ? 2 : 0;
}

// Epilogue of output (m, n) of tile t, value s (already row-scaled); pre from
// epi_load, pos0 from epi_pos0.  Lanes l and l ^ 1 hold columns n and n ^ 1
// of the same row m, and 16-lane groups one row of one tile (whole waves call
// this).
//   store: Y[m][n] = s
//   rope:  RoPE pair (n, n+1) at the row's position (rope_pos: its sequence's
//          first position + j, or + depth(j) for a tree; Q and K rows, angles
//          from epi_load), then fp16 Q -> q16[m][n], K -> kc[row][n - qdim],
//          V -> vc[row][n - qdim - kvdim], row = kv_row(m)
//          (y0 = x0 c - x1 s, y1 = x0 s + x1 c; src/shaders/rope.glsl:50-73)
//   silu:  rows interleaved (2i = gate i, 2i+1 = up i): a = g * (1 / (1 +
//          e^-g)) * u, split: act[m][i] = hi, act[M + m][i] = lo
//   resid: h[m][n] += s (in place); pss[m][t] = sum over the tile's 16 columns
//          of h^2 (xor tree over the 16 lanes), the RMSNorm partial of row m;
//          with xn, the next GEMM's split X: xn[m][n] = hi, xn[xn_lo + m][n] =
//          lo of h * xn_w[n] (the next norm's weights)
__device__ __forceinline__ void epilogue(const GemmArgs& a, float s, int m, int n, int t, int l, float2 pre,
                                         EpiPos pos0)
{
    const bool ok = m < a.M && n < a.N;
    const GemmFuse& f = a.f;
    switch (f.epi) {
    case kEpiRope: {
        const float other = xor_lane<1>(s);
        if (!ok) break;
        const bool odd = n & 1;
        const size_t pos = kv_row(f, pos0, m);
        if (n < f.qdim + f.kvdim) {
            const int nn = n < f.qdim ? n : n - f.qdim;
            const float2 cs = pre;
            const float x0 = odd ? other : s, x1 = odd ? s : other;
            float y;
            if (!odd) {
                const float p0 = x0 * cs.x, p1 = x1 * cs.y;
                y = p0 - p1;
            } else {
                const float p0 = x0 * cs.y, p1 = x1 * cs.x;
                y = p0 + p1;
            }
            if (n < f.qdim) f.q16[(size_t)m * f.qdim + nn] = (_Float16)y;
            else f.kc[(size_t)pos * f.kvdim + nn] = (_Float16)y;
        } else {
            f.vc[(size_t)pos * f.kvdim + (n - f.qdim - f.kvdim)] = (_Float16)s;
        }
        break;
    }
    case kEpiSilu: {
        const float u = xor_lane<1>(s);
        if (ok && !(n & 1)) {
            const float sg = s * (1.0f / (1.0f + det_expf(-s)));
            _Float16 hi, lo;
            split_hl(sg * u, hi, lo);
            f.act[(size_t)m * (a.N / 2) + n / 2] = hi;
            f.act[(size_t)(a.M + m) * (a.N / 2) + n / 2] = lo;
        }
        break;
    }
    case kEpiResid: {
        float v = 0.0f;
        if (ok) {
            v = pre.x + s;
            f.h[(size_t)m * a.N + n] = v;
            if (f.xn) {
                _Float16 hi, lo;
                split_hl(v * pre.y, hi, lo);
                f.xn[(size_t)m * a.N + n] = hi;
                f.xn[(size_t)(f.xn_lo + m) * a.N + n] = lo;
            }
        }
        float sq = v * v;
        sq += xor_lane<1>(sq);
        sq += xor_lane<2>(sq);
        sq += xor_lane<4>(sq);
        sq += xor_lane<8>(sq);
        if (m < a.M && t < a.n_tiles && (l & 15) == 0) f.pss_out[(size_t)m * a.n_tiles + t] = sq;
        break;
    }
    default:
        if (ok) a.out[(size_t)m * a.N + n] = s;
    }
}

}  // namespace
}  // namespace ulspec
