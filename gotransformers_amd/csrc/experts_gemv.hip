// Expert kernels for few tokens per expert (decode): a dequantizing GEMV
// that streams each weight row from HBM once per slice of at most 8 tokens,
// with the multiply-adds on the matrix cores at fp32-level accuracy.
//
// Work split: grid (panels of 64 output rows, token slices of all groups);
// a workgroup's NW waves share one panel and split its K range between them,
// each with RING chunks of weights and tokens in flight.
// Lane l of a wave owns row l of the panel, so with the panel layout of the
// weights every 16-byte load of the wave reads 1 KiB of codes contiguously.
//
// Arithmetic: v_mfma_f32_4x4x4_16b_bf16 holds 16 independent 4x4x4
// products; block b of it multiplies 4 tokens (A) by 4 k-values of rows
// 4b..4b+3 (B, one row per lane), so a wave computes 4 tokens x 64 rows per
// instruction and lane l ends up holding row l's dot products for the 4
// tokens -- no cross-lane reduction.  The instruction can broadcast the A of
// any one block to all of them (CBSZ, ABID), so one register pair holds a
// token quad's values for 16 steps, step b in lanes 4b .. 4b + 3: the tokens
// travel in the weights' register ring, split where they are used, and need
// no LDS, no staging pass and no barrier before the main loop (they were
// staged in LDS and read back four times per scale block and quad: with the
// four-wave workgroups this allows, 2048 -> 1024 FP4 gate/up over 64 tokens
// and 64 + 1 experts went 46.2 -> 41 us, down 26.6 -> 24.3; over 113 tokens
// 59.9 -> 51.5 and 31.2 -> 28.6; 1024 -> 2048 Int8, 16 experts, 32 tokens
// 19.2 -> 18.3 and 13.3 -> 12.2).  What bounds it now is the load path: with
// the arithmetic left out the same loads take 41.5 us, without the tokens'
// loads 37.8.  Weight codes are
// exact in bf16 (Int8 magnitudes <= 127, e2m1 values); the tokens are split
// as x = hi + lo with hi = bf16(x) and lo = bf16(x - hi), which represents
// x to about 2^-17 relative, and both halves go through the MFMA with fp32
// accumulation.  Four chained instructions cover one 16-value scale block;
// the block sum is then scaled once into an fp32 accumulator, the order of
// the reference's DotRow (lowprecision/rows.go:207-257).  float32 weights
// are split the same way (three products: hi*hi, lo*hi, hi*lo) and need no
// block scaling.
//
// Gate/up fuse the SwiGLU epilogue (feedforward/gatedfeedforward.go:49-57):
// hidden = act_g(gate + b_g) * act_u(up + b_u).  Down adds its bias.
#include <algorithm>

#include "common.h"

namespace gtmoe {

namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Per precision: 16-byte units and scale blocks per pipeline chunk.
template <int PREC>
struct Chunk;
template <>
struct Chunk<kInt8> {
    static constexpr int U = 4, CB = 4;  // 64 values
};
template <>
struct Chunk<kFP4> {
    static constexpr int U = 2, CB = 4;  // 64 values
};
template <>
struct Chunk<kFloat32> {
    static constexpr int U = 4, CB = 1;  // 16 values
};

template <int PREC, int MATS>
struct ChunkRegs {
    uint4 c[MATS][Chunk<PREC>::U];
    float s[MATS][Chunk<PREC>::CB];
};
// the lane's four values of its token of every quad
template <int NQ>
struct TokenRegs {
    float4 x[NQ];
};

// One weight matrix's panel as buffer resources: the panel's codes (64 rows
// side by side in 16-byte units) and its scales.  The resources live in
// scalar registers; a lane addresses its row with one 32-bit offset and a
// chunk with a scalar offset, so the loads cost one vector register of
// address in all, and a load past the panel returns zeros.
struct PanelSrc {
    __amdgpu_buffer_rsrc_t codes;
    __amdgpu_buffer_rsrc_t scales;
};

// descriptor word 3 for raw (untyped) buffer access on CDNA
constexpr int kRawBufferWord3 = 0x00020000;

template <int I>
__device__ __forceinline__ uint32_t comp(const uint4 &v)
{
    return I == 0 ? v.x : I == 1 ? v.y : I == 2 ? v.z : v.w;
}

__device__ __forceinline__ uint32_t comp_rt(const uint4 &v, int i)
{
    return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}

__device__ __forceinline__ s16x4 as_s16x4(uint32_t lo, uint32_t hi)
{
    const u32x2 v = {lo, hi};
    return __builtin_bit_cast(s16x4, v);
}

// bf16 bits of two floats that bf16 holds exactly (small integers): their
// upper halves, packed.
__device__ __forceinline__ uint32_t upper_halves(float lo, float hi)
{
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two floats rounded to bf16 (nearest even) and packed, lo in the low half:
// one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t bf16_rne_pair(float lo, float hi)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}

// x = hi + lo for two values: hi = bf16(x) rounded to nearest, lo = bf16 of
// the (exact) remainder.
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t &hi, uint32_t &lo)
{
    hi = bf16_rne_pair(x0, x1);
    const float h0 = __uint_as_float(hi << 16), h1 = __uint_as_float(hi & 0xffff0000u);
    lo = bf16_rne_pair(x0 - h0, x1 - h1);
}

// B operand of step S (k-values 4S..4S+3) of block J of a chunk.
template <int PREC, int J, int S>
__device__ __forceinline__ s16x4 weights_step(const uint4 (&c)[Chunk<PREC>::U])
{
    if constexpr (PREC == kInt8) {
        const uint32_t d = comp<S>(c[J]);
        const float f0 = (float)(int)(int8_t)d, f1 = (float)(int)(int8_t)(d >> 8);
        const float f2 = (float)(int)(int8_t)(d >> 16), f3 = (float)(int)(int8_t)(d >> 24);
        return as_s16x4(upper_halves(f0, f1), upper_halves(f2, f3));
    } else {
        // FP4: block J is half J&1 of unit J/2; step S is bytes 2S, 2S+1 of
        // it, and each byte holds two values, the even one in the low nibble
        const uint32_t d = comp<(J & 1) * 2 + (S >> 1)>(c[J >> 1]);
        const auto a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, 1.0f, (S & 1) * 2);
        const auto b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, 1.0f, (S & 1) * 2 + 1);
        return as_s16x4(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
    }
}
template <int S>
__device__ __forceinline__ void weights_step_f32(const uint4 (&c)[Chunk<kFloat32>::U], s16x4 &hi, s16x4 &lo)
{
    const uint4 v = c[S];
    uint32_t h01, l01, h23, l23;
    split_pair(__uint_as_float(v.x), __uint_as_float(v.y), h01, l01);
    split_pair(__uint_as_float(v.z), __uint_as_float(v.w), h23, l23);
    hi = as_s16x4(h01, h23);
    lo = as_s16x4(l01, l23);
}

// 4 tokens x 64 rows: every block takes its A (4 tokens x 4 k-values) from
// block ABID, lanes 4 ABID .. 4 ABID + 3 (CBSZ = 4).
template <int ABID>
__device__ __forceinline__ f32x4 mfma4(s16x4 a, s16x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(a, b, c, 4, ABID, 0);
}

// x * sigmoid(x) with the hardware exp and reciprocal (about 1 ulp each)
__device__ __forceinline__ float silu(float x) { return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

// Codes (and scales) of chunk ch of the lane's row, for every matrix.  A
// chunk of scaled codes is one 4-block scale group.  vo = lane * 16; ch is
// uniform across the wave.
template <int PREC, int MATS>
__device__ __forceinline__ void load_chunk(ChunkRegs<PREC, MATS> &r, const PanelSrc (&src)[MATS], uint32_t vo, int ch)
{
    constexpr int U = Chunk<PREC>::U;
    static_assert(PREC == kFloat32 || Chunk<PREC>::CB == 4, "a chunk's scales are one 16-byte load");
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            r.c[m][u] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(src[m].codes, vo,
                                                                                        (ch * U + u) * 1024, 0));
        if constexpr (PREC != kFloat32) {
            const float4 v = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(src[m].scales, vo, ch * 1024, 0));
            r.s[m][0] = v.x;
            r.s[m][1] = v.y;
            r.s[m][2] = v.z;
            r.s[m][3] = v.w;
        }
    }
}

template <int PREC, int NQ>
__device__ __forceinline__ void load_tokens(TokenRegs<NQ> &r, __amdgpu_buffer_rsrc_t xin, const uint32_t (&xo)[NQ], int ch)
{
#pragma unroll
    for (int q = 0; q < NQ; ++q)
        r.x[q] = __builtin_bit_cast(
            float4, __builtin_amdgcn_raw_buffer_load_b128(xin, xo[q], ch * (Chunk<PREC>::CB * 64), 0));
}

// Panel `panel` (down: and the next MATS - 1) of group g as buffer resources.
// Where the last workgroup's second panel lies past an odd number of panels,
// it takes the last panel again and its rows are not stored: a resource of no
// bytes would not do, as the range check counts from the scalar offset.
template <int PREC, bool GATEUP, int MATS>
__device__ __forceinline__ void panel_src(const GemvArgs &a, int g, int panel, PanelSrc (&src)[MATS])
{
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
        const int pm = GATEUP ? panel : min(panel + m, (a.rows - 1) / kPanelRows);
        const size_t wpanel = (size_t)pm * kPanelRows * a.row_bytes;
        const size_t spanel = (size_t)pm * kPanelRows * a.nblocks;
        src[m].codes = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(reinterpret_cast<const char *>(GATEUP && m ? a.w1 : a.w0)) + (size_t)g * a.w_group_stride + wpanel,
            0, kPanelRows * a.row_bytes, kRawBufferWord3);
        if constexpr (PREC != kFloat32)
            src[m].scales = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(GATEUP && m ? a.s1 : a.s0) + (size_t)g * a.s_group_stride + spanel, 0,
                kPanelRows * a.nblocks * 4, kRawBufferWord3);
    }
}

// Step S (four k-values) of block J of a chunk: the hi and lo halves of every
// token quad against every matrix.  All hi products come before all lo ones,
// so that an instruction seldom waits for the one before it.
template <int PREC, int MATS, int NQ, int J, int S>
__device__ __forceinline__ void block_step(const ChunkRegs<PREC, MATS> &r, const s16x4 (&xh)[NQ],
                                           const s16x4 (&xl)[NQ], f32x4 (&blk)[MATS][NQ])
{
    constexpr int ABID = 4 * J + S;
    s16x4 wh[MATS], wl[MATS];
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
        if constexpr (PREC == kFloat32) weights_step_f32<S>(r.c[m], wh[m], wl[m]);
        else wh[m] = weights_step<PREC, J, S>(r.c[m]);
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int m = 0; m < MATS; ++m) blk[m][q] = mfma4<ABID>(xh[q], wh[m], blk[m][q]);
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int m = 0; m < MATS; ++m) blk[m][q] = mfma4<ABID>(xl[q], wh[m], blk[m][q]);
    if constexpr (PREC == kFloat32) {
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int m = 0; m < MATS; ++m) blk[m][q] = mfma4<ABID>(xh[q], wl[m], blk[m][q]);
    }
}

template <int PREC, int MATS, int NQ, int J>
__device__ __forceinline__ void chunk_block(const ChunkRegs<PREC, MATS> &r, const s16x4 (&xh)[NQ],
                                            const s16x4 (&xl)[NQ], f32x4 (&blk)[MATS][NQ])
{
#pragma unroll
    for (int m = 0; m < MATS; ++m)
#pragma unroll
        for (int q = 0; q < NQ; ++q) blk[m][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    block_step<PREC, MATS, NQ, J, 0>(r, xh, xl, blk);
    block_step<PREC, MATS, NQ, J, 1>(r, xh, xl, blk);
    block_step<PREC, MATS, NQ, J, 2>(r, xh, xl, blk);
    block_step<PREC, MATS, NQ, J, 3>(r, xh, xl, blk);
}

// acc += the block's sums times its scale
template <int PREC, int MATS, int NQ, int J>
__device__ __forceinline__ void add_block(const ChunkRegs<PREC, MATS> &r, const f32x4 (&blk)[MATS][NQ],
                                          f32x4 (&acc)[MATS][NQ])
{
#pragma unroll
    for (int m = 0; m < MATS; ++m)
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[m][q][i] = fmaf(blk[m][q][i], r.s[m][J], acc[m][q][i]);
}

template <int PREC, int MATS, int NQ>
__device__ __forceinline__ void compute_chunk(const ChunkRegs<PREC, MATS> &r, const TokenRegs<NQ> &x, int turn_src,
                                              f32x4 (&acc)[MATS][NQ])
{
    s16x4 xh[NQ], xl[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        uint32_t h01, l01, h23, l23;
        split_pair(x.x[q].x, x.x[q].y, h01, l01);
        split_pair(x.x[q].z, x.x[q].w, h23, l23);
        auto turn = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_bpermute(turn_src, (int)v); };
        xh[q] = as_s16x4(turn(h01), turn(h23));
        xl[q] = as_s16x4(turn(l01), turn(l23));
    }
    if constexpr (PREC == kFloat32) {
        block_step<PREC, MATS, NQ, 0, 0>(r, xh, xl, acc);
        block_step<PREC, MATS, NQ, 0, 1>(r, xh, xl, acc);
        block_step<PREC, MATS, NQ, 0, 2>(r, xh, xl, acc);
        block_step<PREC, MATS, NQ, 0, 3>(r, xh, xl, acc);
    } else {
        // a block's sums are scaled while the next block's products run
        f32x4 blk[2][MATS][NQ];
        chunk_block<PREC, MATS, NQ, 0>(r, xh, xl, blk[0]);
        chunk_block<PREC, MATS, NQ, 1>(r, xh, xl, blk[1]);
        add_block<PREC, MATS, NQ, 0>(r, blk[0], acc);
        chunk_block<PREC, MATS, NQ, 2>(r, xh, xl, blk[0]);
        add_block<PREC, MATS, NQ, 1>(r, blk[1], acc);
        chunk_block<PREC, MATS, NQ, 3>(r, xh, xl, blk[1]);
        add_block<PREC, MATS, NQ, 2>(r, blk[0], acc);
        add_block<PREC, MATS, NQ, 3>(r, blk[1], acc);
    }
}

// Where the M rows of a slice come from: positions p0 .. p0 + M - 1 of the
// dispatch (kByPosition), the routed (token, slot) entries list[0 .. M) of one
// expert, entry i = token * k + slot (kByEntry), or tokens t0 .. t0 + M - 1 of
// shared expert s (kShared).
enum { kByPosition = 0, kByEntry = 1, kShared = 2 };
struct SliceSrc {
    int mode;
    int p0;
    const int *list;
    int t0, s;
};

// input row (token row for gate/up, hidden row for down) and output row of
// slice token t
template <bool GATEUP, int MODE>
__device__ __forceinline__ int slice_in_row(const GemvArgs &a, const SliceSrc &sl, int t)
{
    if constexpr (MODE == kByPosition) return GATEUP ? a.tok[sl.p0 + t] : sl.p0 + t;
    else if constexpr (MODE == kByEntry) return GATEUP ? sl.list[t] / a.k : a.S * a.T + sl.list[t];
    else return GATEUP ? sl.t0 + t : sl.s * a.T + sl.t0 + t;
}
template <int MODE>
__device__ __forceinline__ int slice_out_row(const GemvArgs &a, const SliceSrc &sl, int t)
{
    if constexpr (MODE == kByPosition) return sl.p0 + t;
    else if constexpr (MODE == kByEntry) return a.S * a.T + sl.list[t];
    else return sl.s * a.T + sl.t0 + t;
}

// One slice of M <= 4*NQ tokens of group g against one panel of gate and up
// rows, or against MATS panels of down rows side by side; the workgroup's
// waves split K.
template <int PREC, bool GATEUP, int NQ, int MODE, int MATS, int NW, int RING>
__device__ __forceinline__ void run_slice(const GemvArgs &a, char *lds, int g, const SliceSrc &sl, int M,
                                          int panel)
{
    constexpr int CB = Chunk<PREC>::CB;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // this wave's chunks of K
    const int nch = a.nblocks / CB;
    const int c0 = wave * nch / NW, c1 = (wave + 1) * nch / NW;
    PanelSrc src[MATS];
    panel_src<PREC, GATEUP, MATS>(a, g, panel, src);
    const uint32_t vo = (uint32_t)lane * 16;

    // tokens: with NB = 4 CB steps per chunk, lane NB t + b loads the four
    // k-values of step b of token t of each quad (whole cache lines; lanes
    // past 4 NB repeat), and once split, lane 4 b + t fetches them from it,
    // where the matrix instruction of step b broadcasts its A from (loading
    // them there directly touches four rows per 64 bytes: down 26.4 -> 25.5
    // us, 33.4 -> 31.3 at 113 tokens, 2048 x 1024 FP4 rows).  Padding tokens
    // (t >= M) read past the input buffer and get zeros.
    const __amdgpu_buffer_rsrc_t xin = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.in), 0, (int)(a.in_rows * a.ld_in * 4), kRawBufferWord3);
    uint32_t xo[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int t = 4 * q + ((lane / (4 * CB)) & 3);
        xo[q] = 0x80000000u;  // past the buffer: zeros
        if (t < M)
            xo[q] = (uint32_t)slice_in_row<GATEUP, MODE>(a, sl, t) * (uint32_t)a.ld_in * 4u +
                    (uint32_t)(lane & (4 * CB - 1)) * 16u;
    }
    const int turn_src = ((lane & 3) * (4 * CB) + ((lane >> 2) & (4 * CB - 1))) * 4;

    // the epilogue's biases are requested before the ring, so that the loads
    // in flight at the main loop's entry are the ring's alone, in ring order,
    // as on its back edge
    const int row = panel * 64 + lane;
    const bool writer = wave < 4 && row < a.rows;
    float bias[MATS];
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
        const int rm = GATEUP ? row : min(row + 64 * m, a.rows - 1);
        bias[m] = writer ? (GATEUP && m ? a.b1 : a.b0)[(size_t)g * a.rows + rm] : 0.f;
    }

    // Every load of the ring is issued unconditionally, so that the compiler
    // can count the loads in flight and wait for one chunk at a time (loads
    // under a branch make it wait for all of them).  Past the wave's last
    // chunk the ring re-loads that chunk: cache hits, never used.
    const int clast = c1 > c0 ? c1 - 1 : c0;
    ChunkRegs<PREC, MATS> r[RING];
    TokenRegs<NQ> x[RING];
#pragma unroll
    for (int i = 0; i < RING; ++i) {
        // the scheduling barriers keep the ring's loads in ring order here
        // and in the loop: the compiler's wait before each chunk must hold
        // for the loads in flight both at the loop's entry and on its back
        // edge, so a different order here (say all codes, then all scales)
        // would make it wait for the next chunk's loads as well
        __builtin_amdgcn_sched_barrier(0);
        load_chunk<PREC, MATS>(r[i], src, vo, min(c0 + i, clast));
        load_tokens<PREC, NQ>(x[i], xin, xo, min(c0 + i, clast));
    }
    __builtin_amdgcn_sched_barrier(0);

    f32x4 acc[MATS][NQ];
#pragma unroll
    for (int m = 0; m < MATS; ++m)
#pragma unroll
        for (int q = 0; q < NQ; ++q) acc[m][q] = f32x4{0.f, 0.f, 0.f, 0.f};

    // ring of RING chunk buffers: once chunk ch is computed, its buffer
    // takes chunk ch + RING.  The loop body computes every buffer with no
    // branch, so the loads in flight on its back edge are exactly the ring's
    // and the compiler waits, before each chunk, for that chunk's loads only
    // (with a conditional compute in the body it also waited for the next
    // buffer's loads, leaving about one chunk in flight); the last
    // c1 - ch < RING chunks, already in the ring, are computed after it.
    int ch = c0;
    for (; ch + RING <= c1; ch += RING) {
#pragma unroll
        for (int j = 0; j < RING; ++j) {
            compute_chunk<PREC, MATS, NQ>(r[j], x[j], turn_src, acc);
            __builtin_amdgcn_sched_barrier(0);
            load_chunk<PREC, MATS>(r[j], src, vo, min(ch + j + RING, clast));
            load_tokens<PREC, NQ>(x[j], xin, xo, min(ch + j + RING, clast));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int j = 0; j + 1 < RING; ++j)
        if (ch + j < c1) compute_chunk<PREC, MATS, NQ>(r[j], x[j], turn_src, acc);

    // sum the partial K ranges through LDS; wave w < 4 then finishes token
    // 4 q + w of every quad
    static_assert(NW >= 4, "one wave per token of a quad in the epilogue");
    float *red = reinterpret_cast<float *>(lds);
    auto slot = [&](int wv, int m, int q, int i) { return (((wv * MATS + m) * NQ + q) * 4 + i) * 64 + lane; };
#pragma unroll
    for (int m = 0; m < MATS; ++m)
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[slot(wave, m, q, i)] = acc[m][q][i];
    __syncthreads();
    if (!writer) return;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int t = 4 * q + wave;
        if (t >= M) continue;
        float v[MATS];
#pragma unroll
        for (int m = 0; m < MATS; ++m) {
            float s = 0.f;
#pragma unroll
            for (int wv = 0; wv < NW; ++wv) s += red[slot(wv, m, q, wave)];
            v[m] = s;
        }
        const size_t orow = (size_t)slice_out_row<MODE>(a, sl, t) * a.ld_out;
        float *out = a.out + orow + row;
        if (a.raw) {  // the bare products (the adapter path adds its terms and the bias)
            *out = v[0];
            if constexpr (GATEUP) a.raw_up[orow + row] = v[MATS - 1];
            else if constexpr (MATS == 2) {
                if (row + 64 < a.rows) out[64] = v[1];
            }
        } else if constexpr (GATEUP) {
            float gv = v[0] + bias[0];
            float uv = v[1] + bias[MATS - 1];
            if (a.clamp > 0.f) {
                gv = fminf(gv, a.clamp);                   // ClampedSiLU: x > L -> silu(L)
                uv = fminf(fmaxf(uv, -a.clamp), a.clamp);  // ClampedLinear
            }
            *out = silu(gv) * uv;
        } else if (a.final_out) {
            // the combine of mixtureofexperts.go:192-205 for at most two
            // contributions per row: shared experts with weight 1, a routed
            // expert with its token's gate for it
            int tk;
            float wgt = 1.0f;
            if constexpr (MODE == kByEntry) {
                tk = sl.list[t] / a.k;
                wgt = a.gates32[sl.list[t]];
            } else if constexpr (MODE == kShared) {
                tk = sl.t0 + t;
            } else {
                tk = a.tok_all[sl.p0 + t];
                if (g >= a.S) {
                    const int e = g - a.S;
                    for (int j = 0; j < a.k; ++j)
                        if (a.chosen[(size_t)tk * a.k + j] == e) wgt = a.gates32[(size_t)tk * a.k + j];
                }
            }
#pragma unroll
            for (int m = 0; m < MATS; ++m)
                if (row + 64 * m < a.rows)
                    __hip_atomic_fetch_add(a.final_out + (size_t)tk * a.rows + row + 64 * m, wgt * (v[m] + bias[m]),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
#pragma unroll
            for (int m = 0; m < MATS; ++m)
                if (row + 64 * m < a.rows) out[64 * m] = v[m] + bias[m];
        }
    }
}

}  // namespace

// blockIdx.x = panel of 64 output rows, blockIdx.y = token slice (the
// dispatch wrote the slice count and a (group, first position, positions)
// descriptor per slice; slices past the last exit).
template <int PREC, bool GATEUP, bool SELF, int MATS, int NW, int RING>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 3 : 4) void gemv_kernel(GemvArgs a)
{
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int y = blockIdx.y;
    if constexpr (!SELF) {
        const int nslices = *a.count;
        const int4 dsc = a.desc[y];  // in bounds for every slice of the grid
        if (y >= nslices) return;    // workgroup-uniform
        const SliceSrc sl{kByPosition, dsc.y, nullptr, 0, 0};
        if (dsc.z <= 0) return;  // workgroup-uniform
        const int panel0 = blockIdx.x * (GATEUP ? 1 : MATS);
        if (dsc.z <= 4) run_slice<PREC, GATEUP, 1, kByPosition, MATS, NW, RING>(a, lds, dsc.x, sl, dsc.z, panel0);
        else run_slice<PREC, GATEUP, 2, kByPosition, MATS, NW, RING>(a, lds, dsc.x, sl, dsc.z, panel0);
        return;
    } else {
        const int nsh = a.S * a.shared_slices;
        if (y < nsh) {  // 8 tokens of a shared expert
            const int s = y / a.shared_slices;
            const SliceSrc sl{kShared, 0, nullptr, (y - s * a.shared_slices) * kGemvSlice, s};
            const int m = min(kGemvSlice, a.T - sl.t0);
            const int panel0 = blockIdx.x * (GATEUP ? 1 : MATS);
            if (m <= 4) run_slice<PREC, GATEUP, 1, kShared, MATS, NW, RING>(a, lds, s, sl, m, panel0);
            else run_slice<PREC, GATEUP, 2, kShared, MATS, NW, RING>(a, lds, s, sl, m, panel0);
            return;
        }
        // routed experts: rows [nsh, nsh + E) are each expert's first 8
        // entries, the T k / 8 rows after them whatever the experts hold beyond
        // (at most that many passes of 8 in all): extra row j counts every
        // expert's entries and takes the j-th further pass in expert order, so
        // a crowded expert's passes run side by side.
        int *list = reinterpret_cast<int *>(lds + a.list_off);
        int *found = list + a.T * a.k;  // entries of the expert, or the extra row's expert and pass
        const int n = a.T * a.k;
        int e = y - nsh, first = 0;
        if (e >= a.E) {
            int *hist = found + 2;
            for (int i = threadIdx.x; i < a.E; i += 64 * NW) hist[i] = 0;
            __syncthreads();
            for (int i = threadIdx.x; i < n; i += 64 * NW) atomicAdd(&hist[a.chosen[i]], 1);
            __syncthreads();
            if (threadIdx.x < 64) {
                const int j = e - a.E, lane = threadIdx.x;
                const int per = (a.E + 63) >> 6, e0 = lane * per, e1 = min(a.E, e0 + per);
                int more = 0;  // further passes of this lane's experts
                for (int i = e0; i < e1; ++i) more += max(0, (hist[i] - 1) / kGemvSlice);
                int before = more;
#pragma unroll
                for (int off = 1; off < 64; off <<= 1) {
                    const int v = __shfl_up(before, off);
                    if (lane >= off) before += v;
                }
                before -= more;
                if (lane == 63) {
                    found[0] = before + more > j ? 0 : -1;  // -1: no such pass
                }
                for (int i = e0; i < e1; ++i) {
                    const int m = max(0, (hist[i] - 1) / kGemvSlice);
                    if (j >= before && j < before + m) {
                        found[1] = i * 64 + (j - before + 1);  // T <= 512: at most 64 passes
                    }
                    before += m;
                }
            }
            __syncthreads();
            if (found[0] < 0) return;  // workgroup-uniform
            e = __builtin_amdgcn_readfirstlane(found[1] >> 6);
            first = __builtin_amdgcn_readfirstlane(found[1] & 63) * kGemvSlice;
            __syncthreads();  // before the list overwrites what was read
        }
        // expert e's entries in token order (the order of the reference's
        // rowsForExpert, mixtureofexperts.go:175-180), found by wave 0 with
        // ballots over `chosen` (four loads in flight per round)
        if (threadIdx.x < 64) {
            const int lane = threadIdx.x;
            int c = 0;
            for (int b0 = 0; b0 < n; b0 += 256) {
                int ch[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) ch[j] = a.chosen[min(b0 + j * 64 + lane, n - 1)];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int i = b0 + j * 64 + lane;
                    const bool hit = i < n && ch[j] == e;
                    const unsigned long long bal = __ballot(hit);
                    if (hit) list[c + __popcll(bal & ((1ull << lane) - 1ull))] = i;
                    c += __popcll(bal);
                }
            }
            if (lane == 0) *found = c;
        }
        __syncthreads();
        const int c = __builtin_amdgcn_readfirstlane(*found);
        if (c <= first) return;  // workgroup-uniform
        const SliceSrc sl{kByEntry, 0, list + first, 0, 0};
        const int m = min(kGemvSlice, c - first);
        const int panel0 = blockIdx.x * (GATEUP ? 1 : MATS);
        if (m <= 4) run_slice<PREC, GATEUP, 1, kByEntry, MATS, NW, RING>(a, lds, a.S + e, sl, m, panel0);
        else run_slice<PREC, GATEUP, 2, kByEntry, MATS, NW, RING>(a, lds, a.S + e, sl, m, panel0);
    }
}

// A few tokens (T <= kFewTokens, self-dispatching): only k T routed
// (token, slot) pairs and S T shared (expert, token) pairs have work, so
// each pair's rows are spread over the whole GPU.  A workgroup takes R rows
// of one pair (R divides the 64-row panel) and all of K; lane l of each of
// its 4 waves owns row l % R and unit phase l / R, so a load of the wave
// reads R rows' 16-byte units side by side (R x 16 contiguous bytes per
// phase).  Phase p of the workgroup takes units p, p + 4 * 64 / R, ... of
// its rows.  The pair's input row is staged once in LDS as fp32.  Per
// 16-value block: the codes times the input values, summed in order with
// fp32 FMAs, then times the block's scale into the lane's sum (the order of
// lowprecision/rows.go:207-257 within a block); the lanes' sums are added
// across phases and waves.  Same epilogues as gemv_kernel.
template <int PREC, bool GATEUP, int R>
__global__ __launch_bounds__(256) void gemv_few_kernel(GemvArgs a)
{
    constexpr int MATS = GATEUP ? 2 : 1;
    constexpr int PH = 64 / R;       // unit phases per wave
    constexpr int STRIDE = 4 * PH;   // units between a lane's units
    constexpr int VPU = PREC == kInt8 ? 16 : 32;  // values per 16-byte unit
    extern __shared__ __attribute__((aligned(16))) char lds[];
    float *xs = reinterpret_cast<float *>(lds);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // token t = blockIdx.z; blockIdx.y = shared expert s < S (row s T + t
    // of the self-dispatch layout), else routed slot j = blockIdx.y - S
    // (entry t k + j, row S T + t k + j).  The input row (the token, or the
    // pair's hidden row) is requested first: it does not depend on the
    // routing.
    const int t = blockIdx.z, yy = blockIdx.y;
    const int n0 = blockIdx.x * R;
    const int K = a.nblocks * 16;
    const int entry = t * a.k + yy - a.S;  // routed pairs only
    const int y = yy < a.S ? yy * a.T + t : a.S * a.T + entry;
    const int in_row = GATEUP ? t : y;
    const int out_row = y;
    const float4 *xin = reinterpret_cast<const float4 *>(a.in + (size_t)in_row * a.ld_in);
    // K <= 4096: four float4 per thread, loaded unconditionally (the index
    // clamped) and stored unconditionally into a 16 KiB row buffer (the
    // copies past K are never read): with a store under a branch the
    // compiler moved each load into the branch, behind the weight loads and
    // with a wait of its own
    float4 xv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) xv[i] = xin[min(tid + 256 * i, K / 4 - 1)];
    int g = yy;
    float wgt = 1.0f;
    if (yy >= a.S) {
        g = a.S + a.chosen[entry];
        wgt = a.gates32[entry];
    }
    g = __builtin_amdgcn_readfirstlane(g);
    const int nunits = a.row_bytes / 16;
    const int r = lane % R;
    const int n = n0 + r;
    const int panel = n0 >> 6, prow = (n0 & 63) + r;

    PanelSrc src[MATS];
    {
        const size_t wpanel = (size_t)panel * 64 * a.row_bytes;
        const int wbytes = 64 * a.row_bytes;
        const size_t spanel = (size_t)panel * 64 * a.nblocks;
        const int sbytes = 64 * a.nblocks * 4;
#pragma unroll
        for (int m = 0; m < MATS; ++m) {
            const void *w = m == 0 ? a.w0 : a.w1;
            const float *sc = m == 0 ? a.s0 : a.s1;
            src[m].codes = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<char *>(reinterpret_cast<const char *>(w)) + (size_t)g * a.w_group_stride + wpanel, 0,
                wbytes, kRawBufferWord3);
            src[m].scales = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(sc) + (size_t)g * a.s_group_stride + spanel, 0, sbytes, kRawBufferWord3);
        }
    }
    constexpr int UB = 4;  // units of a lane in flight together
    float sum[MATS];
#pragma unroll
    for (int m = 0; m < MATS; ++m) sum[m] = 0.f;
    const int ulanes = nunits / STRIDE;  // units per lane (the launcher checks the division)

    // unit u = U0 + q of the lane: U0 = wave PH + j STRIDE (uniform, a
    // multiple of 4) and q = lane / R; its first scale block b = u BPU sits
    // at (b / 4) 1024 + (b % 4) 4 + row 16 in the panel's scales
    constexpr int BPU = VPU / 16;  // scale blocks per unit
    const int q = lane / R;
    const uint32_t cvo = (uint32_t)prow * 16u + (uint32_t)q * 1024u;
    const uint32_t svo = (uint32_t)prow * 16u + (uint32_t)((q * BPU) >> 2) * 1024u + (uint32_t)((q * BPU) & 3) * 4u;
    uint4 c[UB][MATS];
    float sc[UB][MATS][BPU];
    // the lane's units j0 .. j0 + UB - 1 (past its last unit: the last unit
    // again, never used)
    auto load_units = [&](int j0) {
#pragma unroll
        for (int i = 0; i < UB; ++i) {
            const int U0 = wave * PH + min(j0 + i, ulanes - 1) * STRIDE;
#pragma unroll
            for (int m = 0; m < MATS; ++m) {
                c[i][m] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(src[m].codes, cvo,
                                                                                         U0 * 1024, 0));
                const int soff = (U0 * BPU / 4) * 1024;
                if constexpr (BPU == 1) {
                    sc[i][m][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src[m].scales, svo,
                                                                                                soff, 0));
                } else {
                    const float2 v = __builtin_bit_cast(
                        float2, __builtin_amdgcn_raw_buffer_load_b64(src[m].scales, svo, soff, 0));
                    sc[i][m][0] = v.x;
                    sc[i][m][1] = v.y;
                }
            }
        }
    };
    load_units(0);
    // the input row into LDS (K fp32 values, K a multiple of 64)
#pragma unroll
    for (int i = 0; i < 4; ++i) reinterpret_cast<float4 *>(xs)[tid + 256 * i] = xv[i];
    __syncthreads();
    for (int j0 = 0;;) {
#pragma unroll
        for (int i = 0; i < UB; ++i) {
            if (j0 + i >= ulanes) break;  // wave-uniform
            const int u = wave * PH + (j0 + i) * STRIDE + q;
            const float4 *xq = reinterpret_cast<const float4 *>(xs + u * VPU);
#pragma unroll
            for (int blk = 0; blk < BPU; ++blk) {
                float xb[16];
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const float4 v = xq[blk * 4 + h];
                    xb[4 * h] = v.x;
                    xb[4 * h + 1] = v.y;
                    xb[4 * h + 2] = v.z;
                    xb[4 * h + 3] = v.w;
                }
#pragma unroll
                for (int m = 0; m < MATS; ++m) {
                    float acc = 0.f;
                    if constexpr (PREC == kInt8) {
#pragma unroll
                        for (int h = 0; h < 4; ++h) {
                            const uint32_t d = comp_rt(c[i][m], h);
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                acc = fmaf((float)(int)(int8_t)(d >> (8 * e)), xb[4 * h + e], acc);
                        }
                    } else {
                        // FP4: block blk is dwords 2 blk, 2 blk + 1; each byte
                        // holds two values, the even one in the low nibble
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const uint32_t d = comp_rt(c[i][m], 2 * blk + h);
                            const f32x2 f[4] = {__builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 0),
                                                __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 1),
                                                __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 2),
                                                __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 3)};
#pragma unroll
                            for (int sel = 0; sel < 4; ++sel) {
                                acc = fmaf(f[sel].x, xb[8 * h + 2 * sel], acc);
                                acc = fmaf(f[sel].y, xb[8 * h + 2 * sel + 1], acc);
                            }
                        }
                    }
                    sum[m] = fmaf(acc, sc[i][m][blk], sum[m]);
                }
            }
        }
        j0 += UB;
        if (j0 >= ulanes) break;
        load_units(j0);
    }
    // across the phases of the wave, then across the waves in wave order
#pragma unroll
    for (int m = 0; m < MATS; ++m)
#pragma unroll
        for (int off = R; off < 64; off <<= 1) sum[m] += __shfl_xor(sum[m], off);
    __syncthreads();  // every read of the staged row is done
    float *red = xs;  // [4][MATS][R]
    if (lane < R)
#pragma unroll
        for (int m = 0; m < MATS; ++m) red[(wave * MATS + m) * R + lane] = sum[m];
    __syncthreads();
    if (wave != 0 || lane >= R || n >= a.rows) return;
    float v[MATS];
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
        float t = 0.f;
#pragma unroll
        for (int wv = 0; wv < 4; ++wv) t += red[(wv * MATS + m) * R + lane];
        v[m] = t;
    }
    const float b0 = a.b0[(size_t)g * a.rows + n];
    if constexpr (GATEUP) {
        float gv = v[0] + b0;
        float uv = v[1] + a.b1[(size_t)g * a.rows + n];
        if (a.clamp > 0.f) {
            gv = fminf(gv, a.clamp);                   // ClampedSiLU: x > L -> silu(L)
            uv = fminf(fmaxf(uv, -a.clamp), a.clamp);  // ClampedLinear
        }
        a.out[(size_t)out_row * a.ld_out + n] = silu(gv) * uv;
    } else if (a.final_out) {
        // at most two contributions per output row (see gemv_kernel)
        __hip_atomic_fetch_add(a.final_out + (size_t)t * a.rows + n, wgt * (v[0] + b0), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    } else {
        a.out[(size_t)out_row * a.ld_out + n] = v[0] + b0;
    }
}

namespace {

// LDS: the cross-wave partial sums.
size_t gemv_lds_bytes(int mats, int nw)
{
    return (size_t)nw * mats * 2 * 4 * 64 * sizeof(float);
}

template <int PREC, bool GATEUP, int MATS, int NW, int RING>
hipError_t launch_panels(const GemvArgs &a0, int max_slices, hipStream_t s)
{
    GemvArgs a = a0;
    size_t lds = gemv_lds_bytes(MATS, NW);
    if (a.self_dispatch) {
        // after the slice's LDS: the routed expert's entry list, its length (two
        // ints) and an extra row's count per expert
        a.list_off = (int)((lds + 15) / 16 * 16);
        lds = (size_t)a.list_off + ((size_t)a.T * a.k + 2 + a.E) * sizeof(int);
    }
    if (lds > 64 * 1024) return hipErrorInvalidValue;  // 32 KiB and lists of at most 512 choices and 256 experts
    constexpr int kRows = kPanelRows * (GATEUP ? 1 : MATS);  // rows of a workgroup
    const dim3 grid((a.rows + kRows - 1) / kRows, max_slices);
    if (a.self_dispatch)
        hipLaunchKernelGGL((gemv_kernel<PREC, GATEUP, true, MATS, NW, RING>), grid, dim3(64 * NW), lds, s, a);
    else hipLaunchKernelGGL((gemv_kernel<PREC, GATEUP, false, MATS, NW, RING>), grid, dim3(64 * NW), lds, s, a);
    return hipGetLastError();
}

template <bool GATEUP, int PREC>
hipError_t launch_prec(const GemvArgs &a, int max_slices, hipStream_t s)
{
    static_assert(kGemvSlice <= 8, "at most two token quads per slice");
    if (a.nblocks % Chunk<PREC>::CB) return hipErrorInvalidValue;
    const long long busy = a.self_dispatch ? (long long)a.S * a.shared_slices + std::min(a.E, a.T * a.k)
                                           : (long long)max_slices;
    // Down over many workgroups: a wave takes two panels side by side, so that
    // its tokens are read and split once for both (2048 x 1024 FP4 rows, 64
    // experts: 25.6 -> 24.3 us at 64 tokens, 31.1 -> 28.6 us at 113).  With
    // fewer than two rounds of busy workgroups at the halved count the grid no
    // longer fills the GPU (1024 x 2048 Int8 rows, 16 experts: 12.2 -> 15.3
    // us), so those keep one panel per wave.
    if (!GATEUP && a.rows >= 128 && (long long)(a.rows / 128) * busy >= 1024)
        return launch_panels<PREC, GATEUP, 2, 4, 2>(a, max_slices, s);
    constexpr int MATS = GATEUP ? 2 : 1;
    // Four waves over a ring of two chunks, except where K holds a chunk for
    // each of eight and these do better: gate/up over fewer than 512 busy
    // workgroups (Int8 and FP4: eight waves over a ring of one; d = 2048, h =
    // 1024, 64 + 1 experts over 7 tokens, the layer 48.4 -> 44.9 us in FP4 and
    // 62.5 -> 58.9 in Int8; over 16 tokens, with twice the workgroups, 54.8
    // against 59.3 in FP4), and Float32 with K >= 1024 in a self-dispatching
    // launch (a ring of two; d = 1024, h = 2048, 16 experts over 32 tokens 88.4
    // -> 82.7; elsewhere it loses: K = 256, 700 tokens 43.7 against 48.6).
    if constexpr (PREC == kFloat32) {
        if (a.self_dispatch && a.nblocks >= 64) return launch_panels<PREC, GATEUP, MATS, 8, 2>(a, max_slices, s);
    } else if (GATEUP && a.nblocks >= 32 && (long long)((a.rows + kPanelRows - 1) / kPanelRows) * busy < 512) {
        return launch_panels<PREC, GATEUP, MATS, 8, 1>(a, max_slices, s);
    }
    return launch_panels<PREC, GATEUP, MATS, 4, 2>(a, max_slices, s);
}

// Up to this many tokens the few-token kernel runs: it streams an expert's
// weights once per (token, slot) pair, where gemv_kernel streams them once per
// slice of up to 8 tokens, and measured faster up to 6 tokens (C2 and a C5
// block; about even at 8).
constexpr int kFewTokens = 6;
// LDS of the few-token kernel: its row buffer, four float4 per thread
constexpr size_t kFewRowBytes = 4 * 256 * sizeof(float4);

template <bool GATEUP, int PREC, int R>
hipError_t launch_few(const GemvArgs &a, hipStream_t s)
{
    const size_t lds = kFewRowBytes;  // the token row (K <= 4096 values); >= the reduction's 4 x 2 x R floats
    const dim3 grid((a.rows + R - 1) / R, a.S + a.k, a.T);
    hipLaunchKernelGGL((gemv_few_kernel<PREC, GATEUP, R>), grid, dim3(256), lds, s, a);
    return hipGetLastError();
}

// A few tokens through a layer of K >= 512 values: the few-token kernel, with
// R = 16 rows per workgroup when that still gives 256 workgroups, else 8.  Int8 and
// FP4 rows whose 16-byte units divide evenly among a workgroup's unit
// phases.  Returns false (nothing launched) otherwise.
template <bool GATEUP>
bool launch_few_tokens(const GemvArgs &a, int precision, hipStream_t s, hipError_t &e)
{
    if (!a.self_dispatch || a.T < 1 || a.T > kFewTokens || a.raw || (precision != kInt8 && precision != kFP4))
        return false;
    if (a.nblocks < 32 || a.nblocks * 16 > 4096) return false;
    const int nunits = a.row_bytes / 16;
    const int R = (long long)(a.rows / 16) * (a.S + a.k) * a.T >= 256 ? 16 : 8;
    if (a.row_bytes % 16 != 0 || nunits % (4 * (64 / R)) != 0) return false;
    if (precision == kInt8)
        e = R == 16 ? launch_few<GATEUP, kInt8, 16>(a, s) : launch_few<GATEUP, kInt8, 8>(a, s);
    else
        e = R == 16 ? launch_few<GATEUP, kFP4, 16>(a, s) : launch_few<GATEUP, kFP4, 8>(a, s);
    return true;
}

template <bool GATEUP>
hipError_t launch_any(const GemvArgs &a, int precision, int max_slices, hipStream_t s)
{
    if (max_slices <= 0) return hipSuccess;
    hipError_t e1 = hipSuccess;
    if (launch_few_tokens<GATEUP>(a, precision, s, e1)) return e1;
    // the input rows are read through a buffer resource with 32-bit offsets
    if (a.in_rows <= 0 || a.in_rows * a.ld_in * 4 > 0x7fffffffLL) return hipErrorInvalidValue;
    switch (precision) {
    case kInt8: return launch_prec<GATEUP, kInt8>(a, max_slices, s);
    case kFP4: return launch_prec<GATEUP, kFP4>(a, max_slices, s);
    case kFloat32: return launch_prec<GATEUP, kFloat32>(a, max_slices, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_gemv_gateup(const GemvArgs &a, int precision, int max_slices, hipStream_t s)
{
    return launch_any<true>(a, precision, max_slices, s);
}

hipError_t launch_gemv_down(const GemvArgs &a, int precision, int max_slices, hipStream_t s)
{
    return launch_any<false>(a, precision, max_slices, s);
}

}  // namespace gtmoe
