// Prompts of a few tokens (at most kPfSmallRows): layer_prefill (model.cpp:144-181) in five
// kernels per layer.
//
// k_pf_small_split  the prompt's embedding rows, prepared for the first GEMM
// k_pf_small        one GEMM of the layer, M <= 16 rows against a matrix in its HBM layout:
//                   rmsnorm (layers.cpp:7-12) of the rows where the reference applies it, then
//                   store (+ bias), residual add, or silu(gate) * up, and the result prepared
//                   for the GEMM that reads it
// k_pf_small_attn   RoPE of q and k, the KV store, and causal attention of the rows over
//                   themselves (attn_prefill, attention.cpp:82-111: a prompt that starts its
//                   prefill call attends to nothing else)
//
// What bounds it: every weight is read once whatever M is, so the floor is the weight stream;
// above it stand the kernels' launch, fill and drain. The tiles for longer prompts
// (k_prefill.hip) need row scales, which no workgroup of the GEMM before knows, and K in slices
// over workgroups to fill the chip at so few rows: ten dependent kernels a layer, three of
// them to add slices and two to split rows. Here a workgroup takes one 16-column tile over
// the whole of K, its waves a K range each with the sums added through LDS, and its epilogue
// leaves its columns as the next GEMM's operand. (With fp32 rows between the kernels, each
// workgroup splitting all of its input, the splitting's VALU work set the time.) A whole prompt,
// device time before and now: Llama-3.2-1B shape, 6 tokens, Q8_0 1,399 -> 902 us, mixed Q4 1,336
// -> 840, Q6_K 9,120 -> 1,066, F16 1,347 -> 1,141; 16 tokens of the Qwen2.5-0.5B shape 1,914 ->
// 1,025, of the Qwen2.5-1.5B shape 3,348 -> 1,631. Of a layer's 54 us at 6 tokens the weights'
// floor is 10; gate / up take 16.7, QKV 8.9, attention 4.7, wo and down 22.
//
// Numerics: an fp32 activation is the sum of three bf16 (8 bits each, by truncation, exact
// with fp32's range, so no row scales), and the block integers of Q8_0, Q4_0 and Q4_1 are exact
// in bf16: every product of three v_mfma_f32_16x16x32_bf16 is exact, their sum over a block is
// fp32's, and d (and Q4_1's m) scale the block sums in fp32 (quant.cpp:266-321). F16 weights
// and Q6_K's sc (u - 32) (at most 13 bits) are two bf16, five MFMAs (the dropped third piece
// times second piece is 2^-24 of the product). rmsnorm's weights multiply the activations before
// they are split, its row factor the finished sum. (F32 weights would be three pieces, with more
// MFMAs and registers than pay: such models take the longer prompts' kernels.)
//
// Operand layout: xa[32-element block][piece 0..2][lane group c][row][8], the rows
// rounded up to 4 (every workgroup reads the whole operand, so its bytes count). The sums of
// squares come as one partial per row and 16-column tile, ssp[tile][row]. Rows M.. hold
// anything: an MFMA's output row depends on its own input row only.
#include "dev_common.hpp"
#include "tf_internal.hpp"

namespace tfk {
namespace {

typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4_t mfma(b8_t a, b8_t b, f4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The upper halves of a and b: two bf16 by truncation.
__device__ __forceinline__ uint32_t pack_hi(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float trunc_bf16(float v) { return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u); }

__device__ __forceinline__ b8_t pack8(const float (&v)[8]) {
    const tf_u32x4 p = {pack_hi(v[0], v[1]), pack_hi(v[2], v[3]), pack_hi(v[4], v[5]), pack_hi(v[6], v[7])};
    return __builtin_bit_cast(b8_t, p);
}
// v as the sum of N bf16 pieces (v holds the remainder after each)
template <int N>
__device__ __forceinline__ void split_bf16(float (&v)[8], b8_t (&p)[N]) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
        p[n] = pack8(v);
        if (n + 1 < N)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = v[e] - trunc_bf16(v[e]);
    }
}

// Weight and activation fragments hold the four 8-element units of a 32-element block in the
// order 0, 2, 1, 3: lane group c = l / 16 takes unit kUnit(c). With it, a lane can load 16
// contiguous bytes of its row (64 bytes a row and instruction; the 8 bytes a lane wants of each
// block would be 32 a row, and the rows' lines fetched several times over), and lane swaps turn
// that into fragments.
__device__ __forceinline__ int unit_of(int c) { return ((c & 1) << 1) | (c >> 1); }

// a's lanes 32..63 for b's lanes 0..31
__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
// even: v's 16-lane rows 0, 0, 2, 2; odd: its rows 1, 1, 3, 3
__device__ __forceinline__ void spread16(uint32_t v, uint32_t& even, uint32_t& odd) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    even = r[0];
    odd = r[1];
}

// A weight format. A stage is four 32-element blocks of 16 rows (row l % 16 in lane l):
//   kPieces  bf16 pieces of an element
//   kSuper   Q6_K: kScale's bytes are sub-block scales, d comes per 8 blocks
//   kScale   bytes a block in the s stream (0: none); the scales come from LDS, put there as
//            they lie (16 rows of a matrix are one run of the stream)
//   kMin     Q4_1's min term
//   load()   the stage's bytes: lane group c's share of blocks 4 s .. (past the row: the last
//            whole stage's place, which the zero scale of blocks past K takes out)
//   spread() those bytes as the fragments' raw values
//   vals()   the lane's eight elements of block j as floats, without the block scale
template <int T>
struct SmW;

// bytes of a row of the q stream from which 16 can be loaded at 64 s: in bounds for every s
__device__ __forceinline__ int clamp_off(int off, int row_bytes) { return off + 16 <= row_bytes ? off : row_bytes - 16; }

template <>
struct SmW<TF_HIP_TYPE_Q8_0> {
    static constexpr int kPieces = 1, kScale = 2;
    static constexpr bool kMin = false, kSuper = false;
    struct Raw {
        uint4 q[2];
    };
    __device__ static void load(const DevMat& m, int64_t row, int s, int c, Raw& w) {
        const uint8_t* p = m.q + row * m.K;
        w.q[0] = gload_u4(p + clamp_off(128 * s + 16 * c, (int)m.K));
        w.q[1] = gload_u4(p + clamp_off(128 * s + 64 + 16 * c, (int)m.K));
    }
    // lane group c holds units 2 c, 2 c + 1 of two blocks' eight: swapping halves leaves units
    // 0 2 1 3 of the first block in x, y and of the second in z, w
    __device__ static void spread(Raw& w, int) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            swap32(w.q[i].x, w.q[i].z);
            swap32(w.q[i].y, w.q[i].w);
        }
    }
    __device__ static void vals(const Raw& w, int j, int, uint32_t, float (&v)[8]) {
        const uint4 q = w.q[j >> 1];
        const uint32_t a = j & 1 ? q.z : q.x, b = j & 1 ? q.w : q.y;
        v[0] = sb0(a); v[1] = sb1(a); v[2] = sb2(a); v[3] = sb3(a);
        v[4] = sb0(b); v[5] = sb1(b); v[6] = sb2(b); v[7] = sb3(b);
    }
};

// Four blocks of 16 nibble bytes, a block a lane group: bytes 0..7 hold units 0 (low nibbles)
// and 2 (high), bytes 8..15 units 1 and 3. p[j]: block j's 8 bytes for this lane group,
// low nibbles in groups 0 and 2, high in 1 and 3.
struct Nib {
    uint2 p[4];
    __device__ void spread(uint4 q) {
        swap32(q.x, q.z);
        swap32(q.y, q.w);
        spread16(q.x, p[0].x, p[1].x);
        spread16(q.y, p[0].y, p[1].y);
        spread16(q.z, p[2].x, p[3].x);
        spread16(q.w, p[2].y, p[3].y);
    }
};

template <bool MIN>
struct SmW4 {
    static constexpr int kPieces = 1, kScale = MIN ? 4 : 2;
    static constexpr bool kMin = MIN, kSuper = false;
    struct Raw {
        uint4 q;
        Nib n;
    };
    __device__ static void load(const DevMat& m, int64_t row, int s, int c, Raw& w) {
        w.q = gload_u4(m.q + row * (m.K / 2) + clamp_off(64 * s + 16 * c, (int)(m.K / 2)));
    }
    __device__ static void spread(Raw& w, int) { w.n.spread(w.q); }
    // nibble n: n - 8 (Q4_0) or n (Q4_1)
    __device__ static void vals(const Raw& w, int j, int c, uint32_t, float (&v)[8]) {
        const int sh = 4 * (c & 1);
        const uint32_t a = (w.n.p[j].x >> sh) & 0x0F0F0F0Fu, b = (w.n.p[j].y >> sh) & 0x0F0F0F0Fu;
        v[0] = ub0(a); v[1] = ub1(a); v[2] = ub2(a); v[3] = ub3(a);
        v[4] = ub0(b); v[5] = ub1(b); v[6] = ub2(b); v[7] = ub3(b);
        if (!MIN)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] -= 8.0f;
    }
};
template <>
struct SmW<TF_HIP_TYPE_Q4_0> : SmW4<false> {};
template <>
struct SmW<TF_HIP_TYPE_Q4_1> : SmW4<true> {};

template <>
struct SmW<TF_HIP_TYPE_Q6_K> {
    static constexpr int kPieces = 2, kScale = 2;
    static constexpr bool kMin = false, kSuper = true;
    struct Raw {
        uint4 q;
        uint2 h;      // the lane group's block's top bits
        Nib n;
        uint2 hi[4];  // every block's
    };
    __device__ static void load(const DevMat& m, int64_t row, int s, int c, Raw& w) {  // K % 256 == 0
        w.q = gload_u4(m.q + row * (m.K / 2) + 64 * s + 16 * c);
        w.h = gload_u2(m.q2 + row * (m.K / 4) + 32 * s + 8 * c);
    }
    __device__ static void spread(Raw& w, int) {
        w.n.spread(w.q);
        uint32_t x0 = w.h.x, x1 = w.h.x, y0 = w.h.y, y1 = w.h.y;
        swap32(x0, x1);  // rows 0 1 0 1, rows 2 3 2 3
        swap32(y0, y1);
        spread16(x0, w.hi[0].x, w.hi[1].x);
        spread16(x1, w.hi[2].x, w.hi[3].x);
        spread16(y0, w.hi[0].y, w.hi[1].y);
        spread16(y1, w.hi[2].y, w.hi[3].y);
    }
    // sc (u - 32); scales: the block's two int8
    __device__ static void vals(const Raw& w, int j, int c, uint32_t scales, float (&v)[8]) {
        const int u8 = unit_of(c), sh = 4 * (c & 1), hs = 2 * u8;
        const uint32_t a = ((w.n.p[j].x >> sh) & 0x0F0F0F0Fu) | (((w.hi[j].x >> hs) & 0x03030303u) << 4);
        const uint32_t b = ((w.n.p[j].y >> sh) & 0x0F0F0F0Fu) | (((w.hi[j].y >> hs) & 0x03030303u) << 4);
        const float sc = (float)(int8_t)(scales >> (8 * (u8 >> 1))), off = -32.0f * sc;
        const float u[8] = {ub0(a), ub1(a), ub2(a), ub3(a), ub0(b), ub1(b), ub2(b), ub3(b)};
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = fmaf(u[e], sc, off);
    }
};

template <>
struct SmW<TF_HIP_TYPE_F16> {
    static constexpr int kPieces = 2, kScale = 0;
    static constexpr bool kMin = false, kSuper = false;
    struct Raw {
        uint4 q[4];
    };
    __device__ static void load(const DevMat& m, int64_t row, int s, int c, Raw& w) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w.q[j] = gload_u4(m.q + row * m.K * 2 + clamp_off(256 * s + 64 * j + 16 * unit_of(c), (int)m.K * 2));
    }
    __device__ static void spread(Raw&, int) {}
    __device__ static void vals(const Raw& w, int j, int, uint32_t, float (&v)[8]) {
        const uint32_t q[4] = {w.q[j].x, w.q[j].y, w.q[j].z, w.q[j].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = h2f((q[e >> 1] >> (16 * (e & 1))) & 0xFFFFu);
    }
};

constexpr int kPieces = 3;
constexpr int kStageBlocks = 4;

// Rows a fragment holds: M rounded up to 4 (whole 64-byte pieces).
__host__ __device__ __forceinline__ int frag_rows(int M) { return (M + 3) / 4 * 4; }

// Writes row m's eight elements 8 e8 .. 8 e8 + 7 (v, consumed) into an operand of M rows.
__device__ __forceinline__ void put_pieces(b8_t* xa, int M, int m, int e8, float (&v)[8]) {
    const int R = frag_rows(M);
    b8_t p[kPieces];
    split_bf16<kPieces>(v, p);
    b8_t* o = xa + (int64_t)(e8 / 4) * kPieces * 4 * R + unit_of(e8 % 4) * R + m;
#pragma unroll
    for (int n = 0; n < kPieces; ++n) o[n * 4 * R] = p[n];
}

// NC columns of values (LDS rows) as the operand columns col0 .. col0 + NC - 1, and with norm
// weights g (LDS, this tile's) their products with g, the rows' sums of squares into ssp, a
// partial per 16 columns.
template <int NC>
__device__ __forceinline__ void put_tile(const float (&val)[kPfSmallRows][NC + 1], int tid, int M, int col0, const float* g, b8_t* xa, double* ssp) {
    if (tid < 2 * NC) {
        const int m = tid / (NC / 8), h = tid % (NC / 8);
        if (m < M) {
            float v[8];
            double ss = 0.0;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = val[m][8 * h + e];
                ss = fma((double)v[e], (double)v[e], ss);
                if (g) v[e] *= g[8 * h + e];
            }
            ss += __shfl_xor(ss, 1);
            if (g && h % 2 == 0) ssp[(int64_t)(col0 / 16 + h / 2) * kPfSmallRows + m] = ss;
            put_pieces(xa, M, m, col0 / 8 + h, v);
        }
    }
}

// x rows [M][D] as the first GEMM's operand: a workgroup per 16 columns.
__global__ __launch_bounds__(kBlock) void k_pf_small_split(const float* x, int D, int M, const float* g, b8_t* xa,
                                                           double* ssp) {
    __shared__ float val[kPfSmallRows][17];
    const int col0 = 16 * blockIdx.x;
    for (int o = threadIdx.x; o < 16 * M; o += kBlock) val[o >> 4][o & 15] = x[(int64_t)(o >> 4) * D + col0 + (o & 15)];
    __syncthreads();
    put_tile<16>(val, threadIdx.x, M, col0, g + col0, xa, ssp);
}

// One workgroup: NT 16-column output tiles (GEMV_SILU: the gate and the up rows of each), a K
// slice of nst stages (a.ks slices; all of K for a.ks = 1): wave w takes a run
// of its stages, two in flight. With K in slices, every workgroup writes its sums through to
// memory and counts itself in; the last one of a tile adds the slices in slice order (the same sum
// whichever is last) and goes on to the epilogue. No workgroup waits for another.
template <int MODE, int T, int NT>
__global__ __launch_bounds__(kBlock) void k_pf_small(const PfSmallArgs a) {
    using F = SmW<T>;
    constexpr int W = kWavesPerBlock;
    constexpr int NI = MODE == GEMV_SILU ? 2 * NT : NT;
    constexpr bool NORM = MODE != GEMV_RESID;  // rmsnorm goes before QKV and gate / up
    constexpr int NC = 16 * NT, NOUT = kPfSmallRows * NC;
    __shared__ float red[W][NI][4][64];
    __shared__ double red_ss[W][kPfSmallRows];
    __shared__ float val[kPfSmallRows][NC + 1], gl[NC];
    __shared__ int arrived;
    extern __shared__ __align__(16) unsigned char scl[];  // the scales of the tile's weight rows
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lc = lane >> 4;
    const int ks = a.ks, kslice = blockIdx.x % ks, grp = blockIdx.x / ks, u0 = grp * NT;
    // this workgroup's matrix and its row there (scalar selects, a segment per matrix; NT > 1
    // only where the segments hold whole groups of NT tiles)
    const int sg = MODE != GEMV_STORE ? 0
                                      : ((a.n_seg > 2 && u0 >= a.seg[2].sub0) ? 2 : ((a.n_seg > 1 && u0 >= a.seg[1].sub0) ? 1 : 0));
#define SM_SEL(f) (sg == 0 ? a.seg[0].f : (sg == 1 ? a.seg[1].f : a.seg[2].f))
    const int col0 = (u0 - SM_SEL(sub0)) * 16;
    DevMat wm[2];
    wm[0].K = wm[1].K = a.K;
    wm[0].q = SM_SEL(w.q);
    wm[0].q2 = SM_SEL(w.q2);
    wm[0].s = SM_SEL(w.s);
    wm[0].s2 = SM_SEL(w.s2);
    wm[1].q = a.seg[0].w2.q;
    wm[1].q2 = a.seg[0].w2.q2;
    wm[1].s = a.seg[0].w2.s;
    wm[1].s2 = a.seg[0].w2.s2;
    // weight tile ni: rows of matrix ni / NT (1: up) from col0 + 16 (ni % NT)

    const int nblk = a.K / 32, S = (nblk + kStageBlocks - 1) / kStageBlocks;
    const int s_lo = S * kslice / ks, s_hi = S * (kslice + 1) / ks, nst = s_hi - s_lo;
    const int sb = s_lo + nst * wave / W, se = s_lo + nst * (wave + 1) / W;
    const int R = frag_rows(a.M), xrow = l16 < R ? l16 : R - 1;
    const TF_GLOBAL b8_t* xp = (const TF_GLOBAL b8_t*)a.xa + lc * R + xrow;
    struct Stage {
        typename F::Raw w[NI];
        b8_t x[kStageBlocks][kPieces];
    };
    auto load = [&](int s, Stage& st) {
        s = s < se ? s : se - 1;
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) F::load(wm[ni / NT], col0 + 16 * (ni % NT) + l16, s, lc, st.w[ni]);
#pragma unroll
        for (int j = 0; j < kStageBlocks; ++j) {
            int blk = kStageBlocks * s + j;
            blk = blk < nblk ? blk : nblk - 1;
#pragma unroll
            for (int n = 0; n < kPieces; ++n) st.x[j][n] = xp[(blk * kPieces + n) * 4 * R];
        }
    };
    // the scales: LDS row (weight tile, row) of the slice's blocks, padded against bank conflicts
    const int b_lo = kStageBlocks * s_lo, n_b = kStageBlocks * nst;
    const int sw = F::kScale * n_b / 4 + 1;  // dwords a row
    const int d_lo = b_lo / 8, n_d = F::kSuper ? (b_lo + n_b + 7) / 8 - d_lo : 0, dw = (n_d + 1) / 2 + ((n_d / 2) % 2 ? 0 : 1);
    uint32_t* sc_lds = (uint32_t*)scl;
    uint16_t* d_lds = (uint16_t*)(sc_lds + NI * 16 * sw);
    // Small loads first, so that nothing below waits for the stages (loads complete in order): a
    // thread's share of a scale row (kTpr threads a row, the first kSc words each in registers),
    // the residual of its outputs, the next norm's weights, and the rows' partial sums of squares
    // (thread (row, group of tiles)).
    constexpr int kTpr = kBlock / (NI * 16), kSc = 4;
    const int sr = tid / kTpr, sk = tid % kTpr, sni = sr / 16;
    const int per = F::kScale * n_b / 4, row_words = F::kScale * nblk / 4, w_lo = F::kScale * b_lo / 4;
    const int64_t srow = col0 + 16 * (sni % NT) + sr % 16;
    const TF_GLOBAL uint32_t* sp = gptr((const uint32_t*)(sni / NT ? wm[1].s : wm[0].s)) + srow * row_words + w_lo;
    uint32_t scv[kSc];
    if (F::kScale)
#pragma unroll
        for (int i = 0; i < kSc; ++i) {
            const int k = sk + i * kTpr;
            scv[i] = sp[w_lo + k < row_words ? k : row_words - 1 - w_lo];
        }
    const TF_GLOBAL uint16_t* dsp = gptr((const uint16_t*)(sni / NT ? wm[1].s2 : wm[0].s2)) + srow * (nblk / 8) + d_lo;
    uint16_t dsv = 0;
    if (F::kSuper) dsv = dsp[sk < n_d ? sk : n_d - 1];
    constexpr int NV = (NOUT + kBlock - 1) / (kBlock);
    float yv[NV];
    if (MODE == GEMV_RESID)
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int o = tid + i * kBlock, row = o / NC;
            yv[i] = gptr(SM_SEL(y))[(int64_t)(row < a.M ? row : a.M - 1) * SM_SEL(ldy) + col0 + o % NC];
        }
    const float gv = a.onorm_w ? gptr(a.onorm_w)[col0 + tid % NC] : 0.0f;
    constexpr int kGroups = kBlock / kPfSmallRows, kSq = 4;
    const int sq_row = tid % kPfSmallRows, n_tiles = NORM ? a.K / 16 : 0;
    double sq[kSq];
    if (NORM)
#pragma unroll
        for (int i = 0; i < kSq; ++i) {
            const int t = tid / kPfSmallRows + i * kGroups;
            sq[i] = gptr(a.ssp)[(int64_t)(t < n_tiles ? t : n_tiles - 1) * kPfSmallRows + sq_row];
        }
    Stage s0, s1;
    if (sb < se) {
        load(sb, s0);
        load(sb + 1, s1);
    }
    if (F::kScale) {
#pragma unroll
        for (int i = 0; i < kSc; ++i) {
            const int k = sk + i * kTpr;
            // a word past the row's end: blocks past K, scale zero
            if (k < per) sc_lds[sr * sw + k] = w_lo + k < row_words ? scv[i] : 0u;
        }
        for (int k = sk + kSc * kTpr; k < per; k += kTpr) sc_lds[sr * sw + k] = w_lo + k < row_words ? sp[k] : 0u;
    }
    if (F::kSuper) {
        if (sk < n_d) d_lds[sr * 2 * dw + sk] = dsv;
        for (int k = sk + kTpr; k < n_d; k += kTpr) d_lds[sr * 2 * dw + k] = dsp[k];
    }
    if (tid < NC) gl[tid] = gv;
    __syncthreads();

    f4_t acc[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) acc[ni] = (f4_t){0.0f, 0.0f, 0.0f, 0.0f};
    const f4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const float one8[8] = {1, 1, 1, 1, 1, 1, 1, 1};
    const b8_t ones = pack8(one8);
    auto compute = [&](int s, Stage& st) {
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) F::spread(st.w[ni], lc);
#pragma unroll
        for (int j = 0; j < kStageBlocks; ++j) {
            const int bl = kStageBlocks * s + j - b_lo;  // block of the slice
            const bool in = kStageBlocks * s + j < nblk;
            b8_t wp[NI][F::kPieces];
            float wv[NI][8], dv[NI], mv[NI];
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) {
                const int r = 16 * ni + l16;
                uint32_t sc = 0;
                if (F::kScale == 2) sc = ((const uint16_t*)(sc_lds + r * sw))[bl];
                if (F::kScale == 4) sc = sc_lds[r * sw + bl];
                F::vals(st.w[ni], j, lc, sc, wv[ni]);
                dv[ni] = F::kSuper ? h2f(d_lds[r * 2 * dw + (b_lo + bl) / 8 - d_lo])
                                   : (F::kScale ? h2f(sc & 0xFFFFu) : (in ? 1.0f : 0.0f));
                mv[ni] = F::kMin ? h2f(sc >> 16) : 0.0f;
                split_bf16<F::kPieces>(wv[ni], wp[ni]);
            }
            const b8_t(&x)[kPieces] = st.x[j];
            f4_t t[NI], ts = zero;
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) t[ni] = mfma(x[0], wp[ni][0], zero);
            if (F::kMin) ts = mfma(x[0], ones, zero);
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) t[ni] = mfma(x[1], wp[ni][0], t[ni]);
            if (F::kMin) ts = mfma(x[1], ones, ts);
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) t[ni] = mfma(x[2], wp[ni][0], t[ni]);
            if (F::kMin) ts = mfma(x[2], ones, ts);
            if constexpr (F::kPieces == 2) {
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) t[ni] = mfma(x[0], wp[ni][1], t[ni]);
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) t[ni] = mfma(x[1], wp[ni][1], t[ni]);
            }
#pragma unroll
            for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float o = F::kMin ? fmaf(mv[ni], ts[r], acc[ni][r]) : acc[ni][r];
                    acc[ni][r] = fmaf(dv[ni], t[ni][r], o);
                }
        }
    };
    if (sb < se) {
        int s = sb;
        for (; s + 2 <= se; s += 2) {
            compute(s, s0);
            load(s + 2, s0);
            compute(s + 1, s1);
            load(s + 3, s1);
        }
        if (s < se) compute(s, s0);
    }

    // the waves' sums: lane holds rows 4 (lane / 16) + r of column l16
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave][ni][r][lane] = acc[ni][r];
    if (NORM) {
        double ss = 0.0;
#pragma unroll
        for (int i = 0; i < kSq; ++i) ss += tid / kPfSmallRows + i * kGroups < n_tiles ? sq[i] : 0.0;
        for (int t = tid / kPfSmallRows + kSq * kGroups; t < n_tiles; t += kGroups)
            ss += gptr(a.ssp)[(int64_t)t * kPfSmallRows + sq_row];
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        if (lane < kPfSmallRows) red_ss[wave][lane] = ss;
    }
    __syncthreads();
    // output o of this thread: row o / NC, column o % NC of the group
    float v[NV][MODE == GEMV_SILU ? 2 : 1];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int o = tid + i * kBlock;
        if (NOUT % (kBlock) != 0 && o >= NOUT) break;
        const int row = o / NC, cc = o % NC;
#pragma unroll
        for (int g = 0; g < (MODE == GEMV_SILU ? 2 : 1); ++g) {
            v[i][g] = 0.0f;
#pragma unroll
            for (int w = 0; w < W; ++w)
                v[i][g] += red[w][g * NT + cc / 16][row & 3][16 * (row >> 2) + cc % 16];
        }
    }
    if (MODE == GEMV_RESID && ks > 1) {
        float* part = a.part + (int64_t)grp * ks * NOUT;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int o = tid + i * kBlock;
            if (NOUT % (kBlock) != 0 && o >= NOUT) break;
            __hip_atomic_store(part + (int64_t)kslice * NOUT + o, v[i][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // written through before the count says so
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) {
            const int n = __hip_atomic_fetch_add(a.count + grp, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            arrived = n;
            // the last one leaves the count as the next launch expects it
            if (n == ks - 1) __hip_atomic_store(a.count + grp, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (arrived != ks - 1) return;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int o = tid + i * kBlock;
            if (NOUT % (kBlock) != 0 && o >= NOUT) break;
            float p[kPfSmallSlices];
#pragma unroll
            for (int k = 0; k < kPfSmallSlices; ++k)
                p[k] = __hip_atomic_load(part + (int64_t)(k < ks ? k : 0) * NOUT + o, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
            v[i][0] = 0.0f;
#pragma unroll
            for (int k = 0; k < kPfSmallSlices; ++k) v[i][0] += k < ks ? p[k] : 0.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int o = tid + i * kBlock;
        if (NOUT % (kBlock) != 0 && o >= NOUT) break;
        const int row = o / NC, cc = o % NC;
        if (row >= a.M) break;
        if (NORM) {
            double t = 0.0;
#pragma unroll
            for (int w = 0; w < W; ++w) t += red_ss[w][row];
            const float inv = 1.0f / sqrtf((float)(t / a.K) + a.eps);
#pragma unroll
            for (int g = 0; g < (MODE == GEMV_SILU ? 2 : 1); ++g) v[i][g] *= inv;
        }
        if (MODE == GEMV_SILU) {
            val[row][cc] = (v[i][0] / (1.0f + expf(-v[i][0]))) * v[i][MODE == GEMV_SILU ? 1 : 0];
        } else {
            float* p = SM_SEL(y) + (int64_t)row * SM_SEL(ldy) + col0 + cc;
            if (MODE == GEMV_STORE) {
                const float* bias = SM_SEL(bias);
                *p = bias ? v[i][0] + bias[col0 + cc] : v[i][0];
            } else {
                const float nv = yv[i] + v[i][0];
                *p = nv;
                if (row == a.tap_row && a.tap) a.tap[col0 + cc] = nv;
                val[row][cc] = nv;
            }
        }
    }
    if (MODE == GEMV_STORE || !a.oxa) return;
    __syncthreads();
    put_tile<NC>(val, tid, a.M, col0, a.onorm_w ? gl : nullptr, (b8_t*)a.oxa, a.ossp);
#undef SM_SEL
}

// A workgroup per query head: q, k and v of the M rows into LDS (q and k rotated with the
// fmaf pattern of the decode path, attention.cpp:31-46), k and v to the cache (the first query head
// of a kv head), then fp32 scores, softmax and P.V over the rows at or before each one.
template <int HD>
__global__ __launch_bounds__(kBlock) void k_pf_small_attn(const PfSmallAttn a) {
    constexpr int LD = HD + 4;  // padded rows: 16 rows' float4 reads spread over the banks
    constexpr int R = kPfSmallRows;
    __shared__ float qs[R][LD], ks[R][LD], vs[R][LD], ps[R][R + 1];
    const int h = blockIdx.x, n_rep = a.H / a.G, g = h / n_rep, tid = threadIdx.x, n = a.n;
    constexpr int D2 = HD / 2;
    for (int t = tid; t < n * D2; t += kBlock) {
        const int i = t / D2, j = t % D2;
        const float* row = a.qkv + (int64_t)i * a.ld;
        const float* q = row + h * HD;
        const float* k = row + (a.H + g) * HD;
        const float* v = row + (a.H + a.G + g) * HD;
        const int64_t ct = (int64_t)(a.pos0 + i) * D2 + j;
        const float c = a.rope_cos[ct], s = a.rope_sin[ct];
        const float q0 = q[j], q1 = q[j + D2], k0 = k[j], k1 = k[j + D2], v0 = v[j], v1 = v[j + D2];
        const float r0 = fmaf(k0, c, -(k1 * s)), r1 = fmaf(k0, s, k1 * c);
        qs[i][j] = fmaf(q0, c, -(q1 * s));
        qs[i][j + D2] = fmaf(q0, s, q1 * c);
        ks[i][j] = r0;
        ks[i][j + D2] = r1;
        vs[i][j] = v0;
        vs[i][j + D2] = v1;
        if (h % n_rep == 0) {
            const int64_t o = kv_offset(a.layout, a.G, a.max_seq, HD, g, a.pos0 + i);
            a.kc[o + j] = r0;
            a.kc[o + j + D2] = r1;
            a.vc[o + j] = v0;
            a.vc[o + j + D2] = v1;
        }
    }
    __syncthreads();
    const float scale = 1.0f / sqrtf((float)HD);
    for (int t = tid; t < n * n; t += kBlock) {
        const int i = t / n, j = t % n;
        if (j > i) continue;
        float s[4] = {0, 0, 0, 0};
#pragma unroll
        for (int d = 0; d < HD; d += 4) {
            const float4 x = *(const float4*)&qs[i][d], y = *(const float4*)&ks[j][d];
            s[0] = fmaf(x.x, y.x, s[0]);
            s[1] = fmaf(x.y, y.y, s[1]);
            s[2] = fmaf(x.z, y.z, s[2]);
            s[3] = fmaf(x.w, y.w, s[3]);
        }
        ps[i][j] = ((s[0] + s[1]) + (s[2] + s[3])) * scale;
    }
    __syncthreads();
    // P.V: thread (row i, 8 dims), each with its row's softmax (few keys, so every thread of a
    // row computes it: no more barriers), written as wo's operand
    for (int t = tid; t < n * (HD / 8); t += kBlock) {
        const int i = t / (HD / 8), d = t % (HD / 8) * 8;
        float m = ps[i][0];
        for (int j = 1; j <= i; ++j) m = fmaxf(m, ps[i][j]);
        float l = 0.0f, o[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int j = 0; j <= i; ++j) {
            const float p = expf(ps[i][j] - m);
            const float4 u = *(const float4*)&vs[j][d], v = *(const float4*)&vs[j][d + 4];
            l += p;
            o[0] = fmaf(p, u.x, o[0]);
            o[1] = fmaf(p, u.y, o[1]);
            o[2] = fmaf(p, u.z, o[2]);
            o[3] = fmaf(p, u.w, o[3]);
            o[4] = fmaf(p, v.x, o[4]);
            o[5] = fmaf(p, v.y, o[5]);
            o[6] = fmaf(p, v.z, o[6]);
            o[7] = fmaf(p, v.w, o[7]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = o[e] / l;
        put_pieces((b8_t*)a.oxa, n, i, (h * HD + d) / 8, o);
    }
}

template <int MODE, int T, int NT>
hipError_t launch_small_k(PfSmallArgs a, int ks, hipStream_t st) {
    using F = SmW<T>;
    constexpr int NI = MODE == GEMV_SILU ? 2 * NT : NT;
    a.ks = ks;
    const int S = (a.K / 32 + kStageBlocks - 1) / kStageBlocks, n_b = (S + ks - 1) / ks * kStageBlocks;
    size_t lds = (size_t)NI * 16 * (F::kScale * n_b / 4 + 1) * 4;  // the kernel's sc_lds and d_lds at the longest slice
    if (F::kSuper) lds += (size_t)NI * 16 * ((n_b / 8 + 2) / 2 + 2) * 4;
    static hipError_t attr = hipFuncSetAttribute((const void*)k_pf_small<MODE, T, NT>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
    if (attr != hipSuccess) return attr;
    if (lds > 80 * 1024) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_pf_small<MODE, T, NT>), dim3((unsigned)(a.n_sub / NT * ks)), dim3(kBlock), lds, st, a);
    return hipGetLastError();
}

// Column tiles a workgroup (NT) and K slices. One tile, four waves: two to four workgroups share
// a CU, so one streams while another reduces (eight waves of one tile are most of a CU's
// registers: Q8_0, 6 tokens of the Llama-3.2-1B shape 1,070 us against 1,035, 16 tokens of the
// Qwen2.5-1.5B shape, whose 560 gate / up tiles were two rounds, 2,095 against 1,750). wo and
// down have few tiles (128 for 2048 columns): pairs of tiles, which halve the reads of the
// operand, in K slices of at least 8 stages until every CU has a workgroup (no slices: 1,130 us).
template <int MODE, int T>
hipError_t launch_small_t(const PfSmallArgs& a, hipStream_t st) {
    if constexpr (MODE == GEMV_RESID) {
        const int cus = device_cu_count(), pairs = a.n_sub % 2 == 0 ? a.n_sub / 2 : 0;
        const int S = (a.K / 32 + kStageBlocks - 1) / kStageBlocks;
        if (a.part && pairs) {
            int ks = 1;
            while (ks < kPfSmallSlices && pairs * ks * 2 <= cus && S / (2 * ks) >= 8) ks *= 2;
            if (ks > 1) return launch_small_k<MODE, T, 2>(a, ks, st);
        }
    }
    return launch_small_k<MODE, T, 1>(a, 1, st);
}

template <int T>
hipError_t launch_small_m(const PfSmallArgs& a, hipStream_t st) {
    switch (a.mode) {
        case GEMV_STORE: return launch_small_t<GEMV_STORE, T>(a, st);
        case GEMV_RESID: return launch_small_t<GEMV_RESID, T>(a, st);
        case GEMV_SILU: return launch_small_t<GEMV_SILU, T>(a, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_pf_small(const PfSmallArgs& a, hipStream_t st) {
    if (a.K % 64 != 0 || a.M <= 0 || a.M > kPfSmallRows || a.n_sub <= 0 || a.n_seg < 1 || a.n_seg > 3 || !a.xa ||
        (a.mode != GEMV_RESID && !a.ssp) || (a.oxa && (a.n_seg != 1 || a.n_sub % 2 != 0)) || (a.onorm_w && !a.ossp) ||
        (a.mode == GEMV_SILU && !a.oxa) || (a.part && (!a.count || a.part_floats < kPfSmallPart((size_t)a.n_sub * 16))))
        return hipErrorInvalidValue;
    const int t = a.seg[0].w.type;
    for (int s = 0; s < a.n_seg; ++s) {
        const PfSeg& g = a.seg[s];
        const int next = s + 1 < a.n_seg ? a.seg[s + 1].sub0 : a.n_sub;
        if (!pf_gemm_supported(g.w.type, g.w.K, g.w.N) || g.w.type != t || g.w.K != a.K || (a.mode != GEMV_SILU && !g.y) ||
            next - g.sub0 != g.w.N / 16)
            return hipErrorInvalidValue;
        if (a.mode == GEMV_SILU && (g.w2.type != t || g.w2.K != a.K || g.w2.N != g.w.N)) return hipErrorInvalidValue;
    }
    if (a.seg[0].sub0 != 0 || (a.mode == GEMV_SILU && a.n_seg != 1)) return hipErrorInvalidValue;
    switch (t) {
        case TF_HIP_TYPE_Q8_0: return launch_small_m<TF_HIP_TYPE_Q8_0>(a, st);
        case TF_HIP_TYPE_Q4_0: return launch_small_m<TF_HIP_TYPE_Q4_0>(a, st);
        case TF_HIP_TYPE_Q4_1: return launch_small_m<TF_HIP_TYPE_Q4_1>(a, st);
        case TF_HIP_TYPE_F16: return launch_small_m<TF_HIP_TYPE_F16>(a, st);
        case TF_HIP_TYPE_Q6_K: return launch_small_m<TF_HIP_TYPE_Q6_K>(a, st);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_pf_small_split(const float* x, int D, int M, const float* norm_w, uint16_t* xa, double* ssp,
                                 hipStream_t st) {
    if (D % 32 != 0 || M <= 0 || M > kPfSmallRows || !norm_w) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(D / 16));
    hipLaunchKernelGGL(k_pf_small_split, grid, dim3(kBlock), 0, st, x, D, M, norm_w, (b8_t*)xa, ssp);
    return hipGetLastError();
}

hipError_t launch_pf_small_attn(const PfSmallAttn& a, int hd, hipStream_t st) {
    if (a.n <= 0 || a.n > kPfSmallRows || a.G <= 0 || a.H % a.G != 0 || a.pos0 < 0 || a.pos0 + a.n > a.max_seq)
        return hipErrorInvalidValue;
    const dim3 grid((unsigned)a.H);
    switch (hd) {
        case 32: hipLaunchKernelGGL(k_pf_small_attn<32>, grid, dim3(kBlock), 0, st, a); break;
        case 64: hipLaunchKernelGGL(k_pf_small_attn<64>, grid, dim3(kBlock), 0, st, a); break;
        case 128: hipLaunchKernelGGL(k_pf_small_attn<128>, grid, dim3(kBlock), 0, st, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace tfk
