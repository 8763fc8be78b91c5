// Ternary prefill GEMM on the 6/4-bit matrix instructions: bn_ternary_matmul with T > 32 (model.rs:455-596 qmm_lora /
// qmm_multi over a prompt; kernels/qmm3.comp).
//
// v_mfma_scale_f32_32x32x64_f8f6f4 multiplies fp6 by fp4 at four times the fp16 rate (measured on MI355X: 6.8 against
// 1.7-1.9 PFLOP/s). Both operands here are exact in those formats:
//   W: a code c becomes the fp4 value 2 (c - 1) in {-2, 0, 2, 4}; the row's fp16 scale multiplies the sum of each
//      128-column group in fp32 afterwards (as qmv.glsl:22-35 does), one fma per output and group.
//   x: 32 columns of a token share the power of two S = 2^floor(log2(max |x|)), and x is written as five fp6 (e2m3)
//      digits, x = S / 2 (q0 + q1 / 32 + ... + q4 / 32^4), each the fp6 value nearest to what the digits before it left
//      (|q| <= 4, in steps of 1/8 up to 2 and of 1/4 above: exact differences), to within S 2^-25 for most values and
//      S 2^-24 for all: fp32's own last bit for the block's largest. The digit's power of two is the instruction's block
//      scale, so one fp32 accumulator takes all five (smallest first), and a group's products are summed without a
//      rounding between its columns' scales.
//   Five MFMAs per 64 columns thus replace the eight of an fp16 hi/lo split, at the same time each.
// Digits end at the same place for all 32 values, so columns far below a block's largest keep fewer bits of their own,
// which a row whose weights are 0 on the large columns shows. Such a block's remainder is written as five more digits and
// multiplied by a second pass over the group (flagged per 32-token tile; blocks that need none are zero there). It is
// made where the digits of at least 12 of the block's columns within S 2^-5, or of 6 within S 2^-7.7, do not end: with up
// to 25 large columns of 32 the others' error is then at most 2.3e-6 of their norm (worst of factors 8 to 10^5 between
// them, weights 0 under the large ones; the digits alone: 3e-3, which fewer small columns keep). The rules are no wider
// because a step with a second pass takes more than twice as long, and the blocks of a call that runs in one round wait
// for it: they take 1e-7 of the blocks of normally distributed values for such (with 2e-5 of them calls of 1,000 to 2,000
// tokens took 10-20% longer; a column that is small in all tokens of a tile says nothing, as tokens may be alike). The
// block scale covers fp32's exponents; a block with an infinity or a NaN gets the scale NaN, and the token's outputs are
// NaN.
// Measured (MI355X, the 4B q/k/v projections of 4,096 tokens): 303 us (digits 17, GEMM 285) against 368 for the fp16
// hi/lo split, whose 1.16 PFLOP/s of products were the rate of a large library product here; error against 64-bit sums
// 0.9e-7 of the output's norm against 4.6e-7. The matrix units are busy two thirds of the time at the 1.7 GHz that the
// power limit leaves (a loop of these MFMAs alone: 1.63 GHz, 157 us for this call's); without the copies the call took
// 254 us, without the output stores 20 less, and neither another order of the loop nor more stages changed it.
//
// Fragment order. MFMA half kh of a group and lane (r = lane % 32, h = lane / 32) hold columns 64 h + 32 kh .. + 31,
// which are code words 4 h + 2 kh, + 1 of the row: 16 bytes of codes per lane and group. Element e of the 32 is column
// 16 (e / 8 / 2) + 2 (e % 8) + (e / 8) % 2: a word's even codes, then its odd ones, as the decode leaves them.
//
// tern_digits_kernel writes x's digits once per call as the tiles the GEMM reads (15 KB per 32 tokens and group);
// tern_mx_kernel<W, MT, KS, NS> multiplies: NS = 0 copies those tiles into LDS, NS = 2 or 3 (no workspace) brings x itself
// into as many stages of LDS and makes the same digits there. All run the same products in the same order: identical
// results.
#pragma once
#include "bn_ternary.h"

namespace bn {

typedef int i8v __attribute__((ext_vector_type(8)));
typedef uint32_t u6v __attribute__((ext_vector_type(6)));
typedef float f32v __attribute__((ext_vector_type(32)));

constexpr int TMX_G = 128;                      // columns per group (one weight scale)
constexpr int TMX_ND = 5;                       // digits
constexpr int TMX_FRAG = 64 * 48;               // bytes of a digit: per lane 12 words (kh = 0, then 1) in three 1 KB planes
constexpr int TMX_DIG = TMX_ND * TMX_FRAG;      // 15,360
// a 32-token tile of a group: fragments, then per lane the scale bytes of its two blocks and whether each is wide
constexpr int TMX_TILE = TMX_DIG + 256;

// 32-token tiles of a call (an even number: the blocks take two)
__host__ __device__ inline int tern_mx_tiles(int T) { return 2 * ((T + 63) / 64); }
// Workspace bytes: per 64 tokens and 64 columns 16 KB and a word (the tiles and flags take 15,620 of the 16,388)
inline size_t tern_pf_work_bytes(int T, int K) {
    return (size_t)((T + 63) / 64) * (size_t)(K / 64) * (16384 + 4);
}
static_assert(2 * (TMX_TILE + 4) <= 2 * (16384 + 4), "the workspace holds the tiles and their flags");

struct TernBlock {
    f16x u, v;  // 32 values of a token by element: u[i] = element 2 i, v[i] = element 2 i + 1
};
__device__ __forceinline__ float tern_pow2(int e) { return __int_as_float(e << 23); }
// word i of 16 six-bit fields of value f in three words
__host__ __device__ constexpr uint32_t tern_fields(uint32_t f, int i) {
    uint32_t r = 0;
    for (int j = 0; j < 16; ++j) {
        const int at = 6 * j - 32 * i;
        if (at > -6 && at < 32) r |= at >= 0 ? f << at : f >> -at;
    }
    return r;
}
// Which of a digit's 32 values are at least Q eighths: a code's magnitude (6 bits: sign, magnitude) plus 32 - Q carries
// into the sign's place if it is. The 16 such places of three words fall on distinct odd bits: bit tern_bit(e) of the
// result is element e.
template <int Q>
__device__ __forceinline__ uint32_t tern_at_least(u6v w) {
    uint32_t r[2] = {0, 0};
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        uint32_t carry = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            r[half] |= __builtin_addc(w[3 * half + i] & tern_fields(31, i), tern_fields(32 - Q, i), carry, &carry) &
                       tern_fields(32, i);
    }
    return r[0] | (r[1] >> 1);
}
__host__ __device__ constexpr int tern_bit(int e) { return (6 * (e & 15) + 5) % 32 - (e >> 4); }
// The digits of 32 values x of a token: each digit's six words through put(d, words). Returns the block's scale byte.
// CHECK = false: x becomes the remainders. CHECK = true: only where some block of the wave may need a second set of
// digits; tells in wide whether this one does.
template <bool CHECK, typename Put>
__device__ __forceinline__ int tern_digits(TernBlock& x, bool& wide, const Put& put) {
    float mx = 0.0f;  // an infinity or a NaN stays
#pragma unroll
    for (int i = 0; i < 16; ++i) asm("v_maximum3_f32 %0, |%1|, |%2|, %0" : "+v"(mx) : "v"(x.u[i]), "v"(x.v[i]));
    const int eb = (__float_as_int(mx) >> 23) & 255;
    const int e = max(eb - 1, 28);  // 28: the last digit's scale stays normal
    // columns above S 2^-5, above S 2^-7.7: by the first two digits
    uint32_t over[2];
    bool ask = false;
#pragma unroll
    for (int d = 0; d < TMX_ND; ++d) {
        const float sc = tern_pow2(e - 5 * d);
        const u6v q = __builtin_bit_cast(u6v, __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(x.u, x.v, sc));
        put(d, q);
        if (CHECK && d == 0) over[0] = tern_at_least<1>(q);
        if (CHECK && d == 1) {
            over[1] = over[0] | tern_at_least<3>(q);
            ask = mx != 0.0f && (__builtin_popcount(over[0]) <= 32 - 12 || __builtin_popcount(over[1]) <= 32 - 6);
        }
        if (CHECK && d == TMX_ND - 1 && __ballot(ask) == 0) break;
        const f32v b = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(q, sc);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            x.u[i] -= b[2 * i];
            x.v[i] -= b[2 * i + 1];
        }
    }
    if constexpr (CHECK) {
        wide = false;
        if (__ballot(ask) != 0) {
            // rare: of these columns, those whose digits do not end
            uint32_t rest = 0;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                rest |= x.u[i] != 0.0f ? 1u << tern_bit(2 * i) : 0u;
                rest |= x.v[i] != 0.0f ? 1u << tern_bit(2 * i + 1) : 0u;
            }
            wide = __builtin_popcount(rest & ~over[0]) >= 12 || __builtin_popcount(rest & ~over[1]) >= 6;
        }
    }
    return eb == 255 ? 255 : e;
}
// element e of the fragment order: its column in the 32
__host__ __device__ constexpr int tern_mx_col(int e) { return 16 * (e >> 4) + 2 * (e & 7) + ((e >> 3) & 1); }
// 32 floats, 16 bytes at a time through ld(i) (floats 4 i .. 4 i + 3), in element order
template <typename Ld>
__device__ __forceinline__ void tern_block_load(TernBlock& x, const Ld& ld) {
    f4 c[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) c[i] = ld(i);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int a = tern_mx_col(2 * i), b = tern_mx_col(2 * i + 1);
        x.u[i] = c[a >> 2][a & 3];
        x.v[i] = c[b >> 2][b & 3];
    }
}
// digit d's six words of (lane, kh) into a tile at p (global memory or LDS): words 6 kh .. of the lane's 12, four of
// them in each 1 KB plane, so that a lane reads both halves' operands in three 16-byte reads. kh: the same for a wave
// (the words are selected by a branch, not by six selects).
__device__ __forceinline__ void tern_mx_put(uint8_t* p, int kh, int d, int lane, u6v q) {
    uint8_t* f = p + d * TMX_FRAG + 16 * lane;
    if (kh) {
        *reinterpret_cast<u2*>(f + 1024 + 8) = u2{q[0], q[1]};
        *reinterpret_cast<u4*>(f + 2048) = u4{q[2], q[3], q[4], q[5]};
    } else {
        *reinterpret_cast<u4*>(f) = u4{q[0], q[1], q[2], q[3]};
        *reinterpret_cast<u2*>(f + 1024) = u2{q[4], q[5]};
    }
}
// A tile made in its block's LDS: 8 KB per kh, which hold the 64 columns of x (32 tokens) that the digits come from until
// the wave has read them. Per digit words 0..3 of a lane, then words 4, 5; the blocks' scale bytes; whether each is wide;
// a word, whether any is.
constexpr int TMX_RAW = 8192, TMX_RDIG = 64 * 24, TMX_RSCALE = TMX_ND * TMX_RDIG, TMX_RANY = TMX_RSCALE + 128;

typedef __attribute__((address_space(3))) void tmx_lds_t;
// 16 (4) bytes per lane from global memory into LDS at lds + 16 lane (4 lane)
__device__ __forceinline__ void tmx_copy16(const void* g, const uint8_t* lds) {
    __builtin_amdgcn_global_load_lds(g, (tmx_lds_t*)const_cast<uint8_t*>(lds), 16, 0, 0);
}
__device__ __forceinline__ void tmx_copy4(const void* g, const uint8_t* lds) {
    __builtin_amdgcn_global_load_lds(g, (tmx_lds_t*)const_cast<uint8_t*>(lds), 4, 0, 0);
}

// x's digits: one block per 64 tokens and group; work: [tile][group] TMX_TILE bytes, then a flag word each. The rows
// come through LDS (a copy moves 512 contiguous bytes of two tokens; a thread then takes 32 columns of one token):
// read straight into registers, a wave would touch 64 lines per load. Tokens past T get zeros.
__global__ __launch_bounds__(256, 4) void tern_digits_kernel(const float* __restrict__ x, int64_t x_ts, int T, int K,
                                                          uint8_t* __restrict__ work) {
    constexpr int PAIR = 1040;  // LDS pitch of two tokens' 512 bytes
    __shared__ __attribute__((aligned(16))) uint8_t rows[32 * PAIR];
    const int ng = K / TMX_G;
    const int tt = (int)blockIdx.x / ng, g = (int)blockIdx.x - tt * ng, t0 = 64 * tt;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        // an odd token's 16-byte chunks are swapped in blocks of 8, so that 16 tokens' reads fall on distinct banks
        const int p = 8 * wave + i, odd = lane >> 5, t = min(t0 + 2 * p + odd, T - 1);
        tmx_copy16(x + (int64_t)t * x_ts + g * TMX_G + 4 * ((lane & 31) ^ (8 * odd)), rows + p * PAIR);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // wave: tile wave / 2, MFMA half kh = wave % 2; lane: token lane % 32, lane half h = lane / 32 of its fragments
    const int u = wave >> 1, kh = wave & 1, m = lane & 31, b = 2 * (lane >> 5) + kh;
    const int tile = 2 * tt + u;
    uint8_t* out = work + ((size_t)tile * ng + g) * TMX_TILE;
    TernBlock v;
    const uint8_t* src = rows + (16 * u + (m >> 1)) * PAIR + 512 * (m & 1);
    tern_block_load(v, [&](int i) { return *reinterpret_cast<const f4*>(src + 16 * ((8 * b + i) ^ (8 * (m & 1)))); });
    if (t0 + 32 * u + m >= T) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v.u[i] = v.v[i] = 0.0f;
    }
    bool wide;
    const int e = tern_digits<true>(v, wide, [&](int d, u6v q) { tern_mx_put(out, kh, d, lane, q); });
    out[TMX_DIG + 4 * lane + kh] = (uint8_t)e;
    out[TMX_DIG + 4 * lane + 2 + kh] = wide;
    __shared__ int wide_lds[4];
    const bool any = __ballot(wide) != 0;
    if (lane == 0) wide_lds[wave] = any;
    __syncthreads();
    if (threadIdx.x < 2) {
        uint32_t* flags = reinterpret_cast<uint32_t*>(work + (size_t)tern_mx_tiles(T) * ng * TMX_TILE);
        flags[(size_t)(2 * tt + threadIdx.x) * ng + g] = wide_lds[2 * threadIdx.x] | wide_lds[2 * threadIdx.x + 1];
    }
}

// 32 codes (two words) as fp4 values 2 (c - 1): bit 3 = !b1, bit 2 = !b0 | b1, bit 1 = b0 & b1 of the code's bits;
// words 0, 1: the even and the odd codes of w0, 2, 3: of w1
__device__ __forceinline__ void tern_fp4(uint32_t w, int& even, int& odd) {
    const uint32_t v = w >> 1, n = ~w | (v & 0x55555555u);
    uint32_t q = w & v & 0x55555555u;
    asm("" : "+v"(q));  // the selects below stay v_bfi_b32 (knowing q's zero bits, the compiler masks and ors instead)
    even = (int)(((n << 2) & 0xCCCCCCCCu) | ((q << 1) & ~0xCCCCCCCCu));
    odd = (int)((n & 0xCCCCCCCCu) | ((q >> 1) & ~0xCCCCCCCCu));
}

// copies of fragments per wave and group of columns (1 KB each, the last repeated where they do not divide)
__host__ __device__ constexpr int tmx_frag_copies(int W, int MT) { return (15 * MT + W - 1) / W; }

// KS wave groups of W waves x 64 rows, 32 MT tokens; the groups split the columns and add their sums at the end, in
// order. Per 128 columns a wave multiplies MT token tiles x 2 row tiles x 2 halves x 5 digits (32 cycles each) into a
// fresh accumulator per tile pair, which one fma per output adds, times the row scale, to the running sums. One barrier
// per step. NS = 0 (PRE): x's digits come from tern_digits_kernel's tiles; two stages in LDS, the next step's copies in
// flight during a step's products. NS = 2: x comes instead, and the next step's digits are made from it after the products.
// NS = 3: x comes two steps ahead, and with twice the waves that a stage's tiles take, half of the waves make the next
// step's digits while the others multiply, turn about (8 waves x 64 rows, 4B q/k/v of 4,096 tokens: 355 us; with two
// stages 371, and 392 with x read by token and block, where each load touches 64 places; the copies' addresses and the
// digits are vector work, two thirds of a step's as long as 256 rows share it).
template <int W, int MT, int KS, int NS>
__global__ __launch_bounds__(64 * W * KS, 2) void tern_mx_kernel(TernArgs a, int row_tiles,
                                                                 const uint8_t* __restrict__ work) {
    constexpr bool PRE = NS == 0;
    static_assert(MT == 1 || MT == 2, "token tiles per block (x's tiles come in pairs)");
    // a stage of a wave group: its MT x tiles, then the waves' codes (64 rows x 32 bytes each)
    constexpr int TILE = PRE ? TMX_TILE : 2 * TMX_RAW, BM = 32 * MT, ST_W = MT * TILE, STAGE = ST_W + W * 2048;
    // separate arrays, so that the compiler can tell one stage's copies from another's reads (PRE = false: pf_copy16's)
    __shared__ __attribute__((aligned(1024))) uint8_t lds0[(PRE ? 1 : NS) * KS * STAGE];
    __shared__ __attribute__((aligned(1024))) uint8_t lds1[PRE ? KS * STAGE : 1];
    static_assert(KS == 1 || (KS - 1) * W * MT * 8192 <= KS * STAGE, "the groups' sums fit a stage");
    const int lane = (int)threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), ks = wv / W, wave = wv % W;
    const int n = lane & 31, h = lane >> 5;
    int rt, tt;
    tern_tile<BM, (BN_TERN_XCD_GROUP * 64 / BM > 0 ? BN_TERN_XCD_GROUP * 64 / BM : 1)>((int)blockIdx.x, row_tiles, a.T, rt, tt);
    const int t0 = tt * BM;
    const int rbase_g = (rt * W + wave) * 64;  // first global row of this wave
    const bool active = rbase_g < a.rows;
    int rbase = active ? rbase_g : 0;          // inactive waves take member 0's first rows (in bounds, not stored)
    const int mi = tern_member(a, rbase);
    const TernMat m = tern_mat(a, mi);
    const int K = a.K, kw = K >> 4, ng = K / TMX_G;
    // the wave group's 128-column groups [g0, g0 + cnt); a step past cnt repeats a group's copies, unused
    const int g0 = ks * ng / KS, cnt = (ks + 1) * ng / KS - g0, steps = (ng + KS - 1) / KS;
    int cnt_ = cnt;
    asm("" : "+s"(cnt_));
    auto group = [&](int j) { return min(g0 + min(j, cnt - 1 > 0 ? cnt - 1 : 0), ng - 1); };
    const int ntiles = tern_mx_tiles(a.T);
    const size_t xt = (size_t)MT * tt;  // the block's first x tile
    const size_t tile_row = (size_t)ng * TMX_TILE;
    const uint8_t* tiles = work + xt * tile_row;
    const uint32_t* flags = reinterpret_cast<const uint32_t*>(work + ntiles * tile_row) + xt * ng;
    // A copy of row tile nt's codes takes a row's two 16-byte halves with neighbouring lanes (a load of 64 separate
    // places costs the address unit 64 cycles, and these loads bound small calls): lane -> row lane / 2, half
    // lane % 2, the halves swapped in every other 8 rows so that the operand reads fall on distinct banks
    const int cr = lane >> 1, ch = (lane & 1) ^ ((cr >> 3) & 1);
    const uint8_t* wsrc = reinterpret_cast<const uint8_t*>(m.w + (int64_t)(rbase + cr) * kw) + 16 * ch;
    const int64_t wtile = (int64_t)32 * kw * 4;
    const int w_lane = wave * 2048 + 32 * n + 16 * (h ^ ((n >> 3) & 1));
    // scales of rows n, 32 + n: four groups' at a time where they lie on 8 bytes (for the same reason), else one
    const bool s4 = (ng & 3) == 0 && ((uintptr_t)m.s & 7) == 0;
    const uint16_t* ssrc = m.s + (int64_t)(rbase + n) * ng;
    uint64_t sw[2];
    auto load_s = [&](int g) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const uint16_t* p = ssrc + (int64_t)32 * nt * ng + g;
            if (s4)
                sw[nt] = *reinterpret_cast<const uint64_t*>(p - (g & 3));
            else
                sw[nt] = *p;
        }
    };
    // PRE = false: the waves that make a stage's tiles, a wave per tile and kh; with waves to spare, others for each stage
    // (mk: the wave's tile and kh). A maker copies 32 tokens x 64 columns in pieces of 128 contiguous bytes (read by token
    // and block, each load would touch 64 places), copy i rows 4 i + lane / 16; a row's 16-byte chunks are swapped by its
    // number, so that 16 tokens' reads below fall on distinct banks: four addresses per lane serve the 8 copies. Rows past
    // T read the lane's first row, if that is past T the last.
    constexpr int MK = 2 * MT, MK_S = 2 * MK <= W ? 2 : 1;
    const int mk = wave % MK, tx = t0 + 32 * (mk >> 1);
    auto makes = [&](int s) { return wave / MK == s % MK_S; };
    const uint8_t* xp[PRE ? 1 : 4];
    if constexpr (!PRE) {
        const int q = lane >> 4, c = (lane & 15) ^ q;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            xp[k] = reinterpret_cast<const uint8_t*>(a.x + (int64_t)min(tx + q, a.T - 1) * a.x_ts + 32 * (mk & 1)) +
                    ((256 * (c >> 3) + 16 * (c & 7)) ^ (64 * (k & 1)) ^ (256 * (k >> 1)));
    }
    // the copies of column group g into a stage (s: its number)
    auto issue = [&](int g, const uint8_t* sb, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            if constexpr (PRE) tmx_copy16(wsrc + nt * wtile + 32 * g, sb + ST_W + wave * 2048 + nt * 1024);
            else pf_copy16(wsrc + nt * wtile + 32 * g, sb + ST_W + wave * 2048 + nt * 1024);
        }
        if constexpr (PRE) {
            constexpr int C = tmx_frag_copies(W, MT);
#pragma unroll
            for (int i = 0; i < C; ++i) {
                const int f = min(wave * C + i, 15 * MT - 1), u = f / 15, o = (f - 15 * u) * 1024;
                tmx_copy16(tiles + u * tile_row + (size_t)g * TMX_TILE + o + 16 * lane, sb + u * TMX_TILE + o);
            }
            const int u = wave & (MT - 1);
            tmx_copy4(tiles + u * tile_row + (size_t)g * TMX_TILE + TMX_DIG + 4 * lane, sb + u * TMX_TILE + TMX_DIG);
        } else if (makes(s)) {
            const int64_t gb = (int64_t)g * TMX_G * 4, row4 = a.x_ts * 16;
            if (tx + 32 <= a.T) {
#pragma unroll
                for (int i = 0; i < 8; ++i) pf_copy16(xp[i & 3] + (gb + i * row4), sb + mk * TMX_RAW + i * 1024);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    pf_copy16(xp[i & 3] + gb + (tx + 4 * i + (lane >> 4) < a.T ? i * row4 : 0),
                              sb + mk * TMX_RAW + i * 1024);
            }
        }
    };
    // PRE = false: a maker's columns of x, copied into a stage, as digits in their place (each lane's reads come before the
    // wave's first write)
    auto make_tiles = [&](uint8_t* sb, int s) __attribute__((always_inline)) {
        if (!makes(s)) return;
        if (NS == 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint8_t* dst = sb + mk * TMX_RAW;
        const int xm = lane & 31;
        TernBlock v;
        tern_block_load(v, [&](int c) {
            return *reinterpret_cast<const f4*>(dst + 256 * xm + 16 * ((8 * (lane >> 5) + c) ^ (xm & 15)));
        });
        if (tx + xm >= a.T) {
#pragma unroll
            for (int c = 0; c < 16; ++c) v.u[c] = v.v[c] = 0.0f;
        }
        bool wide;
        const int e = tern_digits<true>(v, wide, [&](int d, u6v q) {
            *reinterpret_cast<u4*>(dst + d * TMX_RDIG + 16 * lane) = u4{q[0], q[1], q[2], q[3]};
            *reinterpret_cast<u2*>(dst + d * TMX_RDIG + 1024 + 8 * lane) = u2{q[4], q[5]};
        });
        dst[TMX_RSCALE + lane] = (uint8_t)e;
        dst[TMX_RSCALE + 64 + lane] = wide;
        const bool any = __ballot(wide) != 0;
        if (lane == 0) *reinterpret_cast<int*>(dst + TMX_RANY) = any;
    };
    // the second pass: the remainders' digits in the tiles' place, zeros for blocks that need none
    auto make_second = [&](int g, uint8_t* sb) __attribute__((always_inline)) {
        if (wave >= MK) return;
        const int kh = wave & 1, xm = lane & 31, xtok = t0 + 32 * (wave >> 1) + xm;
        TernBlock v;
        const float* p = a.x + (int64_t)min(xtok, a.T - 1) * a.x_ts + g * TMX_G + 64 * (lane >> 5) + 32 * kh;
        tern_block_load(v, [&](int c) { return reinterpret_cast<const f4*>(p)[c]; });
        uint8_t* dst = PRE ? sb + (wave >> 1) * TMX_TILE : sb + wave * TMX_RAW;
        uint8_t* sp = PRE ? dst + TMX_DIG + 4 * lane + kh : dst + TMX_RSCALE + lane;
        const bool drop = sp[PRE ? 2 : 64] == 0;
        bool none;
        int e = 0;
#pragma unroll 1
        for (int pass = 0; pass < 2; ++pass) {
            e = tern_digits<false>(v, none, [&](int d, u6v q) {
                if constexpr (PRE) {
                    tern_mx_put(dst, kh, d, lane, q);
                } else {
                    *reinterpret_cast<u4*>(dst + d * TMX_RDIG + 16 * lane) = u4{q[0], q[1], q[2], q[3]};
                    *reinterpret_cast<u2*>(dst + d * TMX_RDIG + 1024 + 8 * lane) = u2{q[4], q[5]};
                }
            });
            if (drop) {
#pragma unroll
                for (int c = 0; c < 16; ++c) v.u[c] = v.v[c] = 0.0f;
            }
        }
        *sp = (uint8_t)e;
    };
    static_assert(MK <= W, "a thread per 32 columns of a token");

    f16x acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][nt][e] = 0.0f;

    // the digits' powers of two, 2^(-5 d) / 2: fp4 weights are twice c - 1
    const int sw0 = 126 | (121 << 8) | (116 << 16) | (111 << 24), sw1 = 106;
    // the products of a group: codes decoded, then per token tile five digits x two halves, smallest digit first
    auto products = [&](const uint8_t* sb, const float (&sc)[2]) __attribute__((always_inline)) {
        i8v b[2][2];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const u4 wc = *reinterpret_cast<const u4*>(sb + ST_W + w_lane + nt * 1024);
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) {
                int w0, w1, w2, w3;
                tern_fp4(wc[2 * kh], w0, w1);
                tern_fp4(wc[2 * kh + 1], w2, w3);
                b[nt][kh] = i8v{w0, w1, w2, w3, 0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const uint8_t* xl = sb + i * TILE;
            int ex, ex1;  // the blocks' scales: bytes 0 and 1 of ex, or byte 0 of each
            if constexpr (PRE) {
                ex = *reinterpret_cast<const int*>(xl + TMX_DIG + 4 * lane);
            } else {
                ex = xl[TMX_RSCALE + lane];
                ex1 = xl[TMX_RAW + TMX_RSCALE + lane];
            }
            f16x t[2];
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int e = 0; e < 16; ++e) t[nt][e] = 0.0f;
#pragma unroll
            for (int d = TMX_ND - 1; d >= 0; --d) {
                i8v x0, x1;
                if constexpr (PRE) {
                    const u4* f = reinterpret_cast<const u4*>(xl + d * TMX_FRAG + 16 * lane);
                    const u4 w0 = f[0], w1 = f[64], w2 = f[128];
                    x0 = i8v{(int)w0[0], (int)w0[1], (int)w0[2], (int)w0[3], (int)w1[0], (int)w1[1], 0, 0};
                    x1 = i8v{(int)w1[2], (int)w1[3], (int)w2[0], (int)w2[1], (int)w2[2], (int)w2[3], 0, 0};
                } else {
                    auto half = [&](const uint8_t* f) {
                        const u4 w0 = *reinterpret_cast<const u4*>(f + 16 * lane);
                        const u2 w1 = *reinterpret_cast<const u2*>(f + 1024 + 8 * lane);
                        return i8v{(int)w0[0], (int)w0[1], (int)w0[2], (int)w0[3], (int)w1[0], (int)w1[1], 0, 0};
                    };
                    x0 = half(xl + d * TMX_RDIG);
                    x1 = half(xl + TMX_RAW + d * TMX_RDIG);
                }
                // the scale operands' byte selects are immediates: one call per digit
#define TMX_MFMA(DD, SW)                                                                                        \
    for (int nt = 0; nt < 2; ++nt)                                                                              \
        t[nt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x0, b[nt][0], t[nt], 2, 4, 0, ex, DD, SW);      \
    for (int nt = 0; nt < 2; ++nt)                                                                              \
        t[nt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x1, b[nt][1], t[nt], 2, 4, PRE ? 1 : 0,         \
                                                                PRE ? ex : ex1, DD, SW)
                if (d == 4) { TMX_MFMA(0, sw1); }
                if (d == 3) { TMX_MFMA(3, sw0); }
                if (d == 2) { TMX_MFMA(2, sw0); }
                if (d == 1) { TMX_MFMA(1, sw0); }
                if (d == 0) { TMX_MFMA(0, sw0); }
#undef TMX_MFMA
            }
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][nt][e] = fmaf(t[nt][e], sc[nt], acc[i][nt][e]);
        }
    };

    // whether some group of the block's tiles needs a second pass, read before the copies
    bool block_wide = false;
    if constexpr (PRE) {
        uint32_t f = 0;
        for (int g = lane; g < ng; g += 64)
#pragma unroll
            for (int u = 0; u < MT; ++u) f |= flags[(size_t)u * ng + g];
        block_wide = __ballot(f != 0) != 0;
    }
    load_s(group(0));
    // step j from stage sb while a later step is brought into nb (PRE: the next; in place: the next of NS = 2 stages, the
    // one after of 3, whose x the next step's digits are made from before the products)
    auto step = [&](int j, uint8_t* sb, uint8_t* mb, uint8_t* nb) __attribute__((always_inline)) {
        // this step's copies of every wave have landed, and every wave is done with nb
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int g = group(j), gn = group(j + 1);
        float sc[2];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            asm volatile("" : "+v"(sw[nt]));  // the compiler's wait for this load ends here, before the next copies
            sc[nt] = h2f((uint16_t)(sw[nt] >> (s4 ? 16 * (g & 3) : 0)));
        }
        if (!s4 || (gn & 3) == 0) load_s(gn);
        bool wide = false;  // the same for every wave of the block
        if constexpr (PRE) {
            if (block_wide) {
#pragma unroll
                for (int q = 0; q < KS; ++q) {
                    const int q0 = q * ng / KS, gq = min(q0 + j, max((q + 1) * ng / KS - 1, 0));
#pragma unroll
                    for (int u = 0; u < MT; ++u) wide |= flags[(size_t)u * ng + gq] != 0;
                }
            }
        } else {
            const uint8_t* sb0 = sb - ks * STAGE;
#pragma unroll
            for (int q = 0; q < KS; ++q)
#pragma unroll
                for (int k = 0; k < MK; ++k)
                    wide |= *reinterpret_cast<const int*>(sb0 + q * STAGE + k * TMX_RAW + TMX_RANY) != 0;
            wide = __builtin_amdgcn_readfirstlane(wide);
        }
        if constexpr (PRE || NS == 2) issue(gn, nb, j + 1);
        else issue(group(j + 2), nb, j + 2);
        if constexpr (NS == 3) {
            if (j + 1 < steps) make_tiles(mb, j + 1);
        }
        // PRE = false always branches here (in one piece with the digits below, the compiler spills registers)
        if ((KS == 1 && PRE) || j < cnt_) products(sb, sc);
        if constexpr (NS == 2) {
            if (j + 1 < steps) make_tiles(nb, j + 1);
        }
        if (wide) {
            // rare: the remainders of the blocks that need them take the tiles' place
            __syncthreads();
            make_second(g, sb);
            __syncthreads();
            if (KS == 1 || j < cnt) products(sb, sc);
        }
    };
    if constexpr (PRE) {
        uint8_t* const st0 = lds0 + ks * STAGE;
        uint8_t* const st1 = lds1 + ks * STAGE;
        issue(group(0), st0, 0);
        for (int j = 0; j < steps; j += 2) {
            step(j, st0, nullptr, st1);
            if (j + 1 < steps) step(j + 1, st1, nullptr, st0);
        }
    } else {
        uint8_t* s0 = lds0 + ks * STAGE;
        uint8_t* s1 = s0 + KS * STAGE;
        uint8_t* s2 = NS == 3 ? s1 + KS * STAGE : s0;
        issue(group(0), s0, 0);
        if (NS == 3) issue(group(1), s1, 1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        make_tiles(s0, 0);
#pragma unroll 1
        for (int j = 0; j < steps; ++j) {
            step(j, s0, s1, NS == 3 ? s2 : s1);
            uint8_t* const t = s0;
            s0 = s1;
            s1 = NS == 3 ? s2 : t;
            s2 = t;
        }
    }
    // the last copies (repeats into free stages) land before the block's LDS is reused or released
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    if constexpr (KS > 1) {
        // the groups' sums, added in group order by the first group's waves
        float* red = reinterpret_cast<float*>(lds0);
        __syncthreads();
        auto slot = [&](int q, int i, int nt, int e) { return ((((q * W + wave) * MT + i) * 2 + nt) * 16 + e) * 64 + lane; };
        if (ks > 0)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) red[slot(ks - 1, i, nt, e)] = acc[i][nt][e];
        __syncthreads();
        if (ks > 0) return;
#pragma unroll
        for (int q = 0; q < KS - 1; ++q)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][nt][e] += red[slot(q, i, nt, e)];
    }
    // C layout: acc[i][nt][j] = (token 32 i + 8 (j / 4) + 4 h + j % 4, row 32 nt + n)
    if (!active) return;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int t = t0 + 32 * i + 8 * (j >> 2) + 4 * h + (j & 3);
            if (t < a.T)
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) tern_store(a, m, mi, t, rbase + 32 * nt + n, acc[i][nt][j]);
        }
}

}  // namespace bn
