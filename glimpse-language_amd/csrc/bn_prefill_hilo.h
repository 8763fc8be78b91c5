// Causal GQA prefill for long prompts whose query rows come as fp32: the scores keep (nearly) q's full precision.
//
// Semantics follow attn_split.comp:9-58 + attn_combine.comp:6-21 + gate_rotate.comp:19-25 of the reference, as
// prefill_kernel (same arguments, same results within fp32 rounding): row t (position off+t) of head h attends to
// cache rows [0, off+t+1) of kv head h/4; softmax(q.k/16) v, then a * sigmoid(gate), optionally rotated.
//
// prefill_kernel multiplies fp16 q. An fp32 q rounded to fp16 moves a score by about 2^-12 |q||k|, which at scores
// of tens (peaky heads) shows in the output. Here q is split as hi = fp16(q), lo = fp16(q - hi) and S^T = K hi^T +
// K lo^T (two MFMAs per k-step), so the scores keep about 22 of q's 24 bits. The low part takes 64 more registers
// per lane than prefill_kernel's two waves per SIMD can hold, so this kernel runs one wave per SIMD and hides the
// latencies by software pipelining instead of by a second wave:
//   - K/V tiles of 32 keys go HBM/L2 -> LDS by global_load_lds through a ring of 4 stages, three tiles ahead, in
//     prefill_kernel's padded row-pair layout (the same operand addressing);
//   - per tile the wave computes S^T(j + 1) on the MFMA units while the VALU turns S^T(j) into P(j), then O += P(j)
//     V(j); the LDS operand reads are issued a few MFMAs ahead of their use (scheduling groups);
//   - O stays in the accumulation registers for the whole loop.
// Measured on MI355X (4096 rows, 16/4 heads): 248-282 us, against 171-178 us for prefill_kernel on the same rows
// given as fp16 (the hi/lo product adds half again the MFMA work). Run on fp16 q, this design measured 194-226 us,
// slower than prefill_kernel there: one wave per SIMD issues LDS reads at about half the rate of two (130 against 260
// bytes per cycle per CU for ds_read_b128), so a long fp16 prefill stays on prefill_kernel.
//
// HILO = false is the same kernel on fp16 q, and SPLIT = true takes part of a q-tile's keys per block, for calls whose
// q-tiles alone would leave CUs idle; prefill_combine_kernel merges the splits, gates and rotates. Against the kernel
// with 64-key tiles, no pipelining and two separate launches for the merge and the rotation that these calls had
// (MI355X, a layer call, fp32 q): 777 rows over 1,031, 16/4 heads 121 -> 70 us; 500 over 517, 8/2 53 -> 35; 1,900 over
// 4,000, 16/4 492 -> 287; 3,000 over 1,000, 8/2 239 -> 161. Its sums differ from that kernel's within fp16 P's rounding: m per 32
// keys, l over the rounded weights.
#pragma once
#include <type_traits>

#include "bn_prefill.h"

namespace bn {

constexpr int PH_STAGES = 4;           // K/V stages in LDS: the tile in use, the next one, two in flight
constexpr int PH_OP = 1040;             // row pitch (bytes) of a wave's output rows in LDS at the epilogue
#ifndef PH_KAHEAD
#define PH_KAHEAD 6                     // K operand reads in flight ahead of their MFMA
#endif
#ifndef PH_VAHEAD
#define PH_VAHEAD 4                     // V operand read pairs in flight ahead of their MFMA
#endif


// One block per q-tile: 4 waves, one per SIMD, wave w = query head 4 kh + w over the q-tile's 32 tokens. Each wave
// has the SIMD's whole register file (amdgpu_waves_per_eu 1): O (128), Q^T hi and lo (64 each), two S^T tiles and
// the operand reads in flight. The K/V tiles go through a ring of 4 stages (tile j in stage
// j % 4, copied three tiles ahead); one barrier per tile says that tile j + 1 has landed and that every wave has
// left tile j - 1, whose stage the copy of tile j + 3 then reuses. Tile j + 3's 8 copies go out one after every
// second k-step of S^T(j + 1) (a burst of them after the barrier left the SIMD without MFMAs for their issue time:
// 4-5% slower). Per tile the wave computes S^T(j + 1) = K(j + 1)
// Q^T on the MFMA units while the VALU turns S^T(j) into P(j) (one k-step of each at a time), then O += P(j) V(j),
// the operand reads a few MFMAs ahead of their use.
template <bool HILO, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void prefill_hilo_kernel(PrefillArgs a) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[PH_STAGES * PF_STAGE];
    __shared__ f4 bc_lds[4][16];  // per wave: 64 floats broadcast in row order

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, r32 = lane & 31;
    const int KV = a.KV, ntq = a.ntq;

    // block -> (kv head, q-tile, split): longest q-tiles (highest index) first, each kv head on a fixed set of XCDs
    int kh, qt, sp = 0;
    const int off = call_off(a.dyn, a.off);
    if constexpr (SPLIT) {
        // the splits of the q-tiles, one after another, are a kv head's blocks: no block of the launch is without work
        // (but past the last with a smaller device offset), and the XCDs get equal shares
        const int idx = blockIdx.x / KV;
        kh = blockIdx.x % KV;
        qt = -1;
        for (int c = 0, base = 0; c < ntq; c += 64) {
            const int q = ntq - 1 - c - lane;
            const int n = q < 0 ? 0 : pf_splits((off + min(a.T, (q + 1) * PF_BQ) - 1 + PF_BK) / PF_BK, a.ct);
            const int incl = wave_incl_scan(n, lane);
            const uint64_t hit = __ballot(base + incl > idx);
            if (hit) {
                const int f = __builtin_ctzll(hit);
                qt = ntq - 1 - c - f;
                sp = idx - base - __builtin_amdgcn_readlane(incl - n, f);
                break;
            }
            base += __builtin_amdgcn_readlane(incl, 63);
        }
        if (qt < 0) return;
        qt = __builtin_amdgcn_readfirstlane(qt);
        sp = __builtin_amdgcn_readfirstlane(sp);
    } else {
        const int b = blockIdx.x, nb = KV * ntq;
        int idx;
        if (8 % KV == 0 && nb % 8 == 0) {
            const int xcd = b & 7, reps = 8 / KV;
            kh = xcd % KV;
            idx = (b >> 3) * reps + xcd / KV;
        } else {
            kh = b % KV;
            idx = b / KV;
        }
        qt = ntq - 1 - idx;
    }
    const int t0 = qt * PF_BQ;
    const int t_last = min(a.T, t0 + PF_BQ) - 1;
    const int nk = off + a.T;                         // cache rows that exist
    const int nt_all = (off + t_last + PF_BK) / PF_BK;  // key tiles the q-tile attends to
    // the block's key tiles [jb, nt)
    int jb = 0, nt = nt_all;
    if constexpr (SPLIT) {
        const int n = pf_splits(nt_all, a.ct);
        jb = (int)((int64_t)sp * nt_all / n);
        nt = (int)((int64_t)(sp + 1) * nt_all / n);
    }
    const int64_t kvd = (int64_t)KV * D;
    const uint16_t* kb = a.kc + (int64_t)kh * D;
    const uint16_t* vb = a.vc + (int64_t)kh * D;
    const int head = kh * 4 + w;

    // Tile copies: wave w moves row pairs 4w .. 4w+3 of K and of V (8 copies per tile); copy c of tile jt: K (c even)
    // or V (c odd) of row pair 4 w + c / 2, lane l loading row 32 jt + p + 16 (l / 32), clamped to the cache's last row
    // (those keys are masked), 16-byte chunk l % 32, into LDS pair p at byte 16 l.
    auto tile_copy = [&](int jt, uint8_t* st, int c) __attribute__((always_inline)) {
        const int j0 = jt * PF_BK, lim = nk - 1 - j0, p = 4 * w + (c >> 1);
        const uint32_t go = (uint32_t)(min(p + 16 * h, lim) * (int)kvd + r32 * 8) * 2u;
        if (c & 1)
            pf_copy16(reinterpret_cast<const char*>(vb + (int64_t)j0 * kvd) + go, st + PF_KB + p * PF_VP);
        else
            pf_copy16(reinterpret_cast<const char*>(kb + (int64_t)j0 * kvd) + go, st + p * PF_KP);
    };
    // tiles jb, jb + 1, jb + 2 into stages 0, 1, 2 (a tile past the last repeats the last: its stage is never read as
    // such), so that every tile step finds the same copies in flight
#pragma unroll
    for (int j = 0; j < PH_STAGES - 1; j++)
#pragma unroll
        for (int c = 0; c < 8; c++) tile_copy(min(jb + j, nt - 1), lds + j * PF_STAGE, c);

    // Q^T (hi and lo), under the copies' latency: lane l holds token t0 + l % 32 (clamped), dims 16 ks + 8 h .. +7.
    // Read straight into that layout every load touches 64 places (64 cycles of the address unit each, 128 loads of fp32 per
    // CU, at every block's start), so four neighbouring lanes read 64 bytes of a row and the wave turns 256 bytes of its
    // 32 rows at a time in LDS (stage 3, free until the first tile step): 16-byte slot s of row r at
    // s ^ 4 (r % 4) ^ (r / 4) % 4, which keeps the writes (4 rows x 4 slots) and the reads (16 rows) on distinct banks
    // (256 rows over 512, 8/2 heads: 26.4 -> 25.7 us).
    h8 qb[16], ql[HILO ? 16 : 1];
    {
        constexpr int NP = HILO ? 4 : 2, ES = HILO ? 4 : 2;
        u4 raw[NP][4][2];
#pragma unroll
        for (int rh = 0; rh < 2; rh++) {
            const int tq = min(t0 + (lane >> 2) + 16 * rh, a.T - 1);
            const char* qr = (HILO ? reinterpret_cast<const char*>(a.q) : reinterpret_cast<const char*>(a.q16)) +
                             ((int64_t)tq * a.q_ts + (int64_t)head * a.q_hs) * ES + 16 * (lane & 3);
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int g = 0; g < 4; g++) raw[p][g][rh] = *reinterpret_cast<const u4*>(qr + 256 * p + 64 * g);
        }
        uint8_t* const qs = lds + (PH_STAGES - 1) * PF_STAGE + w * 8192;
        auto slot = [&](int r, int s) { return qs + r * 256 + 16 * (s ^ (4 * (r & 3)) ^ ((r >> 2) & 3)); };
#pragma unroll
        for (int p = 0; p < NP; p++) {
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int rh = 0; rh < 2; rh++)
                    *reinterpret_cast<u4*>(slot((lane >> 2) + 16 * rh, 4 * g + (lane & 3))) = raw[p][g][rh];
            wave_lds_sync();
            if constexpr (HILO) {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int ks = 4 * p + k;
                    const f4 x0 = *reinterpret_cast<const f4*>(slot(r32, 4 * k + 2 * h));
                    const f4 x1 = *reinterpret_cast<const f4*>(slot(r32, 4 * k + 2 * h + 1));
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const float x = e < 4 ? x0[e] : x1[e - 4];
                        const _Float16 hi = (_Float16)x;
                        qb[ks][e] = hi;
                        ql[ks][e] = (_Float16)(x - (float)hi);
                    }
                }
            } else {
#pragma unroll
                for (int k = 0; k < 8; k++) qb[8 * p + k] = *reinterpret_cast<const h8*>(slot(r32, 2 * k + h));
            }
            wave_lds_sync();
        }
    }
    // The loads have landed (and the copies before them); the empty asm statements then redefine Q^T, so the compiler's
    // own waits for these loads (which would count the tile copies issued next) end here.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < 16; ks++) {
        asm volatile("" : "+v"(qb[ks]));
        if constexpr (HILO) asm volatile("" : "+v"(ql[ks]));
    }

    f16x o[8];
#pragma unroll
    for (int dt = 0; dt < 8; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[dt][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;
    const float sc = QK_SCALE * LOG2E;
    const int qpos = off + t0 + r32;  // this lane's row sees keys <= qpos
    const int k_lane = (r32 & 15) * PF_KP + (r32 >> 4) * 512 + h * 16;
    const int vs = lane & 15, vnh = (lane >> 4) & 1;
    const int v_lane = PF_KB + (4 * h + (vs >> 2)) * PF_VP + 32 * vnh + 8 * (vs & 3);
    float* bc = reinterpret_cast<float*>(bc_lds[w]);

    // the first tiles landed for every wave; then S^T of the first
    asm volatile("s_barrier" ::: "memory");
    f16x s_cur;
    {
        const uint8_t* kl = lds + k_lane;
#pragma unroll
        for (int r = 0; r < 16; r++) s_cur[r] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 16; ks++) {
            const h8 kop = pf_lds_h8(kl + ks * 32);
            s_cur = mfma32(kop, qb[ks], s_cur);
            if constexpr (HILO) s_cur = mfma32(kop, ql[ks], s_cur);
        }
    }

    // Tile j: S^T(j + 1) from stage j + 1 (MORE; the kernel without splits computes it also after the last tile, from a
    // stage whose copies are done, and drops it), P(j) from S^T(j), O += P(j) V(j) from stage j.
    auto tile_step = [&](int j, auto copy, auto more) __attribute__((always_inline)) {
        constexpr bool COPY = decltype(copy)::value, MORE = decltype(more)::value;
        // tile j + 1 landed (tile j + 2's copies may be in flight), and every wave is done with tile j - 1, whose
        // stage takes tile j + 3 (a repeat of the last tile past the end), copied during the S^T(j + 1) MFMAs below
        if (COPY || j + 2 < nt)
            asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        const int jc = min(j + 3, nt - 1), js = j - jb;
        uint8_t* cst = lds + ((js + 3) & (PH_STAGES - 1)) * PF_STAGE;
        const uint8_t* cur = lds + (js & (PH_STAGES - 1)) * PF_STAGE;
        const uint8_t* nxt = lds + ((js + 1) & (PH_STAGES - 1)) * PF_STAGE;

        // K(j + 1) operand reads run KA k-steps ahead of their MFMAs; the first ones hide behind the row max
        constexpr int KA = PH_KAHEAD, VA = PH_VAHEAD;
        const uint8_t* kl = nxt + k_lane;
        h8 kop[16];
#pragma unroll
        for (int ks = 0; ks < KA; ks++)
            if (MORE) kop[ks] = pf_lds_h8(kl + ks * 32);

        // the row max of S(j); causal mask on tiles that cross the diagonal (register r: key j0 + 8 (r/4) + 4 h + r%4)
        const int j0 = j * PF_BK;
        if (j0 + PF_BK - 1 > off + t0) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int key = j0 + 8 * (r >> 2) + 4 * h + (r & 3);
                s_cur[r] = key <= qpos ? s_cur[r] : -INFINITY;
            }
        }
        float tm = s_cur[0];
#pragma unroll
        for (int r = 1; r < 16; r++) tm = fmaxf(tm, s_cur[r]);
        tm = max_xhalf(tm);
        const float tmax = tm * sc;  // log2 domain
        // Conditional rescale: m_run moves only when the row's tile max exceeds it by more than 8 (log2 units);
        // otherwise p = 2^(x - m_run) <= 256 stays well inside fp16 and the final division by l cancels the common
        // factor. Rows with no key yet (m_run = -inf) have O = 0 and just take the max. In the first
        // a.exact tiles m_run follows the max exactly: the weight of a row's largest key so far is then 1, which fp16
        // holds exactly, and in a short range those weights carry the rounding error (128 keys: 1.6e-4 of the output
        // instead of 1.9e-4). O's rescale costs about a third of a tile.
        float alpha = 1.0f;
        bool moved = false;
        if (tmax > m_run + (j - jb < a.exact ? 0.0f : 8.0f)) {
            moved = m_run != -INFINITY;
            alpha = moved ? __builtin_amdgcn_exp2f(m_run - tmax) : 0.0f;
            m_run = tmax;
        }
        if (__ballot(moved)) {
            if (h == 0) bc[r32] = alpha;
            f4 al[4];
#pragma unroll
            for (int gg = 0; gg < 4; gg++) al[gg] = bc_lds[w][2 * gg + h];
#pragma unroll
            for (int dt = 0; dt < 8; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    float x = o[dt][r];
                    scale_acc(x, al[r >> 2][r & 3]);
                    o[dt][r] = x;
                }
        }
        l_run *= alpha;
        const float m_use = m_run == -INFINITY ? 0.0f : m_run;

        // S(j + 1) on the MFMA units while the VALU turns S(j) into P(j), one k-step at a time; the first V(j)
        // operand reads start in the last k-steps
        f16x s_next;
#pragma unroll
        for (int r = 0; r < 16; r++) s_next[r] = 0.0f;
        h8 pa[2];
        h4 vx[16][2];
        const uint8_t* vl = cur + v_lane;
        auto v_read = [&](int i) {  // PV step i: keys 16 (i / 8) .. +15, dims 32 (i % 8) .. +31
            const int imm0 = (i >> 3) * 512 + 64 * (i & 7);
            vx[i][0] = pf_lds_tr(vl + imm0);
            vx[i][1] = pf_lds_tr(vl + imm0 + 8 * PF_VP);
        };
        // The scheduling groups fix the order per k-step (its LDS reads, its two MFMAs, four VALU instructions), so
        // the reads stay KA (V: VA) steps ahead; left alone, the compiler moves each read next to its MFMA.
#pragma unroll
        for (int ks = 0; ks < 16; ks++) {
            if (MORE && ks + KA < 16) kop[ks + KA] = pf_lds_h8(kl + (ks + KA) * 32);
            if (ks + VA >= 16) v_read(ks + VA - 16);
            if constexpr (MORE) {
                s_next = mfma32(kop[ks], qb[ks], s_next);
                if constexpr (HILO) s_next = mfma32(kop[ks], ql[ks], s_next);
            }
            pa[ks >> 3][ks & 7] = (_Float16)__builtin_amdgcn_exp2f(fmaf(s_cur[ks], sc, -m_use));
            if constexpr (!MORE) continue;
            if (ks + KA < 16 && ks + VA >= 16) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
            else if (ks + KA < 16) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            else if (ks + VA >= 16) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, HILO ? 2 : 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, 4, 0);
            if (COPY && (ks & 1)) {  // one copy after every second k-step's MFMAs, which stay ahead of it
                tile_copy(jc, cst, ks >> 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // l sums the weights as they multiply V, rounded, in fp32: rounding then moves sum and numerator alike (against 64
        // bits, V of mean 1: 0.8-3.2e-5 of the output, with unrounded weights 1.1-4.6e-5; of mean 0 1.5-1.8e-4 both)
        const h2 one = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const h2 pp = {pa[k][2 * e], pa[k][2 * e + 1]};
                l_run = __builtin_amdgcn_fdot2(pp, one, l_run, false);
            }
        // O += P(j) V(j) over the 32 keys: two 16-key steps; V operand rows 16 kk + 8 rd + 4 h + (l % 16) / 4
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if (i + VA < 16) v_read(i + VA);
            const h8 vop = __builtin_shufflevector(vx[i][0], vx[i][1], 0, 1, 2, 3, 4, 5, 6, 7);
            o[i & 7] = mfma32(pa[i >> 3], vop, o[i & 7]);
            if (i == 0) __builtin_amdgcn_sched_group_barrier(0x402, 8, 0);
            if (i + VA < 16) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        s_cur = s_next;
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    if constexpr (SPLIT) {
        // ranges are short: their last three tiles bring no others, and the last computes no further S (300 rows over 100,
        // 16/4 heads, fp16 q, with the records' stores below: kernel 18.2 -> 15.2 us)
        int j = jb;
        for (; j < nt - 3; j++) tile_step(j, yes, yes);
        for (; j < nt - 1; j++) tile_step(j, no, yes);
        tile_step(j, no, no);
    } else {
        for (int j = jb; j < nt; j++) tile_step(j, yes, yes);
    }

    // Epilogue. O / l goes to LDS as each wave's [32 tokens][256 dims] (pitch PH_OP), then rows are read back 16
    // bytes per lane for coalesced gated stores, or, with signs, per (token, head pair) for the rotation. A wave's rows
    // are head w's 32 tokens, or (rotated) head pair w % 2 of the tokens w / 2 + 2 k; their gate rows are all requested
    // here: read row by row between the stores (which may alias them) they cost a round trip each, 16 or 8 in a row on a
    // CU that runs nothing else (a layer call of 4,096 rows, 16/4 heads: 276 against 257 us; of 70 rows, 8/2: 31 against
    // 27).
    f4 z[32], sg[2];
    if constexpr (!SPLIT) {
        if (a.gate) {
#pragma unroll
            for (int k = 0; k < 32; k++) {
                const int tl = a.signs ? (w >> 1) + 2 * (k >> 1) : k;
                const int hd = a.signs ? kh * 4 + 2 * (w & 1) + (k & 1) : head;
                z[k] = *reinterpret_cast<const f4*>(a.gate + (int64_t)min(t0 + tl, a.T - 1) * a.g_ts +
                                                    (int64_t)hd * a.g_hs + 4 * lane);
            }
        }
        if (a.signs)
#pragma unroll
            for (int i = 0; i < 2; i++)
                sg[i] = *reinterpret_cast<const f4*>(a.signs + (int64_t)(kh * 4 + 2 * (w & 1) + i) * D + 4 * lane);
    }
    const float l_tot = sum_xhalf(l_run);
    if (h == 0) bc[r32] = SPLIT ? 1.0f : 1.0f / l_tot;
    f4 lv[4];
#pragma unroll
    for (int gg = 0; gg < 4; gg++) lv[gg] = bc_lds[w][2 * gg + h];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last tile steps' copies (repeats) have landed
    __syncthreads();  // every wave is done with the stages
    uint8_t* orow = lds + w * 32 * PH_OP;
#pragma unroll
    for (int dt = 0; dt < 8; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int tl = 8 * (r >> 2) + 4 * h + (r & 3);
            *reinterpret_cast<float*>(orow + tl * PH_OP + 4 * (32 * dt + r32)) = o[dt][r] * lv[r >> 2][r & 3];
        }
    __syncthreads();
    if constexpr (SPLIT) {
        // the split's record: unnormalised rows, m and l per row
        const int64_t row = (((int64_t)kh * ntq + qt) * a.max_splits + sp) * PF_ROWS + w * PF_BQ;
        if (h == 0) {
            a.part_ml[(row + r32) * 2] = m_run;
            a.part_ml[(row + r32) * 2 + 1] = l_tot;
        }
        // Short ranges end together, and their stores with them: non-temporal, these leave the L2s at once instead of at the
        // kernel's end (96 rows over 512, 32/8 heads, 20 MB: kernel 20.2 -> 18.7 us, the merge 0.4 longer). Not where
        // longer ranges end apart anyway, nor where the merge reads a row's splits in several round trips (65 rows over
        // 5,000, one kv head: 36 us, 41 with them).
        float* const rec = a.part_acc + row * D + 4 * lane;
        const uint8_t* const src = orow + 16 * lane;
        if (a.ct <= 8 && a.max_splits <= 16) {
#pragma unroll 4
            for (int tl = 0; tl < PF_BQ; tl++)
                __builtin_nontemporal_store(*reinterpret_cast<const f4*>(src + tl * PH_OP),
                                            reinterpret_cast<f4*>(rec + tl * D));
        } else {
#pragma unroll 4
            for (int tl = 0; tl < PF_BQ; tl++)
                *reinterpret_cast<f4*>(rec + tl * D) = *reinterpret_cast<const f4*>(src + tl * PH_OP);
        }
        return;
    }
    if (!a.signs) {
#pragma unroll
        for (int tl = 0; tl < PF_BQ; tl++) {
            const int t = t0 + tl;
            f4 y = *reinterpret_cast<const f4*>(orow + tl * PH_OP + 16 * lane);
            if (a.gate) {
#pragma unroll
                for (int e = 0; e < 4; e++) y[e] = gate_mul_fast(y[e], z[tl][e]);
            }
            if (t < a.T)
                __builtin_nontemporal_store(y, reinterpret_cast<f4*>(a.out + (int64_t)t * a.o_ts +
                                                                   (int64_t)head * a.o_hs + 4 * lane));
        }
        return;
    }
    // rotation: lane l holds dims 4l .. 4l+3 of heads 2p and 2p + 1
    const int p = w & 1;
#pragma unroll
    for (int k = 0; k < PF_BQ / 2; k++) {
        const int tl = (w >> 1) + 2 * k, t = t0 + tl;
        float v[8];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            f4 y = *reinterpret_cast<const f4*>(lds + (2 * p + i) * 32 * PH_OP + tl * PH_OP + 16 * lane);
            if (a.gate) {
#pragma unroll
                for (int e = 0; e < 4; e++) y[e] = gate_mul_fast(y[e], z[2 * k + i][e]);
            }
            y *= sg[i];
#pragma unroll
            for (int c = 0; c < 4; c++) v[4 * i + c] = y[c];
        }
        fwht512_wave(v, lane);
        float* o_ = a.out + (int64_t)t * a.o_ts + (int64_t)(kh * 4 + 2 * p) * a.o_hs;
        if (t < a.T)
#pragma unroll
            for (int i = 0; i < 2; i++)
                __builtin_nontemporal_store(f4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]} * INV_SQRT512,
                                            reinterpret_cast<f4*>(o_ + i * a.o_hs + 4 * lane));
    }
}

// Merge of the key splits of one (token, head pair) in split order (attn_combine.comp:10-20), then the gate and, with
// signs, the rotation of the pair's 512 elements (gate_rotate.comp:18-25). Grid (T, H / 2) x 128 threads; a wave per head,
// thread: dims 4 lane .. +3 of it; with signs the second head's row goes through LDS to the first's wave, which transforms
// the pair. Bound by the records' round trips: the first 16 splits' accumulators are requested with the (m, l) terms, the
// others 8 at a time (one wave for both heads, the first 8 up front and the others one by one, took 11 us instead of 6 for
// 96 rows over 1,031, 18 splits, 8/2 heads).
__global__ __launch_bounds__(128) void prefill_combine_kernel(PrefillArgs a) {
    constexpr int PRE = 16, FEW = 8;
    __shared__ f4 row1[64];
    const int t = blockIdx.x, lane = threadIdx.x & 63, kh = blockIdx.y >> 1, p = blockIdx.y & 1;
    const int i = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);  // head of the pair
    const int qt = t / PF_BQ, t_last = min(a.T, qt * PF_BQ + PF_BQ) - 1;
    const int hd = kh * 4 + 2 * p;  // the pair's first head
    f4 z = {0.0f, 0.0f, 0.0f, 0.0f}, sg = z;
    if (a.gate) z = *reinterpret_cast<const f4*>(a.gate + (int64_t)t * a.g_ts + (int64_t)(hd + i) * a.g_hs + 4 * lane);
    if (a.signs) sg = *reinterpret_cast<const f4*>(a.signs + (int64_t)(hd + i) * D + 4 * lane);
    const int ns = pf_splits((call_off(a.dyn, a.off) + t_last + PF_BK) / PF_BK, a.ct);
    // row of the head's split 0; split s is PF_ROWS rows on
    const int64_t row0 = ((int64_t)kh * a.ntq + qt) * a.max_splits * PF_ROWS + (2 * p + i) * PF_BQ + t % PF_BQ;
    auto acc_of = [&](int s) {
        return *reinterpret_cast<const f4*>(a.part_acc + (row0 + (int64_t)s * PF_ROWS) * D + 4 * lane);
    };
    const float* ml = a.part_ml + row0 * 2;
    f4 pre[PRE];
#pragma unroll
    for (int u = 0; u < PRE; u++) pre[u] = u < ns ? acc_of(u) : f4{0.0f, 0.0f, 0.0f, 0.0f};
    float L = 0.0f;
    f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    if (ns <= FEW) {
        // few splits: every lane takes all their terms, without the exchanges below
        float m[FEW], l[FEW];
#pragma unroll
        for (int u = 0; u < FEW; u++) {
            const float* r = ml + (int64_t)min(u, ns - 1) * PF_ROWS * 2;
            m[u] = u < ns ? r[0] : -INFINITY;
            l[u] = r[1];
        }
        float M = m[0];
#pragma unroll
        for (int u = 1; u < FEW; u++) M = fmaxf(M, m[u]);
#pragma unroll
        for (int u = 0; u < FEW; u++) {
            const float wu = m[u] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m[u] - M);
            L = fmaf(l[u], wu, L);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] = fmaf(pre[u][e], wu, acc[e]);
        }
    } else {
        auto m_of = [&](int s) { return s < ns ? ml[(int64_t)s * PF_ROWS * 2] : -INFINITY; };
        auto l_of = [&](int s) { return s < ns ? ml[(int64_t)s * PF_ROWS * 2 + 1] : 0.0f; };
        const float m0 = m_of(lane), l0 = l_of(lane);
        float M = m0;
        for (int s = lane + 64; s < ns; s += 64) M = fmaxf(M, m_of(s));
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) M = fmaxf(M, __shfl_xor(M, o));
        for (int base = 0; base < ns; base += 64) {
            const float ms = base == 0 ? m0 : m_of(base + lane), ls = base == 0 ? l0 : l_of(base + lane);
            const float wgt = ms == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ms - M);  // split base + lane
            const int cnt = min(64, ns - base);
            auto add = [&](int u, f4 v) {
                const float wu = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wgt), u));
                L = fmaf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(ls), u)), wu, L);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[e] = fmaf(v[e], wu, acc[e]);
            };
            int u0 = 0;
            if (base == 0) {
#pragma unroll
                for (int u = 0; u < PRE; u++)
                    if (u < cnt) add(u, pre[u]);
                u0 = PRE;
            }
            for (; u0 < cnt; u0 += 8) {
                f4 v[8];
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (u0 + u < cnt) v[u] = acc_of(base + u0 + u);
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (u0 + u < cnt) add(u0 + u, v[u]);
            }
        }
    }
    f4 y;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        y[e] = acc[e] / L;
        if (a.gate) y[e] = gate_mul(y[e], z[e]);
    }
    f4* const o = reinterpret_cast<f4*>(a.out + (int64_t)t * a.o_ts + (int64_t)(hd + i) * a.o_hs + 4 * lane);
    if (!a.signs) {
        *o = y;
        return;
    }
    y *= sg;
    if (i) row1[lane] = y;
    __syncthreads();
    if (i) return;
    const f4 y1 = row1[lane];
    float v[8] = {y[0], y[1], y[2], y[3], y1[0], y1[1], y1[2], y1[3]};
    fwht512_wave(v, lane);
    *o = f4{v[0], v[1], v[2], v[3]} * INV_SQRT512;
    *reinterpret_cast<f4*>(reinterpret_cast<float*>(o) + a.o_hs) = f4{v[4], v[5], v[6], v[7]} * INV_SQRT512;
}

}  // namespace bn
