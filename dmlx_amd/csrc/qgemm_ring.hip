// Grouped quantized GEMM, ring path: prefill-sized calls on weights in the MLX layout, every quantized format, tiles of up to
// 128 rows of one expert segment. That is dmoe_gather_qmm on the caller's own arrays, and the gate / up launch of a layer whose
// ffn is no multiple of 32 (such stacks are not re-ordered; their down projection is then an unquantized one).
//
// What bounds such a call on these arrays is how the weights are fetched. Operand-layout loads (qgemm_mfma.hip) take 32
// bytes out of each of 64 rows, and one 2-byte scale and bias per row and step: every 128-byte line is touched four times
// per chunk stream and does not survive in the L1 in between. Here EVERYTHING the loop reads goes straight into rings of LDS
// slots (global_load_lds) in pieces that suit the arrays - 64 bytes of 16 rows per weight request, 16 bytes of scales and
// biases per row for 8 groups - and the wavefront reads its operands out of LDS. One projection [256, 2048, 4096] of 8-bit
// weights, 12 480 rows over 187 experts: 1.78 -> 0.50 ms (1.6 GB of weights: 0.9 -> 3.1 TB/s).
//
// One workgroup (4 wavefronts) takes a tile against a strip of 128 (gate and up) or 256 output columns; a wavefront decodes
// its own 64 weight rows into the A operand of v_mfma_f32_32x32x16_bf16. The slots fit 80 KiB, so that two workgroups share a
// compute unit. The loop holds no load the compiler knows about: loads return in issue order, and a compiler-made wait for
// one register load would drain every younger slot request with it.
//
//  * Group i of requests = activations of step i, weights of step i + 1 (decoded one step ahead). It is issued behind the
//    barrier that frees its slot, in the last MFMA group of one step and the first two of the next; with R slots R - 1
//    groups are in flight while a step (64 elements) computes.
//  * Barrier B(s) sits in front of the last MFMA group of step s: group s + 1 has landed ("at most (R - 2) groups
//    outstanding"), and this wavefront's reads of slot s are done, so behind it slot s + 1 may be read and slot s refilled.
//  * Activations: one request moves 8 rows x 128 bytes, piece c of row r at position c ^ ((r >> 1) & 7) (operand reads run
//    free of bank conflicts). Weights and scales are private to their wavefront: no barrier is involved, only the wait.
//  * A weight request takes 64 bytes of 16 rows (four lanes per row): one step of an 8-bit format or a pair of steps of a
//    4-bit format (PAIRS). Piece c of row r lies at c ^ ((r >> 2) & 3).
//
// The reduction loop is software-pipelined: units of [one MFMA | a slice of the decode of the next weights] separated by
// scheduling barriers, as in qgemm_wide.hip.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "qformat.h"
#include "wide_epilogue.h"

namespace dmoe {

constexpr int kRingWaves = 4;
constexpr size_t kRingLdsBytes = 80 * 1024; // two workgroups per compute unit

constexpr int ring_wait_vm(int n) { return 0x0f70 | (n & 15) | ((n >> 4) << 14); }  // vmcnt <= n
constexpr int ring_wait_both(int n) { return 0x0070 | (n & 15) | ((n >> 4) << 14); } // vmcnt <= n, lgkmcnt = 0
constexpr int kRingWaitLgkm = 0xc07f;

// slots and sizes of one instantiation
template <typename Fmt, int MT>
struct RingGeom {
    static constexpr int CH = 32 / Fmt::kVals;                  // 16-byte chunk steps per step: 1 (4-bit) or 2 (8-bit)
    static_assert(CH == 1 || CH == 2, "formats of 4 or 8 bits");
    static constexpr bool PAIRS = CH == 1;                      // weights come two steps at a time
    static constexpr int ACT = MT * 4096;                       // activations of a step
    static constexpr int WB = 4096;                             // weights of a slot, per wavefront
    static constexpr bool META = Fmt::kMetaEntryBytes != 0;
    static constexpr bool BIAS = Fmt::kMetaEntryBytes == 2;
    static constexpr int MBLK = !META ? 0 : BIAS ? 2048 : 1024; // a block of scale (and bias) entries, per wavefront
    static constexpr int fit() {
        const int left = (int)kRingLdsBytes - kRingWaves * 2 * MBLK;
        return left / (ACT + kRingWaves * WB); // 8-bit: 3 slots at MT = 1, else 2; FP8: 4, 3, 2, 2
    }
    static constexpr int RW = PAIRS ? (MT == 1 ? 3 : 2) : fit();            // weight slots
    static constexpr int RA = PAIRS ? (MT <= 2 ? 4 : 2) : fit();            // activation slots
    static constexpr int W_OFF = RA * ACT, M_OFF = W_OFF + kRingWaves * RW * WB;
    static constexpr int TOTAL = M_OFF + kRingWaves * 2 * MBLK;
    static_assert(RA >= 2 && RA <= 4 && RW >= 2 && TOTAL <= (int)kRingLdsBytes, "the ring does not fit, or holds more groups than the waits below tell apart");
    static constexpr int NW = 4;                                // weight requests of a slot
};

template <typename Fmt, bool GATE_UP, int MT>
__device__ __forceinline__ void ring_tile(const GemmArgs &g, const Tile &t, uint8_t *lds, const int strip) {
    using G = RingGeom<Fmt, MT>;
    constexpr int KV = Fmt::kVals, CH = G::CH, NJ = 4, NT = 2, NJC = NJ / CH;
    constexpr int NUC = NJC * MT * NT;    // units (MFMAs) per chunk step
    constexpr int NPC = NT * (KV / 2);    // packed pairs to decode per chunk step
    constexpr int RA = G::RA, RW = G::RW;
    constexpr bool PAIRS = G::PAIRS;
    const int tid = (int)threadIdx.x, lane = tid & 63, ln = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cols = g.b0.cols, n_out = g.b0.rows;
    const int n_steps = cols / 64;
    const size_t e = t.expert;
    const uint32_t lds_addr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;

    // ---- this wavefront's weight rows (gate_up: tile 0 = gate, tile 1 = up rows of the same 32 columns) ----
    const int col_base = (strip * kRingWaves + wave) * (GATE_UP ? 32 : 64);
    const bool wave_on = col_base < n_out;
    const uint8_t *w_base[NT];            // uniform: first byte of the matrix
    uint32_t w_lane[NT][2];               // this lane's row and piece for the two requests of a tile
    const uint8_t *m_ptr = nullptr, *b_ptr = nullptr; // scale / bias row of this lane: row `ln` of tile `h`
    bool has_bias[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const QView &b = (GATE_UP && nt == 1) ? g.b1 : g.b0;
        const int base = GATE_UP ? col_base : col_base + 32 * nt;
        const int row0 = wave_on && base < n_out ? base : 0; // a switched-off tile aliases valid memory, never stored
        has_bias[nt] = b.biases != nullptr;
        w_base[nt] = b.w + e * b.w_mat;
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            const int r = 16 * o + (lane >> 2);
            const int n = row0 + r < n_out ? row0 + r : n_out - 1;
            w_lane[nt][o] = (uint32_t)n * (uint32_t)b.w_row + (uint32_t)(((lane & 3) ^ ((r >> 2) & 3)) * 16);
        }
        const int n = row0 + ln < n_out ? row0 + ln : n_out - 1;
        if (G::META && h == nt) {
            m_ptr = b.scales + e * b.s_mat + (size_t)n * b.s_row;
            b_ptr = (b.biases ? b.biases : b.scales) + e * b.s_mat + (size_t)n * b.s_row;
        }
    }

    // ---- requests ---------------------------------------------------------------------------------------------
    // (a wait state between the write of M0 and the request that reads it; nothing else in this kernel uses M0)
    auto dma16 = [&](const uint8_t *base, uint32_t off, uint32_t la) { // uniform base, 32-bit lane offset
        // (no streaming hint: a half line comes back for its other half; 32 rows of 8-bit weights: 300 -> 460 us with it)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(la) : "memory");
    };
    auto dma16p = [&](const uint8_t *p, uint32_t la) {
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(p), "s"(la) : "memory");
    };
    // activation request i of this wavefront: rows (wave + 4 i) * 8 .. + 7; rows past the segment alias its first row
    const uint8_t *a_src[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int r = (wave + 4 * i) * 8 + (lane >> 3);
        const uint32_t pr = t.row0 + (uint32_t)(r < (int)t.nrows ? r : 0);
        const size_t src = g.a_rows ? g.a_rows[pr] : pr;
        a_src[i] = (const uint8_t *)(g.a + src * (size_t)cols) + (((lane & 7) ^ ((r >> 1) & 7)) * 16);
    }
    const uint32_t w_lds = lds_addr + (uint32_t)(G::W_OFF + wave * RW * G::WB);
    const uint32_t m_lds = lds_addr + (uint32_t)(G::M_OFF + wave * 2 * G::MBLK);
    auto issue_a = [&](int i, int step, int slot) {
        dma16p(a_src[i] + (size_t)step * 128, lds_addr + (uint32_t)(slot * G::ACT + (wave + 4 * i) * 1024));
    };
    // weight request k of a slot: step `step` (not PAIRS), pair of steps `step` (PAIRS)
    auto issue_w = [&](int k, int step, int slot) {
        const int nt = k / (G::NW / NT), o = k % (G::NW / NT);
        const uint32_t la = w_lds + (uint32_t)(slot * G::WB + k * 1024);
        dma16(w_base[nt] + (size_t)step * 64, w_lane[nt][o], la); // PAIRS: whole pairs only, see qgemm_ring_supports
    };
    // block `b` of scale and bias entries, 16 bytes of every row
    const int sb_log = G::MBLK ? (G::BIAS ? __builtin_ctz(g.b0.group) - 3 : 3) : 0; // log2 of the steps a block spans
    const int n_blocks = G::MBLK ? n_steps >> sb_log : 0;
    auto issue_block = [&](int b) {
        if (b >= n_blocks) return;
        const uint32_t la = m_lds + (uint32_t)((b & 1) * G::MBLK);
        dma16p(m_ptr + (size_t)b * 16, la);
        if (G::BIAS) dma16p(b_ptr + (size_t)b * 16, la + 1024u);
    };
    constexpr int NOPS = MT + (PAIRS ? 0 : G::NW); // requests of a group (PAIRS: every other step has NW more)
    // request o of group i (activations of step i; weights of step i + 1, the last step's again past the end)
    auto issue = [&](int o, int i, int slot) {
        const int wstep = i + 1 < n_steps ? i + 1 : n_steps - 1;
        if (o < MT) {
            if (i >= 0) issue_a(o, i, slot);
        } else if (!PAIRS) {
            issue_w(o - MT, wstep, slot);
        }
    };

    // ---- LDS reads -----------------------------------------------------------------------------------------------
    // fragment (mt, j) of a step: row mt * 32 + ln, the piece that holds this lane's eight reduction elements of MFMA
    // group j (chunk step j / NJC of the step, elements (2 c + h) * KV + 8 (j % NJC) onwards)
    uint32_t x_rd[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int piece = ((2 * (j / NJC) + h) * KV + 8 * (j % NJC)) >> 3;
        x_rd[j] = (uint32_t)((ln >> 3) * 1024 + (ln & 7) * 128 + ((piece ^ ((ln >> 1) & 7)) * 16));
    }
    bf16x8_t xf[2][MT]; // activation fragments of the current / next MFMA group
    auto read_x = [&](int slot, int j, int mt) {
        const uint4 q = *(const uint4 *)(lds + x_rd[j] + slot * G::ACT + mt * 4096);
        xf[j & 1][mt] = __builtin_bit_cast(bf16x8_t, q);
    };
    const uint8_t *const w_mine = lds + G::W_OFF + wave * RW * G::WB;
    const uint8_t *const m_mine = lds + G::M_OFF + wave * 2 * G::MBLK;
    uint32_t w_rd[2]; // position of this lane's chunk (row ln; piece 2 c + h) in a slot, c = chunk or step of the pair
#pragma unroll
    for (int c = 0; c < 2; ++c) w_rd[c] = (uint32_t)((ln >> 4) * 1024 + (ln & 15) * 64 + (((2 * c + h) ^ ((ln >> 2) & 3)) * 16));
    // chunk c of a step (PAIRS: of step c of the pair) for tile nt
    auto read_raw = [&](int slot, int c, int nt) {
        return *(const uint4 *)(w_mine + slot * G::WB + nt * 2048 + w_rd[c]);
    };
    auto read_meta = [&](int step, int c, int nt) {
        uint32_t sb[2] = {0u, 0u};
        if (G::META) {
            const uint8_t *blk = m_mine + ((step >> sb_log) & 1) * G::MBLK + (nt * 32 + ln) * 16;
            const int rest = step & ((1 << sb_log) - 1);
            if (G::BIAS) {
                // entry of this lane's chunk among the block's eight: elements 64 rest (+ 32 for the second chunk) on
                const int el = 64 * rest + 32 * (CH == 1 ? h : c);
                const int ent = el >> __builtin_ctz(g.b0.group);
                sb[0] = *(const uint16_t *)(blk + ent * 2);
                sb[1] = has_bias[nt] ? *(const uint16_t *)(blk + 1024 + ent * 2) : 0u;
            } else {
                sb[0] = blk[2 * rest + h];
            }
        }
        return Fmt::pair_meta(Fmt::meta_from_raw(sb));
    };

    f32x16_t acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.0f;
    uint32_t wp[2][NT][KV / 2]; // decoded weights of the current / next chunk step
    uint4 raw[2][NT];           // CH == 1: chunks of the next / next but one step; CH == 2: the step's first / second chunk
    Meta meta[2][NT];

    // ---- prologue: groups -1 .. R - 2 requested (group -1 = weights of step 0), first decode -----------------------
    if (G::MBLK) {
        issue_block(0);
        issue_block(1);
    }
    if (PAIRS) {
#pragma unroll
        for (int q = 0; q < RW; ++q)
            if (2 * q < n_steps)
#pragma unroll
                for (int k = 0; k < G::NW; ++k) issue_w(k, q, q);
    } else {
#pragma unroll
        for (int o = MT; o < NOPS; ++o) issue(o, -1, RA - 1);
    }
#pragma unroll
    for (int i = 0; i < RA - 1; ++i)
        if (i < n_steps)
#pragma unroll
            for (int o = 0; o < NOPS; ++o) issue(o, i, i);
    // group 0 (and everything older) has landed
    if (n_steps >= RA - 1) __builtin_amdgcn_s_waitcnt(ring_wait_vm((RA - 2) * NOPS));
    else __builtin_amdgcn_s_waitcnt(ring_wait_vm(0));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    {
        // chunk step 0 decoded; then the chunk the loop decodes first
        uint4 r0[NT];
        Meta m0[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            r0[nt] = read_raw(PAIRS ? 0 : RA - 1, 0, nt);
            m0[nt] = read_meta(0, 0, nt);
            if (CH == 2) {
                raw[1][nt] = read_raw(RA - 1, 1, nt);
                meta[1][nt] = read_meta(0, 1, nt);
            } else {
                raw[1][nt] = read_raw(0, PAIRS ? 1 : 0, nt);
                meta[1][nt] = read_meta(1, 0, nt);
            }
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            uint32_t st[Fmt::kPairState] = {};
#pragma unroll
            for (int p = 0; p < KV / 2; ++p) Fmt::decode_pair(r0[nt], m0[nt], p, wp[0][nt], st);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) read_x(0, 0, mt);
    __builtin_amdgcn_s_waitcnt(kRingWaitLgkm); // slot R - 1 has been read: group R - 1 may overwrite it
    asm volatile("" ::: "memory");
    if (RA - 1 < n_steps)
#pragma unroll
        for (int o = 0; o < NOPS; ++o) issue(o, RA - 1, RA - 1);

    // requests of a group spread over the units behind its barrier: 2 MT of the last MFMA group of a step, then 4 MT of
    // the first two of the next one
    constexpr int kWindow = 6 * MT, kTailUnits = 2 * MT;
    int cur = 0, nxt = 1 % RA, prv = RA - 1; // slots of steps s, s + 1, s - 1
    int wcur = 0, wnxt = 1 % RW;             // PAIRS: slots of the pair of step s, of the next pair
    // The loop runs pairs of steps; the surplus step of an odd reduction multiplies zeroed activations.
#pragma unroll 1
    for (int s0 = 0; s0 < n_steps; s0 += 2) {
#pragma unroll
        for (int par = 0; par < 2; ++par) {
            const int s = s0 + par;
            const bool stage_now = s + RA < n_steps, stage_prev = s > 0 && s - 1 + RA < n_steps; // uniform
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int which = CH == 1 ? par : c;     // wp slot of the chunk step computed now
                const int src = which ^ 1;               // raw / meta slot of the chunk step decoded now
                uint32_t dstate[Fmt::kPairState] = {};
                Fmt::pair_state(dstate);
#pragma unroll
                for (int jc = 0; jc < NJC; ++jc) {
                    const int jj = c * NJC + jc; // MFMA group within the step
                    if (jj == NJ - 2 && s + 1 == n_steps && par == 0) { // the surplus step reads zeros
#pragma unroll
                        for (int i = 0; i < MT; ++i)
                            *(uint4 *)(lds + nxt * G::ACT + (wave + 4 * i) * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
                    }
                    if (jj == NJ - 1) { // B(s)
                        if (PAIRS) {
                            // Requests younger than the activations of step s + 1 and, in even steps, than the pair of
                            // step s + 2 (requested in step s + 3 - 2 RW). The first step has only the prologue's behind it.
                            constexpr int N_ACT = (RA - 2) * MT, N_PAIR = (2 * RW - 3) * MT + (RW - 2) * G::NW;
                            constexpr int N_ODD = N_ACT + (RA > 2 ? G::NW : 0), N_EVEN = N_ODD < N_PAIR ? N_ODD : N_PAIR;
                            static_assert(!PAIRS || RA == 2 || RA == 4, "a window of two steps holds one pair");
                            if (s - 1 + (RA > 2 * RW ? RA : 2 * RW) >= n_steps) __builtin_amdgcn_s_waitcnt(ring_wait_both(0));
                            else if (par == 1) __builtin_amdgcn_s_waitcnt(ring_wait_both(N_ODD));
                            else if (s == 0) __builtin_amdgcn_s_waitcnt(ring_wait_both(N_ACT < N_PAIR ? N_ACT : N_PAIR));
                            else __builtin_amdgcn_s_waitcnt(ring_wait_both(N_EVEN));
                        } else {
                            const int young = n_steps - 2 - s; // groups behind s + 1 that exist
                            if (young >= RA - 2) __builtin_amdgcn_s_waitcnt(ring_wait_both((RA - 2) * NOPS));
                            else if (RA > 3 && young >= 1) __builtin_amdgcn_s_waitcnt(ring_wait_both(NOPS));
                            else __builtin_amdgcn_s_waitcnt(ring_wait_both(0));
                        }
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_s_barrier();
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_sched_barrier(0);
                        // the block of entries behind the one whose last step has just been read
                        if (G::MBLK && ((s + 2) & ((1 << sb_log) - 1)) == 0) issue_block(((s + 2) >> sb_log) + 1);
                    }
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt) {
                            const int uc = (jc * MT + mt) * NT + nt; // unit within the chunk step
                            const int ug = mt * NT + nt;             // unit within the MFMA group
                            const uint4 q = make_uint4(wp[which][nt][4 * jc], wp[which][nt][4 * jc + 1], wp[which][nt][4 * jc + 2],
                                                       wp[which][nt][4 * jc + 3]);
                            acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, q), xf[jj & 1][mt],
                                                                                  acc[mt][nt], 0, 0, 0);
                            if (nt == 0) { // a whole MFMA group ahead
                                if (jj + 1 < NJ) read_x(cur, jj + 1, mt);
                                else read_x(nxt, 0, mt);
                            }
                            // chunks and scales to decode next: the following step's behind its barrier (one chunk per
                            // step), or the two of step s + 1 as their registers fall free (two chunks)
                            if (CH == 1) {
                                if (jj == NJ - 1 && mt == 0) {
                                    raw[which][nt] = PAIRS ? read_raw(wnxt, par, nt) : read_raw(nxt, 0, nt);
                                    meta[which][nt] = read_meta(s + 2, 0, nt);
                                }
                            } else if (mt == 0 && jj == 1) {
                                raw[0][nt] = read_raw(cur, 0, nt);
                                meta[0][nt] = read_meta(s + 1, 0, nt);
                            } else if (mt == 0 && jj == 2) {
                                raw[1][nt] = read_raw(cur, 1, nt);
                                meta[1][nt] = read_meta(s + 1, 1, nt);
                            }
#pragma unroll
                            for (int o = 0; o < NOPS; ++o) {
                                const int at = o * kWindow / NOPS;
                                if (jj == NJ - 1 && at == ug) {
                                    if (stage_now) issue(o, s + RA, cur);
                                } else if (jj < 2 && at == kTailUnits + jj * 2 * MT + ug) {
                                    if (stage_prev) issue(o, s - 1 + RA, prv);
                                }
                            }
                            if (PAIRS && par == 1 && jj == 0 && mt == 0) { // the pair of step s - 1 is used up
                                if ((s - 1) + 2 * RW < n_steps) {
                                    issue_w(2 * nt, ((s - 1) >> 1) + RW, wcur);
                                    issue_w(2 * nt + 1, ((s - 1) >> 1) + RW, wcur);
                                }
                            }
#pragma unroll
                            for (int p = uc * NPC / NUC; p < (uc + 1) * NPC / NUC; ++p) {
                                Fmt::decode_pair(raw[src][p / (KV / 2)], meta[src][p / (KV / 2)], p % (KV / 2), wp[which ^ 1][p / (KV / 2)], dstate);
                                // pin the slice here (the optimiser would sink a trip's last decode into the next trip)
                                asm volatile("" : "+v"(wp[which ^ 1][p / (KV / 2)][p % (KV / 2)]));
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            }
            prv = cur;
            cur = nxt;
            nxt = nxt + 1 == RA ? 0 : nxt + 1;
            if (PAIRS && par == 1) {
                wcur = wnxt;
                wnxt = wnxt + 1 == RW ? 0 : wnxt + 1;
            }
        }
    }

    __builtin_amdgcn_s_waitcnt(ring_wait_both(0)); // nothing of the ring is in flight when the epilogue reuses the LDS
    __syncthreads();
    if (!wave_on) return;
    wide_epilogue<Fmt, GATE_UP, MT>(g, t, lds + wave * 16384, acc, col_base);
}

template <typename Fmt, bool GATE_UP>
__global__ __launch_bounds__(kRingWaves * 64, 2) void qgemm_ring_kernel(GemmArgs g) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t ring_lds[];
    Tile t;
    // workgroup -> (tile, strip): an XCD takes every fourth tile of the list and one half of its strips (see qgemm_wide.hip)
    const uint32_t nx = gridDim.x, b = blockIdx.y * nx + blockIdx.x, k = b >> 3, xcd = b & 7u;
    uint32_t slot;
    int strip;
    if (nx % 2u == 0u) {
        const uint32_t half = nx / 2u;
        slot = 4u * (k / half) + (xcd >> 1);
        strip = (int)((xcd & 1u) * half + k % half);
    } else {
        slot = (k / nx) * 8u + xcd;
        strip = (int)(k % nx);
    }
    if (g.tiles) {
        const uint32_t n_tiles = *g.n_tiles;
        t = g.tiles[slot < (uint32_t)g.max_tiles ? slot : 0u];
        if (slot >= n_tiles) return;
        if ((int)t.nrows < g.min_rows || (int)t.nrows > g.max_rows) return; // another launch's tiles
    } else {
        t.expert = 0;
        t.flags = 0;
        t.row0 = slot * (uint32_t)g.tile_m;
        if ((int)t.row0 >= g.dense_rows) return;
        uint32_t left = (uint32_t)g.dense_rows - t.row0;
        t.nrows = left < (uint32_t)g.tile_m ? left : (uint32_t)g.tile_m;
    }
    // the tile is the same for the whole workgroup; saying so keeps the variants apart as scalar branches
    t.expert = (uint32_t)__builtin_amdgcn_readfirstlane((int)t.expert);
    const int mt = __builtin_amdgcn_readfirstlane((int)((t.nrows + 31u) >> 5));
    if (mt <= 1) ring_tile<Fmt, GATE_UP, 1>(g, t, ring_lds, strip);
    else if (mt == 2) ring_tile<Fmt, GATE_UP, 2>(g, t, ring_lds, strip);
    else if (mt == 3) ring_tile<Fmt, GATE_UP, 3>(g, t, ring_lds, strip);
    else if (mt == 4) ring_tile<Fmt, GATE_UP, 4>(g, t, ring_lds, strip);
}

bool qgemm_ring_supports(const QView &b) {
    if (b.packed || b.mode == DMOE_QUANT_NONE || b.cols % 64 != 0 || b.rows % 4 != 0) return false;
    // 32-bit offsets within a matrix, rows of scales (and biases) in whole 16-byte blocks
    if ((uint64_t)b.rows * (uint64_t)b.w_row >= (1ull << 32) || ((uintptr_t)b.w % 16) != 0 || b.w_row % 16 != 0) return false;
    if (b.mode == DMOE_QUANT_FP8_ROW) return true;
    // (whole blocks of entries also mean an even number of steps: a block spans at least four)
    return b.s_row % 16 == 0 && ((uintptr_t)b.scales % 16) == 0 && (!b.biases || ((uintptr_t)b.biases % 16) == 0);
}

template <typename Fmt, bool GATE_UP>
static int ring_raise_limit() {
    static LdsLimit limit; // per instantiation
    return raise_lds_limit(limit, (const void *)qgemm_ring_kernel<Fmt, GATE_UP>, (int)kRingLdsBytes);
}
template <typename Fmt>
static int ring_prepare_format() {
    DMOE_TRY((ring_raise_limit<Fmt, true>()));
    return ring_raise_limit<Fmt, false>();
}
int qgemm_ring_prepare() {
    DMOE_TRY(ring_prepare_format<FmtAffine4>());
    DMOE_TRY(ring_prepare_format<FmtAffine8>());
    DMOE_TRY(ring_prepare_format<FmtMxfp4>());
    return ring_prepare_format<FmtFp8Row>();
}

struct RingLaunch {
    const GemmArgs &g;
    hipStream_t st;
    template <typename Fmt, bool GATE_UP>
    int go() {
        auto kern = qgemm_ring_kernel<Fmt, GATE_UP>;
        DMOE_TRY((ring_raise_limit<Fmt, GATE_UP>())); // done by dmoe_init for its device; a flag test otherwise
        const int cols_per_block = kRingWaves * (GATE_UP ? 32 : 64);
        dim3 grid((unsigned)ceil_div(g.b0.rows, cols_per_block), (unsigned)((g.max_tiles + 7) / 8 * 8)), block(kRingWaves * 64);
        hipLaunchKernelGGL(kern, grid, block, kRingLdsBytes, st, g);
        DMOE_LAUNCH_CHECK();
        return DMOE_OK;
    }
    template <typename Fmt>
    int operator()() {
        return g.gate_up ? go<Fmt, true>() : go<Fmt, false>();
    }
};

int launch_qgemm_ring(const GemmArgs &g, hipStream_t st) {
    DMOE_REQUIRE(qgemm_ring_supports(g.b0) && (!g.gate_up || qgemm_ring_supports(g.b1)),
                 "ring GEMM: unsupported weight format or shape (rows=%d cols=%d)", g.b0.rows, g.b0.cols);
    DMOE_REQUIRE(g.tile_m > 0 && std::min(g.tile_m, g.max_rows) <= kMfmaTileM, "ring GEMM: bad tile size %d", g.tile_m);
    DMOE_REQUIRE(g.max_tiles >= 0 && g.max_tiles <= kRingMaxTiles, "ring GEMM: %d tiles exceed the grid limit", g.max_tiles);
    DMOE_REQUIRE(g.a && g.out && g.ldo > 0 && g.ldo % 4 == 0 && ((uintptr_t)g.out % 8) == 0 && ((uintptr_t)g.a % 16) == 0,
                 "ring GEMM: bad output / activation pointer or pitch");
    if (g.gate_up)
        DMOE_REQUIRE(g.b1.rows == g.b0.rows && g.b1.cols == g.b0.cols && g.b1.mode == g.b0.mode &&
                         g.b1.bits == g.b0.bits && g.b1.group == g.b0.group && g.b1.packed == g.b0.packed,
                     "ring GEMM: gate and up projections differ in shape or format");
    if (g.max_tiles == 0) return DMOE_OK;
    return dispatch_format(g.b0, RingLaunch{g, st});
}

} // namespace dmoe
