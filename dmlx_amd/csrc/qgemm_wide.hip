// Grouped quantized GEMM, wide MFMA path (prefill, every quantized format in the packed resident layout).
//
// One workgroup (4 wavefronts) = one tile of up to 128 rows of ONE expert segment against a strip of output columns;
// each wavefront dequantizes its own 64 weight rows straight into the A operand of v_mfma_f32_32x32x16_bf16 and
// holds 128 x 64 f32 accumulators. The kernel is built so that TWO workgroups fit a compute unit (at most 256
// registers per wavefront, 64 KiB of LDS): a lone wavefront on a SIMD issues a vector instruction only every ~5
// cycles, two wavefronts every ~2.8, and the 4-bit decode (2.1 vector instructions per weight) is the largest
// item beside the MFMAs. A variant with 256-row tiles (every decoded fragment feeds eight MFMAs instead of four, but one
// wavefront per SIMD: all 512 registers, 128 KiB of LDS) measured 5 % slower on the 8k-token ragged prefill.
// The 8-bit formats run the same loop with two 16-byte chunk steps per 64-element step. Differences from the
// MLX-layout kernel in qgemm_mfma.hip:
//
//  * Activations go from global memory into LDS without passing through registers (global_load_lds_dwordx4).
//    One such instruction moves 1 KiB: 8 rows x 128 bytes (one reduction step of 64 bf16). Inside that KiB the
//    16-byte pieces of row r are stored at position piece ^ ((r >> 1) & 7). The LDS serves a 16-byte read
//    instruction 16 lanes (256 bytes, all 64 banks) per cycle, and a lane's place among the banks is
//    (row & 1) * 8 + position: rows 2q and 2q + 1 differ in the first term, the eight row pairs of a 16-lane group in
//    the second, so the MFMA operand reads (32 rows at the same reduction offset) run at the full 256 bytes per
//    cycle (position piece ^ (r & 7) made rows r and r + 8 collide: 155 bytes per cycle measured). The swizzle
//    costs nothing because each lane picks its global source address freely.
//  * A ring of LDS buffers of one reduction step each: while step s computes, the loads of the next steps are in flight.
//    The compiler does not know about these loads (they are issued from inline assembly), so their completion is
//    tracked by hand: VMEM operations return in order, hence "at most N operations outstanding" three quarters into
//    step s, with N = what has been issued since the loads of step s + 1, implies that these have landed. One s_barrier
//    per step then publishes the buffer.
//  * The same in-order rule ties the two streams together: a wait for a weight chunk also waits for every older staging
//    request and the other way round, so that only looking ahead further with BOTH helps. Tiles of at most 64 rows have
//    the room (64 or 96 accumulator registers less, LDS buffers of 4 or 8 KiB instead of 16), and on the 4-bit formats they
//    use it: a step of theirs is 8 or 16 matrix instructions long, a memory round trip as long as several, so they keep
//    four steps of weights and four blocks of activations in flight. Eight of either measured level on a full chip and
//    slower on a small one; the 8-bit and unquantized formats, whose steps bring two and four times the bytes, gained
//    nothing. 256 experts, one projection [2048, 4096], with 32 / 64 rows each, two steps of weights -> this: 4-bit affine
//    322 / 357 -> 282 / 337 us, MXFP4 250 / 290 -> 217 / 281; 8 experts [1536, 3072]: MXFP4 20.7 / 26.9 -> 18.3 / 24.4.
//  * Such a tile is often its expert's only one, whose weights nobody else reads: see kWideStreamBytes.
//  * Rows past the end of a tile are zeros in LDS and never requested: the chip is power-limited here, and multiplying
//    zeros costs less of it than multiplying copies of a row (33 rows per expert: MXFP4 263 -> 251 us, 4-bit affine 324 ->
//    311, 65 and 97 rows 1 to 3 %).
//  * Activation fragments are single-buffered (except for tiles of at most 64 rows): the fragment of row tile mt
//    is reloaded for the next MFMA group right after its last use in this one, 2*MT-1 units before it is needed
//    again.
//
// The reduction loop is software-pipelined like the other MFMA kernel: units of [one MFMA | a slice of the decode
// of the next step's weights] separated by scheduling barriers.
#include <type_traits>

#include "common.h"
#include "qformat.h"
#include "wide_epilogue.h"

namespace dmoe {

constexpr int kWideWaves = 4;
constexpr size_t kWideLdsBytes = 65536;   // two workgroups per compute unit

// Pipeline depths of a tile of MT row blocks of 32.
template <typename Fmt, int MT>
struct WidePipe {
    static constexpr bool kDeep = Fmt::kVals == 32 && MT <= 2;
    static constexpr int kSlots = MT <= 2 ? 8 : 4; // LDS activation buffers
    static constexpr int kAhead = kDeep ? 4 : MT <= 2 ? 3 : 2; // blocks of activations in flight ahead of the one being computed
    static constexpr int kWeights = kDeep ? 4 : Fmt::kVals == 8 ? 1 : 2; // steps of weights held in registers
    // the loop runs whole trips (surplus steps multiply zeros), or ends behind the last step
    // (leaving in mid-trip costs the larger tiles the registers they do not have)
    static constexpr bool kWholeTrips = MT > 2;
};

// s_waitcnt immediates (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt_hi[15:14])
constexpr int wait_vmcnt(int n) { return 0x0f70 | (n & 15) | ((n >> 4) << 14); }
constexpr int wait_vmcnt_lgkm0(int n) { return 0x0070 | (n & 15) | ((n >> 4) << 14); }
// the same for a count that is a constant only once the loops around it are unrolled
__device__ __forceinline__ void wait_vmcnt_at_most(int n) {
#define DMOE_WAIT(N) case N: __builtin_amdgcn_s_waitcnt(wait_vmcnt(N)); break;
#define DMOE_WAIT8(N) DMOE_WAIT(N) DMOE_WAIT(N + 1) DMOE_WAIT(N + 2) DMOE_WAIT(N + 3) DMOE_WAIT(N + 4) DMOE_WAIT(N + 5) DMOE_WAIT(N + 6) DMOE_WAIT(N + 7)
    switch (n) {
        DMOE_WAIT8(0) DMOE_WAIT8(8) DMOE_WAIT8(16) DMOE_WAIT8(24) DMOE_WAIT8(32) DMOE_WAIT8(40) DMOE_WAIT8(48) DMOE_WAIT8(56)
    default: __builtin_amdgcn_s_waitcnt(wait_vmcnt(63)); // the counter's largest value
    }
#undef DMOE_WAIT8
#undef DMOE_WAIT
}
constexpr int kWaitLgkm0 = 0xc07f;

template <typename Fmt, bool GATE_UP, int MT, bool STREAM = false>
__device__ __forceinline__ void wide_tile(const GemmArgs &g, const Tile &t, uint8_t *lds, const int strip) {
    using CS = ChunkStream<Fmt, true>;
    // A step is 64 reduction elements = one 128-byte activation granule. A lane's 16-byte weight chunk holds 32 (4-bit
    // formats) or 16 (8-bit formats) of them: the weights come in chunk steps of 2 * KV elements, CH of them per step,
    // and ring, decode and the double-buffered decoded operands advance by chunk steps.
    constexpr int KV = Fmt::kVals, KSTEP = 64, NJ = 4, NT = 2;
    constexpr int CH = 32 / KV;           // chunk steps per step
    static_assert(CH == 1 || CH == 2 || CH == 4, "chunks of 32, 16 or 8 values");
    constexpr int NJC = NJ / CH;          // MFMA groups per chunk step
    constexpr int NUC = NJC * MT * NT;    // units (MFMAs) per chunk step
    constexpr int NPC = NT * (KV / 2);    // packed pairs to decode per chunk step
    using P = WidePipe<Fmt, MT>;
    constexpr int TRIP = 4, SLOTS = P::kSlots, AHEAD = P::kAhead, WR = P::kWeights, WRC = WR * CH; // (WRC: chunk steps held in registers)
    constexpr bool WHOLE = P::kWholeTrips;
    constexpr int BUF = MT * 4096; // one LDS slot: one reduction step (64 bf16) of every row of the tile
    static_assert(TRIP % WR == 0 && (TRIP * CH) % 2 == 0 && (SLOTS == TRIP || SLOTS == 2 * TRIP), "ring slots must line up across trips");
    static_assert(SLOTS * BUF <= (int)kWideLdsBytes && SLOTS >= AHEAD + 2, "a slot is refilled two barriers after its last read");
    const int tid = (int)threadIdx.x, lane = tid & 63, ln = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cols = g.b0.cols, n_out = g.b0.rows;
    const int n_steps = cols / KSTEP, n_csteps = n_steps * CH;
    const size_t e = t.expert;

    // ---- this wavefront's weight rows (gate_up: tile 0 = gate, tile 1 = up rows of the same 32 columns) ----
    const int col_base = (strip * kWideWaves + wave) * (GATE_UP ? 32 : 64);
    const bool wave_on = col_base < n_out;
    CS cs[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const QView &b = (GATE_UP && nt == 1) ? g.b1 : g.b0;
        const int base = GATE_UP ? col_base : col_base + 32 * nt;
        const bool on = wave_on && base < n_out;
        int n = base + ln;
        if (n >= n_out) n = n_out - 1;
        cs[nt].init(b, e, (on ? base : 0) >> 5, ln, h, n); // a switched-off tile aliases valid memory, never stored
    }
    // Loads with a scalar base for the larger tiles and for MXFP4; in the small tiles of the other formats the scalar additions in front
    // of each load are on the path of a launch that is one round of workgroups (us per step, vector | scalar: 8 experts, hidden 3072,
    // ffn 768, 33 tokens top-4 8-bit 56.4 | 59.2, 80 tokens top-2 4-bit 64.4 | 67.8; 1531 tokens MXFP4 908 | 900).
    constexpr bool SCALAR = MT > 2 || Fmt::kMetaEntryBytes == 1;
    uint4 ring_raw[WRC][NT];
    uint32_t ring_sb[WRC][NT][2];
    auto load_b = [&](int cstep, int slot_) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const QView &b = (GATE_UP && nt == 1) ? g.b1 : g.b0;
            if constexpr (SCALAR) {
                ring_raw[slot_][nt] = cs[nt].template load_chunk_scalar<STREAM>(cstep);
                cs[nt].load_meta_scalar(b, cstep, ring_sb[slot_][nt]);
            } else {
                ring_raw[slot_][nt] = STREAM ? cs[nt].load_chunk_stream(cstep) : cs[nt].load_chunk(cstep);
                cs[nt].load_meta(b, cstep, ring_sb[slot_][nt]);
            }
        }
    };

    // ---- activation staging -------------------------------------------------------------------------------
    // operation i of this wavefront moves rows (wave + 4 i) * 8 .. + 7; lane = (row r8 of the eight, position c),
    // and fetches piece c ^ ((row >> 1) & 7) of its row. Rows past the segment end: see last_on.
    const int r8 = lane >> 3, c = lane & 7;
    const uint8_t *a_src[MT];
    uint32_t a_row[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int r = (wave + 4 * i) * 8 + r8;
        a_row[i] = t.row0 + (uint32_t)(r < (int)t.nrows ? r : 0);
    }
    if (g.a_rows) { // (requested ahead of the weights: loads return in order)
#pragma unroll
        for (int i = 0; i < MT; ++i) a_row[i] = g.a_rows[a_row[i]];
    }
    // (the first step of weights follows; the rest of the ring: see the prologue)
    auto load_step = [&](int step) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int cstep = step * CH + c;
            load_b(cstep < n_csteps ? cstep : n_csteps - 1, cstep);
            asm volatile("" ::: "memory"); // every load stays one of its own: they are counted below
        }
    };
    constexpr int WR0 = P::kDeep ? 1 : WR;
#pragma unroll
    for (int j = 0; j < WR0; ++j) load_step(j);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int r = (wave + 4 * i) * 8 + r8;
        const size_t src = a_row[i];
        a_src[i] = (const uint8_t *)(g.a + src * (size_t)cols) + ((c ^ (((r >> 1) & 7))) * 16);
    }
    // Only the last operation can hold rows past the segment end. Their lanes request nothing, and their places in the
    // buffers are zeroed here, once. (A wavefront whose last operation has no row at all still requests one lane's piece,
    // of the tile's first row, so that every operation counts as one in the waits below.)
    const bool last_on = (wave + 4 * (MT - 1)) * 8 + r8 < (int)t.nrows;
    const uint64_t last_lanes = __ballot(last_on), last_mask = last_lanes ? last_lanes : 1ull;
    if (!last_on) {
#pragma unroll
        for (int b = 0; b < SLOTS; ++b) *(uint4 *)(lds + b * BUF + (wave + 4 * (MT - 1)) * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
    }
    const uint32_t lds_addr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    auto stage_op = [&](int blk, int buf, int i) {
        const uint8_t *gp = a_src[i] + (size_t)blk * 128;
        const uint32_t la = lds_addr + (uint32_t)(buf * BUF + (wave + 4 * i) * 1024); // uniform
        // (a wait state between the write of M0 and the request that reads it; nothing else in this kernel uses M0)
        if (i < MT - 1)
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(gp), "s"(la) : "memory");
        else
            asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 exec, %2\n\tglobal_load_lds_dwordx4 %0, off\n\ts_mov_b64 exec, -1"
                         : : "v"(gp), "s"(la), "s"(last_mask) : "memory"); // (control flow is uniform: every lane is on)
    };
    // surplus steps of the last trip (WHOLE, n_steps not a multiple of the trip) must multiply zeros
    const int n_whole = (n_steps + TRIP - 1) / TRIP * TRIP;
    auto zero_block = [&](int buf) {
#pragma unroll
        for (int i = 0; i < MT; ++i) *(uint4 *)(lds + buf * BUF + (wave + 4 * i) * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
        __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
    };

    f32x16_t acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.0f;

    uint32_t wp[2][NT][KV / 2]; // decoded weights of the current / next step
    // activation fragment of each row tile for the current MFMA group; small tiles have registers to spare and too
    // few units per group to hide an LDS round trip, so they keep a second set and fetch a whole group ahead
    constexpr int XB = MT <= 2 ? 2 : 1;
    bf16x8_t xf[XB][MT];
    // fragment (mt, j) of a step: row mt * 32 + ln, the piece that holds this lane's eight reduction elements of MFMA
    // group j (chunk step c = j / NJC of the step, elements (2 c + h) * KV + 8 (j % NJC) onwards), stored at
    // piece ^ ((row >> 1) & 7)
    uint32_t x_rd[NJ]; // (offset in LDS)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int piece = ((2 * (j / NJC) + h) * KV + 8 * (j % NJC)) >> 3;
        x_rd[j] = (uint32_t)((ln >> 3) * 1024 + (ln & 7) * 128 + ((piece ^ ((ln >> 1) & 7)) * 16));
    }
    // SLOTS = 2 * TRIP: the trips alternate between the halves of the ring; x_rd points into the trip's own half
    constexpr uint32_t HALF = TRIP * BUF;
    auto read_x = [&](int buf, int j, int mt, bool next_trip = false) {
        const uint32_t at = SLOTS == TRIP || !next_trip ? x_rd[j] : x_rd[j] ^ HALF;
        xf[j % XB][mt] = __builtin_bit_cast(bf16x8_t, *(const uint4 *)(lds + at + buf * BUF + mt * 4096));
    };

    // ---- prologue: the first AHEAD blocks, first decode ----------------------------------------------------------
    // Activations and weights in the order of their use, so that the first step waits for its own data only: a launch starts
    // with all of its workgroups at this point, and everybody's full rings are 10 us worth of the chip's bandwidth.
    constexpr int LOADS = CH * NT * (Fmt::kMetaEntryBytes ? 2 : 1); // loads of one step of weights
#pragma unroll
    for (int b = 0; b < AHEAD || b + WR0 < WR; ++b) {
        if (b < AHEAD && b < n_steps) {
#pragma unroll
            for (int i = 0; i < MT; ++i) stage_op(b, b, i);
        } else if (WHOLE && b < AHEAD) {
            zero_block(b);
        }
        if (b + WR0 < WR) load_step(b + WR0);
    }
    // block 0, and the zeros
    if (n_steps >= AHEAD) __builtin_amdgcn_s_waitcnt(wait_vmcnt_lgkm0((AHEAD - 1) * MT + (WR - WR0) * LOADS));
    else __builtin_amdgcn_s_waitcnt(wait_vmcnt_lgkm0(0));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) Fmt::decode_fast(ring_raw[0][nt], CS::meta(ring_sb[0][nt]), wp[0][nt]);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) read_x(0, 0, mt);

    // Step j of a trip computes from slot j, requests block s + AHEAD into slot (j + AHEAD) % SLOTS during its first three
    // MFMA groups, and at the start of the fourth waits for block s + 1 and synchronises, so that the first fragments of
    // the next step can be fetched during that last group.
    bool more = true;
#pragma unroll 1
    for (int s0 = 0; more; s0 += TRIP) {
#pragma unroll
        for (int j = 0; j < TRIP; ++j) {
            const int s = s0 + j;
            const bool stage = s + AHEAD < n_steps; // uniform
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int ci = j * CH + c; // chunk step within the trip
                const int cs_ahead = s * CH + c + WRC < n_csteps ? s * CH + c + WRC : n_csteps - 1;
                load_b(cs_ahead, ci % WRC); // this slot was decoded one chunk step ago
                asm volatile("" ::: "memory"); // every load stays one of its own: they are counted below
                const int slot_next = (ci + 1) % WRC, which = ci & 1;
                Meta meta_next[NT];
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) meta_next[nt] = Fmt::pair_meta(CS::meta(ring_sb[slot_next][nt]));
                uint32_t dstate[Fmt::kPairState] = {};
                Fmt::pair_state(dstate);
#pragma unroll
                for (int jc = 0; jc < NJC; ++jc) {
                    const int jj = c * NJC + jc; // MFMA group within the step
                    if (jj == NJ - 1) {
                        // Block s + 1 must have landed. Younger than its requests are those of the AHEAD - 1 blocks
                        // behind it (near the end of the reduction there are fewer: none is counted on) and the loads
                        // of the weight chunks (and their scales) of the steps since then: AHEAD - 1 steps' worth, in the
                        // first trip those of the prologue's and the loop's that follow it.
                        constexpr int REQS = (AHEAD - 1) * MT, later = (AHEAD - 1) * LOADS;
                        const int since = j + 1 > WR - WR0 ? j + 1 : WR - WR0, first = since < AHEAD - 1 ? since * LOADS : later;
                        const bool in_first = first < later && s0 == 0;
                        if (in_first) wait_vmcnt_at_most(first);
                        else if (stage) wait_vmcnt_at_most(REQS + later);
                        else wait_vmcnt_at_most(later);
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_s_barrier();
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt) {
                            const int uc = (jc * MT + mt) * NT + nt; // unit within the chunk step
                            const int u = c * NUC + uc;              // unit within the step
                            uint4 q = make_uint4(wp[which][nt][4 * jc], wp[which][nt][4 * jc + 1], wp[which][nt][4 * jc + 2],
                                                 wp[which][nt][4 * jc + 3]);
                            acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, q),
                                                                                  xf[jj % XB][mt], acc[mt][nt], 0, 0, 0);
                            // fetch the fragment of the next group: after the last use of this one (one register set),
                            // or at the first (two sets)
                            if (nt == (XB == 1 ? NT - 1 : 0)) {
                                if (jj + 1 < NJ) read_x(j, jj + 1, mt);
                                else read_x((j + 1) % TRIP, 0, mt, j == TRIP - 1);
                            }
                            if (u % 6 == 0 && u / 6 < MT) { // the staging requests all fall into the first three groups
                                if (stage) stage_op(s + AHEAD, (s + AHEAD) % SLOTS, u / 6);
                            }
#pragma unroll
                            for (int p = uc * NPC / NUC; p < (uc + 1) * NPC / NUC; ++p) {
                                Fmt::decode_pair(ring_raw[slot_next][p / (KV / 2)], meta_next[p / (KV / 2)], p % (KV / 2),
                                                 wp[which ^ 1][p / (KV / 2)], dstate);
                                // pin the slice here (the optimiser would sink a trip's last decode into the next trip)
                                asm volatile("" : "+v"(wp[which ^ 1][p / (KV / 2)][p % (KV / 2)]));
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            }
            if (WHOLE) {
                if (!stage && s + AHEAD < n_whole) zero_block((s + AHEAD) % SLOTS); // a surplus step: zeros
                if (j == TRIP - 1) more = s + 1 < n_whole;
            } else if (s + 1 >= n_steps) { // uniform
                more = false;
                break;
            }
        }
        if (SLOTS != TRIP) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) x_rd[j] ^= HALF;
        }
    }

    // ---- epilogue: the activation ring is free once every wavefront has left the loop; each uses its own 16 KiB --------
    __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
    __syncthreads();
    if (!wave_on) return;
    wide_epilogue<Fmt, GATE_UP, MT>(g, t, lds + wave * (kWideLdsBytes / kWideWaves), acc, col_base);
}

// Consecutive tiles whose workgroups for one column strip start back to back on one XCD. Unquantized weights: a tile of 128
// rows does 128 flops per byte of weights, so experts of several tiles are bound by fetching their weights through the L2s
// again for every tile (256 rows per expert: 0.83 PFLOP/s x 1 byte / 128 flops = 6.5 TB/s). With runs of four the second to
// fourth workgroup of a strip find the weights in their L2: one projection [256, 2048, 4096], 256 / 512 rows per expert 1321 /
// 2533 -> 1139 / 1978 us; a step of 8192 tokens, Zipf-skewed, 3379 -> 3076 us. Not where most experts have one tile (128 rows
// each: 831 -> 844 us), and not the last tiles of a list that make no whole group: four of them would go to one XCD pair. The
// quantized formats stay at one: 2080 tokens on 8-bit experts +1.5 %, 8192 tokens on 4-bit ones +5 %.
template <typename Fmt>
__host__ __device__ constexpr uint32_t wide_run() {
    return Fmt::kVals == 8 ? 4u : 1u;
}

// Experts of several tiles: an eighth more tiles than live experts. The dense tiles of a shared expert in the list count on
// neither side, so that the choice is the routing's alone.
__host__ __device__ constexpr bool wide_several_tiles(uint32_t tiles, uint32_t dense_tiles, uint32_t live) {
    return 8u * (tiles - dense_tiles) >= 9u * live;
}
static_assert(!wide_several_tiles(64, 0, 64) && !wide_several_tiles(64 + 8, 8, 64) && wide_several_tiles(72, 0, 64) && wide_several_tiles(72 + 64, 64, 64),
              "the same choice with and without a shared expert in the list");

template <typename Fmt, bool GATE_UP>
__global__ __launch_bounds__(kWideWaves * 64, 2) void qgemm_wide_kernel(GemmArgs g) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t wide_lds[]; // [slots][rows of the tile][128 bytes], swizzled
    constexpr uint32_t RUN = wide_run<Fmt>();
    // Workgroups go to the eight XCDs round-robin in launch order; gridDim.y is a multiple of 8, which makes the maps
    // below permutations of the grid. XCD x = (tile class x / 2, strip half x % 2): it takes every fourth tile of the
    // list and one half of the tile's column strips, a tile's strips back to back. A tile's activations then enter two
    // L2s instead of eight, and consecutive tiles of an expert find the half of its weights they need in the L2 they
    // run on. Same box, against all strips of a tile on one XCD (the map before, kept for strip counts that are odd):
    // C3 step -0.7 % (down launch -1.6 %), C4 step -1.7 % (gate/up launch -2.4 %); four strip groups x two tile classes
    // -0.6 % / -1.3 %, eight strip groups (an XCD = two strips of every tile) +0.8 % / -0.9 %. (Giving an XCD runs of
    // 2..16 consecutive tiles with ALL their strips, so that the tiles of an expert could share its weights through
    // that L2, measured 0.5 % to 15 % slower the longer the run: an expert's weights do not fit one L2.)
    const uint32_t nx = gridDim.x, b = blockIdx.y * nx + blockIdx.x, k = b >> 3, xcd = b & 7u;
    uint32_t slot, n_slots, run = 1;
    bool stream = false; // weight loads with the streaming hint
    if (g.tiles) {
        n_slots = *g.n_tiles;
        if (g.n_live) {
            const bool shared = wide_several_tiles(n_slots, (uint32_t)g.dense_tiles, *g.n_live);
            run = shared ? RUN : 1u;
            stream = g.stream_weights && !shared;
        }
    } else {
        n_slots = (uint32_t)((g.dense_rows + g.tile_m - 1) / g.tile_m);
        run = RUN;
    }
    int strip;
    if (nx % 2u == 0u) {
        const uint32_t half = nx / 2u, group = k / (RUN * half), r = k % (RUN * half); // a group: 4 * RUN tiles (fewer at the grid's end)
        if (run > 1u && (group + 1u) * 4u * RUN <= n_slots) {
            slot = 4u * RUN * group + RUN * (xcd >> 1) + r % RUN;
            strip = (int)((xcd & 1u) * half + r / RUN);
        } else {
            slot = 4u * (RUN * group + r / half) + (xcd >> 1);
            strip = (int)((xcd & 1u) * half + r % half);
        }
    } else {
        slot = (k / nx) * 8u + xcd;
        strip = (int)(k % nx);
    }
    Tile t;
    if (g.tiles) {
        t = g.tiles[slot < (uint32_t)g.max_tiles ? slot : 0u];
        if (slot >= n_slots) return;
        if ((int)t.nrows < g.min_rows) return; // left to the weight-streaming kernel
    } else {
        t.expert = 0;
        t.flags = 0;
        t.row0 = slot * (uint32_t)g.tile_m;
        if ((int)t.row0 >= g.dense_rows) return;
        uint32_t left = (uint32_t)g.dense_rows - t.row0;
        t.nrows = left < (uint32_t)g.tile_m ? left : (uint32_t)g.tile_m;
    }
    // the tile is the same for the whole workgroup; saying so keeps the variants apart as scalar branches
    const int mt = __builtin_amdgcn_readfirstlane((int)((t.nrows + 31u) >> 5));
    if (mt <= 1) stream ? wide_tile<Fmt, GATE_UP, 1, true>(g, t, wide_lds, strip) : wide_tile<Fmt, GATE_UP, 1>(g, t, wide_lds, strip);
    else if (mt == 2) stream ? wide_tile<Fmt, GATE_UP, 2, true>(g, t, wide_lds, strip) : wide_tile<Fmt, GATE_UP, 2>(g, t, wide_lds, strip);
    else if (mt == 3) wide_tile<Fmt, GATE_UP, 3>(g, t, wide_lds, strip);
    else if (mt == 4) wide_tile<Fmt, GATE_UP, 4>(g, t, wide_lds, strip);
}

bool qgemm_wide_supports(const QView &b) {
    return b.mode != DMOE_QUANT_NONE && b.packed && b.cols % 64 == 0 && b.rows % 4 == 0;
}

template <typename Fmt, bool GATE_UP>
static int wide_raise_limit() {
    static LdsLimit limit; // per instantiation
    return raise_lds_limit(limit, (const void *)qgemm_wide_kernel<Fmt, GATE_UP>, (int)kWideLdsBytes);
}
template <typename Fmt>
static int wide_prepare_format() {
    DMOE_TRY((wide_raise_limit<Fmt, true>()));
    return wide_raise_limit<Fmt, false>();
}
int qgemm_wide_prepare() {
    DMOE_TRY(wide_prepare_format<FmtBf16>());
    DMOE_TRY(wide_prepare_format<FmtAffine4>());
    DMOE_TRY(wide_prepare_format<FmtAffine8>());
    DMOE_TRY(wide_prepare_format<FmtMxfp4>());
    return wide_prepare_format<FmtFp8Row>();
}

// Weight loads of tiles of at most 64 rows carry the streaming hint where most experts have one tile and the launch's
// weights are more than the memory-side cache holds, so that neither a second tile nor the next step would find them there
// (256 experts, one projection [2048, 4096], 32 / 64 rows each, us without -> with: 8-bit 430 / 458 -> 396 / 431, bf16 765 / 780
// -> 690 / 712, MXFP4 231 / 290 -> 217 / 281). Without that rule: 8 experts top-4, hidden 3072, ffn 768, bf16, 324 tokens 79 -> 95
// us per step, 64 experts top-6, hidden 1536, ffn 768, 8-bit, 1548 tokens (145 rows per expert) 168 -> 175.
constexpr size_t kWideStreamBytes = (size_t)256 << 20;

template <typename Fmt, bool GATE_UP>
static int launch_wide(const GemmArgs &g, hipStream_t st) {
    auto kern = qgemm_wide_kernel<Fmt, GATE_UP>;
    DMOE_TRY((wide_raise_limit<Fmt, GATE_UP>())); // done by dmoe_init for its device; a flag test otherwise
    const int cols_per_block = kWideWaves * (GATE_UP ? 32 : 64);
    dim3 grid((unsigned)ceil_div(g.b0.rows, cols_per_block), (unsigned)((g.max_tiles + 7) / 8 * 8)), block(kWideWaves * 64);
    GemmArgs a = g;
    a.stream_weights = (size_t)g.b0.n_mats * (g.gate_up ? 2 : 1) * (g.b0.w_mat + g.b0.m_mat) > kWideStreamBytes;
    hipLaunchKernelGGL(kern, grid, block, kWideLdsBytes, st, a);
    DMOE_LAUNCH_CHECK();
    return DMOE_OK;
}

bool qgemm_wide_bf16_supports(const QView &b) {
    return b.mode == DMOE_QUANT_NONE && b.packed && b.cols % 64 == 0 && b.rows % 32 == 0 && ((uintptr_t)b.w % 16) == 0;
}

int launch_qgemm_wide(const GemmArgs &g, hipStream_t st) {
    DMOE_REQUIRE(qgemm_wide_supports(g.b0) || qgemm_wide_bf16_supports(g.b0),
                 "wide MFMA GEMM: unsupported weight format or shape (rows=%d cols=%d)", g.b0.rows, g.b0.cols);
    DMOE_REQUIRE(g.tile_m > 0 && g.tile_m <= kMfmaWideTileM && g.tile_m % 32 == 0, "wide MFMA GEMM: bad tile size %d",
                 g.tile_m);
    DMOE_REQUIRE(g.max_tiles >= 0 && g.max_tiles <= 65528, "wide MFMA GEMM: %d tiles exceed the grid limit", g.max_tiles);
    DMOE_REQUIRE(g.a && g.out && g.ldo > 0 && g.ldo % 4 == 0 && ((uintptr_t)g.out % 8) == 0 &&
                     ((uintptr_t)g.a % 16) == 0,
                 "wide MFMA GEMM: bad output / activation pointer or pitch");
    if (g.gate_up)
        DMOE_REQUIRE(g.b1.rows == g.b0.rows && g.b1.cols == g.b0.cols && g.b1.mode == g.b0.mode &&
                         g.b1.bits == g.b0.bits && g.b1.group == g.b0.group && g.b1.packed == g.b0.packed,
                     "wide MFMA GEMM: gate and up projections differ in shape or format");
    if (g.max_tiles == 0) return DMOE_OK;
    if (g.b0.mode == DMOE_QUANT_NONE)
        return g.gate_up ? launch_wide<FmtBf16, true>(g, st) : launch_wide<FmtBf16, false>(g, st);
    if (g.b0.mode == DMOE_QUANT_MXFP4)
        return g.gate_up ? launch_wide<FmtMxfp4, true>(g, st) : launch_wide<FmtMxfp4, false>(g, st);
    if (g.b0.mode == DMOE_QUANT_FP8_ROW)
        return g.gate_up ? launch_wide<FmtFp8Row, true>(g, st) : launch_wide<FmtFp8Row, false>(g, st);
    if (g.b0.bits == 8)
        return g.gate_up ? launch_wide<FmtAffine8, true>(g, st) : launch_wide<FmtAffine8, false>(g, st);
    return g.gate_up ? launch_wide<FmtAffine4, true>(g, st) : launch_wide<FmtAffine4, false>(g, st);
}

} // namespace dmoe
