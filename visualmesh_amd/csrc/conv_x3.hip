/*
 * conv_x3.hip - 64 -> 64 graph-convolution layers of the fp32 engine on the bf16 matrix instructions, with every fp32 factor
 * split into three bf16 parts: neighbour gather + dense + bias + activation in one kernel (reference engine/cpu/engine.hpp:213-264,
 * apply_activation.hpp:34-84).
 *
 * Arithmetic. x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m) holds exactly for every float above 2^-97 (three
 * times eight bits, and the signs, cover the 24 of a float; below, the parts leave bf16's normal range one after the other and at most
 * 2^-118 is lost). A product x w is the sum of nine exact products of parts; six of them are computed, what is dropped (m l, l m, l l) is
 * 2^-25 of a product and of either sign. The products of the high parts have an accumulator of their own and the five small ones
 * another, so that the many small terms meet no large partial sum. Against 64 bits, over sums of 112 to 448 products of normal,
 * selu, relu and tanh inputs, the result is 2.6 to 4 times closer than the chain of v_mfma_f32_16x16x4_f32 (relative 5.3e-8 to 1.1e-7,
 * there 1.4e-7 to 3.8e-7): a chain of 28 roundings instead of 112. The parts of an infinity or a NaN are not the value's, so the
 * engine takes this kernel only for networks in which no activation can reach 1e30, by the weights (api.hip).
 * Six bf16 instructions do the work of sixteen fp32 ones: six times 32 cycles for 32 x 32 x 16 products against 512.
 *
 * Instruction: v_mfma_f32_32x32x16_bf16, a 32 (output channels) x 32 (rows) block over 16 values of the reduction index.
 *   A operand: lane l supplies W[k(l / 32, e)][o = l % 32], e = 0..7     (weights)
 *   B operand: lane l supplies in[src(row = l % 32)][k(l / 32, e)]        (gathered rows)
 *   D:         lane l holds, for row l % 32, channels 8 * g + 4 * (l / 32) + {0..3}, g = 0..3
 *
 * Where things live. A block is four waves, one per SIMD, and works on a half tile (128 rows) in stages of 32 input channels. The weights as
 * three parts, 172 KB, stay with a persistent block: wave (cb, rw) holds those of its 32 output channels in registers, but for the low
 * parts of the last three slots, 24 KB, which lie in LDS, and works on the 64 rows of row half rw in two blocks of 32. A stage's
 * rows, the half tile's own and up to 128 of other half tiles (conv_bf16.hip's tables), arrive in LDS as fp32 by buffer_load ... lds, are
 * split once and lie there as three planes of bf16 while the stage before is worked on: the next stage's planes are written while this
 * one's are read, and the places the rows arrived in are requested again as they are emptied. Every wave splits what it has
 * brought in itself, so that a stage needs one barrier. (Splitting at every use instead, in the registers of the lane that
 * gathers, is seven times the vector work: 665 us for 1.85 million rows where this took 590. Rows stored as parts would be 384 bytes
 * instead of 256 in memory.)
 *
 * Schedule. A wave issues in order and a matrix instruction keeps its pipe busy for 32 cycles, of which it takes 4 to issue: behind every
 * second one comes a piece of side work of at most what fits (splitting, loads, then activation and stores of the half tile before), behind
 * others the reads of the operands to come. Every load and store of the loop is issued unconditionally (out-of-range offsets move
 * nothing) so that the waits can count them.
 *
 * Half tiles with more than 128 halo rows are computed again from memory at the end of the kernel, with the same parts, instructions and
 * order, so that it does not show in the results which rows were staged.
 *
 * What bounds it: the matrix pipe at the clock that power leaves it. It is busy for 65 % of the cycles, which pass at 1.7 GHz where
 * kernels bound by memory run at 2.4 and those of fp32 products at 2.2. A launch by rocprofv3's trace, fp32 products / so: 29.1 million
 * rows 13.5 / 8.7 ms, 1.85 million 924 / 559 us. By size, a network 3-64-64-4 on fp32 products / so, us a pass: 4 000 rows 86 / 70, 36 000 99 / 94, 65 000 113 / 107, 130 000
 * 155 / 134, 520 000 429 / 331; with three such layers 162 / 97, 191 / 154, 212 / 173, 311 / 236, 937 / 634.
 */
#include <atomic>

#include "conv_x3.h"

namespace {

constexpr int BT = VMHIP_HTILE;   /* rows of a half tile */
constexpr int BH = VMHIP_HHALO;   /* halo rows staged beside them */
constexpr int BROWS = BT + BH;    /* LDS rows per buffer */
constexpr int NOTE = VMHIP_NOTE_WORDS;
constexpr int C = 64, SLOTS = 7, NN = SLOTS - 1;  /* the shape: C -> C channels */
constexpr int ROWB = C * 4;                       /* bytes of a row */
constexpr int SC = 32, STAGES = C / SC;           /* channels of a stage, stages of a half tile */
constexpr int CHUNKS = SLOTS * 2;                 /* steps of 16 values of a stage */
constexpr int CBW = C / 32;                       /* waves that share a row */
constexpr int RB = CBW;                           /* blocks of 32 rows of a wave: 128 rows over 4 / CBW waves; a stage finishes one */
constexpr int PER = 6 * RB;                       /* matrix instructions of a step */
constexpr int PART = BROWS * SC * 2;              /* one part of a stage's rows */
constexpr int PLANES = 3 * PART;
constexpr int LANDING = BROWS * SC * 4;           /* a stage's rows as they arrive */
constexpr int NBL = 64 * 16;                      /* a wave's rows of the neighbour table */
constexpr int GROUPS = BROWS / 16 / 4;            /* groups of 16 rows that a wave brings in and splits */
constexpr int PIECES = 14;                        /* ... in so many pieces of side work each */
constexpr int N_SLICES = 20;                      /* of a finished row block: 16 activations, 4 stores */
constexpr int N_STORES = 4;
constexpr int LOW_SLOTS = 3, LOW_FROM = SLOTS - LOW_SLOTS; /* the last slots, whose weights' low parts lie in LDS: the registers do not hold them all */
constexpr size_t LDS_BYTES = 2 * PLANES + LANDING + 4 * NBL + 4 * NOTE * 4 + C * 4 + size_t(LOW_SLOTS) * (C / 16) * CBW * 1024;
static_assert(NN <= VMHIP_NBL_STRIDE, "the half-tile neighbour table holds 8 entries per row");
static_assert(STAGES == RB, "a stage finishes one row block");
static_assert(LDS_BYTES <= 160 * 1024, "the block must fit the CU's LDS");

template <int ACT>
__global__ __launch_bounds__(256) void vm_conv_x3_kernel(VmBatchDev B, VmLayerDev L, const float* __restrict__ in, float* __restrict__ out) {
    extern __shared__ float4 lds4[];
    char* const lds = reinterpret_cast<char*>(lds4);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
    const int cb = wave % CBW, rw = wave / CBW;
    const int h = lane >> 5, r32 = lane & 31;
    char* const planes = lds;
    char* const landing = lds + 2 * PLANES + wave * (LANDING / 4);
    char* const nbl_lds = lds + 2 * PLANES + LANDING + wave * NBL;
    uint32_t* const slot = reinterpret_cast<uint32_t*>(lds + 2 * PLANES + LANDING + 4 * NBL) + wave * NOTE;
    float* const b_lds = reinterpret_cast<float*>(lds + 2 * PLANES + LANDING + 4 * NBL + 4 * NOTE * 4);
    v4u* const low_lds = reinterpret_cast<v4u*>(b_lds + C) + cb * (LOW_SLOTS * STAGES * 2 * 64) + lane;

    /* half tiles in use, and this block's share: XCD-aware (block b works for XCD b % 8 on a contiguous eighth) */
    const int n_tiles = B.active_h[L.frame_end], t_first = B.active_h[L.frame_begin]; /* of the launch's frames: half tiles t_first to n_tiles */
    const int xcd = blockIdx.x & 7, lb = blockIdx.x >> 3, gx = gridDim.x >> 3;
    const int per_xcd = (n_tiles - t_first + 7) >> 3;
    const int t_end = min(n_tiles, t_first + (xcd + 1) * per_xcd);
    const int tile0 = t_first + xcd * per_xcd + lb;
    const int count = tile0 < t_end ? (t_end - tile0 + gx - 1) / gx : 0; /* half tiles of this block: tile0 + k * gx, k < count */

    /* the wave's weights: [cb][stage][slot][step][h, m, l][lane] 16 bytes each */
    v4u w[STAGES][SLOTS][2][3];
    {
        const v4u* wp = reinterpret_cast<const v4u*>(L.w_x3) + (size_t) cb * (STAGES * SLOTS * 2 * 3 * 64) + lane;
#pragma unroll
        for (int c = 0; c < STAGES; ++c)
#pragma unroll
            for (int s = 0; s < SLOTS; ++s)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int p = 0; p < 3; ++p) {
                        const v4u t = wp[(((c * SLOTS + s) * 2 + j) * 3 + p) * 64];
                        if (p == 2 && s >= LOW_FROM) low_lds[((c * (SLOTS - LOW_FROM) + s - LOW_FROM) * 2 + j) * 64] = t; /* the waves of a cb write the same */
                        else w[c][s][j][p] = t;
                    }
    }
    if (threadIdx.x < C) b_lds[threadIdx.x] = L.b[threadIdx.x];
    /* Every load the compiler knows of returns before the first one it does not know of is issued. The same statements say where
     * the weights live: at most 64 tuples fill the accumulation registers, from which the matrix instruction reads its operands as
     * well as from vector registers, the others stay in the vector file. No instantiation may spill (conv_bf16.hip says why). */
#pragma unroll
    for (int c = 0; c < STAGES; ++c)
#pragma unroll
        for (int s = 0; s < SLOTS; ++s)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    if (p == 2 && s >= LOW_FROM) continue;
                    if (((c * SLOTS + s) * 2 + j) * 3 + p < 64) asm volatile("" : "+a"(w[c][s][j][p]));
                    else asm volatile("" : "+v"(w[c][s][j][p]));
                }

    const uint32_t total_rows = (uint32_t) B.n_row_tiles * VMHIP_TILE;
    const v4u note_rsrc = raw_rsrc(B.tile_note_h, (uint64_t) n_tiles * NOTE * 4);
    const v4u nbl_rsrc = raw_rsrc(B.row_nbl_h, (uint64_t) total_rows * VMHIP_NBL_STRIDE * 2);

    /* the note of half tile t into the wave's slot: 3 loads */
    auto request_note = [&](int t, bool live) {
        const uint32_t base = lds_address(slot);
        const uint32_t off = live ? (uint32_t) (t * NOTE + lane) * 4u : OOR;
        load_to_lds_b32(note_rsrc, base, off);
        load_to_lds_b32(note_rsrc, base + 256, live ? off + 256 : OOR);
        if (lane < NOTE - 128) load_to_lds_b32(note_rsrc, base + 512, live ? off + 512 : OOR);
    };
    auto read_note = [&]() {
        const v4u d = *reinterpret_cast<const v4u*>(slot);
        return make_int4(__builtin_amdgcn_readfirstlane((int) d.x), __builtin_amdgcn_readfirstlane((int) d.y),
                         __builtin_amdgcn_readfirstlane((int) d.z), __builtin_amdgcn_readfirstlane((int) d.w));
    };
    /* the wave's rows of the neighbour table of the half tile at d */
    auto request_nbl = [&](const int4& d, bool live) {
        load_to_lds_b128(nbl_rsrc, lds_address(nbl_lds), live ? (uint32_t) (d.x + rw * (32 * RB) + lane) * (VMHIP_NBL_STRIDE * 2) : OOR);
    };
    /* Group q of the wave is rows 16 (wave + 4 q) .. + 15 of the half tile's 256. A lane brings in the eight values that it will split, four with
     * each of two loads, so that it finds them at its own place in both. The first two groups are rows of the half tile itself, the others halo rows, whose numbers are in the note. */
    struct Source {
        v4u rsrc;
        int own, frame_row, halos; /* uniform */
        bool live;
    };
    auto source = [&](const int4& d, bool live) {
        /* offsets are relative to the frame's first row: a frame's rows fit 32 bits, a batch's need not */
        return Source{raw_rsrc(reinterpret_cast<const char*>(in) + (size_t) (uint32_t) d.w * ROWB, (uint64_t) (total_rows - (uint32_t) d.w) * ROWB), d.x - d.w, d.w,
                      live ? (d.z & ~VMHIP_NOTE_FAR) : 0, live};
    };
    auto request_rows = [&](int q, int half, int stage, const Source& S) {
        const int row = 16 * (wave + 4 * (q & 1)) + (lane >> 2);
        const uint32_t piece = (uint32_t) (stage * (SC * 4) + (lane & 3) * 32 + half * 16);
        uint32_t off;
        if (q < 2) off = S.live ? (uint32_t) (S.own + row) * ROWB + piece : OOR;
        else off = row < S.halos ? (slot[4 + row] - (uint32_t) S.frame_row) * ROWB + piece : OOR;
        load_to_lds_b128(S.rsrc, lds_address(landing) + (uint32_t) ((q * 2 + half) * 1024), off);
    };
    /* The splitting of a group: a lane takes eight values of a row. Piece q8 (eight channels, 16 bytes) of row R of a part lies at
     * R * 64 + (q8 ^ ((R >> 2) & 3)) * 16: sixteen lanes that read the same piece of sixteen consecutive rows meet no bank twice. */
    const uint32_t split_to = (uint32_t) ((lane >> 2) * 64 + (((lane & 3) ^ ((lane >> 4) & 3)) * 16)); /* (R >> 2) & 3 = lane / 16 in every group */
    v4f raw[2];
    uint32_t parts[3][4];
    float rest[2][2];
    /* piece i of group q: read, ten pieces of arithmetic of two to five instructions (at most as many fit into the time of a matrix
     * instruction), write. (v_dot2c_f32_bf16 would take a part off a value in one instruction instead of two, but it runs where the
     * matrix instructions do and costs them 8 to 16 cycles.) */
    auto split_piece = [&](int i, int q, char* to) {
        auto take_off = [&](int p, uint32_t packed, float x0, float x1) {
            rest[p & 1][0] = x0 - __uint_as_float(packed << 16);
            rest[p & 1][1] = x1 - __uint_as_float(packed & 0xffff0000u);
        };
        auto high = [&](int p) {
            const float x0 = raw[p >> 1][(p & 1) * 2], x1 = raw[p >> 1][(p & 1) * 2 + 1];
            parts[0][p] = pack_bf16(x0, x1);
            take_off(p, parts[0][p], x0, x1);
        };
        auto middle = [&](int p) {
            parts[1][p] = pack_bf16(rest[p & 1][0], rest[p & 1][1]);
            take_off(p, parts[1][p], rest[p & 1][0], rest[p & 1][1]);
        };
        auto low = [&](int p) { parts[2][p] = pack_bf16(rest[p & 1][0], rest[p & 1][1]); };
        if (i == 0) {
            raw[0] = *reinterpret_cast<const v4f*>(landing + q * 2048 + lane * 16);
            raw[1] = *reinterpret_cast<const v4f*>(landing + q * 2048 + 1024 + lane * 16);
        }
        else if (i == 1 || i == 2) high(i - 1);
        else if (i == 3 || i == 4) middle(i - 3);
        else if (i == 5) low(0), low(1);
        else if (i == 6 || i == 7) high(i - 4);
        else if (i == 8 || i == 9) middle(i - 6);
        else if (i == 10) low(2), low(3);
        else if (i == 11) {
            char* const p = to + (wave + 4 * q) * 1024 + split_to;
#pragma unroll
            for (int k = 0; k < 3; ++k) *reinterpret_cast<v4u*>(p + k * PART) = v4u{parts[k][0], parts[k][1], parts[k][2], parts[k][3]};
        }
    };

    auto tile_of = [&](int k) { return tile0 + k * gx; };
    auto walk = [&]() {
        /* ---- prologue: the first stage split, the second on its way ---- */
        int4 d_next; /* half tile k + 1 */
        request_note(tile_of(0), true);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        d_next = read_note();
        {
            const Source S = source(d_next, true);
#pragma unroll
            for (int i = 0; i < 2 * GROUPS; ++i) request_rows(i >> 1, i & 1, 0, S);
            request_nbl(d_next, true);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int q = 0; q < GROUPS; ++q)
#pragma unroll
                for (int i = 0; i < 12; ++i) split_piece(i, q, planes);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the landing has been read: it may be written again */
#pragma unroll
            for (int i = 0; i < 2 * GROUPS; ++i) request_rows(i >> 1, i & 1, 1, S);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* and so has the slot */
            request_note(tile_of(min(1, count - 1)), 1 < count);
        }

        /* the finished sums of the half tile before, waiting for activation and store: a row block per stage */
        v16f done[RB];
        constexpr uint32_t NOWHERE = 0x80000000u; /* past every half tile's results, also with a piece's offset added */
        uint32_t done_first = 0, done_at[RB]; /* their half tile's first row in the batch; where the lane's values go from there */
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            done_at[rb] = NOWHERE;
#pragma unroll
            for (int v = 0; v < 16; ++v) done[rb][v] = 0.0f;
        }
        auto finish_slice = [&](int i, int rb, const __amdgpu_buffer_rsrc_t& rs) {
            if (i < 16) {
                const float x = done[rb][i];
                done[rb][i] = ACT == VMHIP_SELU ? selu(x) : fmaxf(x, 0.0f);
            }
            else if (i < N_SLICES) {
                const int g = i - 16; /* two lanes write 32 bytes of a row with one instruction */
                __builtin_amdgcn_raw_buffer_store_b128(v4u{__float_as_uint(done[rb][g * 4]), __float_as_uint(done[rb][g * 4 + 1]), __float_as_uint(done[rb][g * 4 + 2]), __float_as_uint(done[rb][g * 4 + 3])}, rs,
                                                       done_at[rb] + (uint32_t) (g * 32), 0, 0);
            }
        };
        auto out_window = [&]() {
            return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<char*>(out) + (size_t) done_first * ROWB, 0, BT * ROWB, 0x00020000);
        };

        v16f big[RB], small[RB]; /* the products of the high parts; the others */
        for (int k = 0; k < count; ++k) {
            const int4 d_cur = d_next;
            uint32_t own[RB];
            bool valid[RB];
            v4u nbl[RB];
            static_for<STAGES>([&](auto stage_tag) {
                constexpr int stage = decltype(stage_tag)::value;
                const int at_stage = (k * STAGES + stage) & 1;
                const char* const rows = planes + at_stage * PLANES;
                char* const split_into = planes + (at_stage ^ 1) * PLANES;
                /* My loads of the stage before have landed once nothing but the stores issued after them can be in flight (vector
                 * memory operations complete in order); before the first stores: once nothing is */
                if (k == 0 && stage == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_STORES) : "memory");
                __syncthreads(); /* everyone has split this stage's rows, and read the last of those that are split next */
                if constexpr (stage == 0) {
                    d_next = read_note();
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) {
                        const int own_at = (rw * RB + rb) * 32 + r32;
                        valid[rb] = own_at < d_cur.y && !(d_cur.z & VMHIP_NOTE_FAR); /* a half tile with more halo rows than are staged is computed again below */
                        own[rb] = (uint32_t) max(0, min(own_at, d_cur.y - 1)); /* lanes past the rows in use redo the last one and store nothing */
                        nbl[rb] = *reinterpret_cast<const v4u*>(nbl_lds + (rb * 32 + r32) * 16);
                        if (own_at >= d_cur.y) nbl[rb] = v4u{0, 0, 0, 0};
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const v4f b4 = *reinterpret_cast<const v4f*>(b_lds + cb * 32 + g * 8 + h * 4);
#pragma unroll
                            for (int v = 0; v < 4; ++v) big[rb][g * 4 + v] = b4[v], small[rb][g * 4 + v] = 0.0f;
                        }
                    }
                }
                const Source S = source(d_next, k + 1 < count);
                const __amdgpu_buffer_rsrc_t rs = out_window();

                v4u x[2][RB][3];
                uint32_t at[RB]; /* where the lane's piece of the slot's row lies; the second step is an exclusive or away */
                auto gather = [&](int c, int rb) {
                    const int s = c >> 1, j = c & 1;
                    uint32_t li = s == 0 ? own[rb] : nbl_entry(nbl[rb], s - 1);
                    li = li >= (uint32_t) BROWS ? 0u : li; /* not staged: the row is computed again below */
                    if (j == 0) at[rb] = li * 64u + (((uint32_t) h ^ ((li >> 2) & 3u)) * 16u);
                    const char* const p = rows + (at[rb] ^ (uint32_t) (j * 32));
#pragma unroll
                    for (int t = 0; t < 3; ++t) x[c % 2][rb][t] = *reinterpret_cast<const v4u*>(p + t * PART);
                };
                /* The side work of a stage in the order it is issued: the next stage's four groups of rows are split, the stage after that
                 * is requested into the places they leave; the neighbour table of the next half tile; the note of the one that is
                 * loaded next; activation and stores of a row block of the half tile before. */
                auto item = [&](auto item_tag) {
                    constexpr int i = decltype(item_tag)::value;
                    if constexpr (i < GROUPS * PIECES) {
                        constexpr int q = i / PIECES, piece = i % PIECES;
                        if constexpr (piece < 12) split_piece(piece, q, split_into);
                        else request_rows(q, piece - 12, stage, S);
                    }
                    else if constexpr (i == GROUPS * PIECES) {
                        if constexpr (stage == 0) request_nbl(d_next, k + 1 < count);
                    }
                    else if constexpr (i == GROUPS * PIECES + 1) {
                        if constexpr (stage == STAGES - 1) request_note(tile_of(min(k + 2, count - 1)), k + 2 < count);
                    }
                    else if constexpr (i < GROUPS * PIECES + 2 + N_SLICES) {
                        finish_slice(i - (GROUPS * PIECES + 2), stage, rs);
                    }
                };
                static_assert(CHUNKS * 6 >= GROUPS * PIECES + 2 + N_SLICES, "every item of the side work finds its place");
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) gather(0, rb);
                static_for<CHUNKS>([&](auto chunk) {
                    constexpr int c = decltype(chunk)::value, s = c >> 1, j = c & 1;
                    v4u low;
                    static_for<PER>([&](auto mm) {
                        constexpr int m = decltype(mm)::value, rb = m % RB, kind = m / RB;
                        const v8bf a = __builtin_bit_cast(v8bf, s >= LOW_FROM && kind == 4 ? low : w[stage][s][j][WP[kind]]);
                        const v8bf b = __builtin_bit_cast(v8bf, x[c % 2][rb][XP[kind]]);
                        v16f& acc = kind == 5 ? big[rb] : small[rb];
                        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        /* the operands of a step to come, once the low parts' registers are free */
                        if constexpr (c + 1 < CHUNKS && (m == 6 || m == 8)) gather(c + 1, (m - 6) / 2);
                        if constexpr (m == RB && s >= LOW_FROM) low = low_lds[((stage * (SLOTS - LOW_FROM) + s - LOW_FROM) * 2 + j) * 64];
                        /* an item behind every second matrix instruction, between those that are followed by reads: what does not fit
                         * into an instruction's 32 cycles delays the next */
                        if constexpr (m % 2 == 1) item(std::integral_constant<int, (c * PER + m) / RB>());
                        __builtin_amdgcn_sched_barrier(0);
                    });
                });
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* every operand has been read, every part written */
            });
            done_first = (uint32_t) d_cur.x;
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                done_at[rb] = valid[rb] ? own[rb] * ROWB + (uint32_t) (cb * 32 + h * 4) * 4 : NOWHERE;
#pragma unroll
                for (int v = 0; v < 16; ++v) done[rb][v] = big[rb][v] + small[rb][v];
            }
        }
        /* the last half tile's results; and no LDS load may outlive the wave */
        {
            const __amdgpu_buffer_rsrc_t rs = out_window();
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int i = 0; i < N_SLICES; ++i) finish_slice(i, rb, rs);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };

    __syncthreads(); /* biases and low parts are in LDS */
    if (count > 0) walk();

    /* Half tiles with more halo rows than are staged (three in a hundred on dense meshes): every neighbour straight from memory, 64 rows
     * at a time, the operands of DEEP steps under way at once. The same instructions on the same parts in the same order as
     * above: which neighbours were staged does not show in the results. (Lanes that fetched only what was not staged, a step
     * ahead, took 40 us for a half tile.) */
    constexpr int DEEP = 6, PER_TILE = CBW;
    const int n_far = B.active_h[B.n_frames + 1] * PER_TILE;
    for (int t = blockIdx.x; t < n_far; t += gridDim.x) {
        const int number = B.far_h[t / PER_TILE];
        if (number < t_first || number >= n_tiles) continue; /* another launch's: the rows that it reads may no longer be what they were */
        const uint32_t* const note = B.tile_note_h + (size_t) number * NOTE;
        const uint32_t first = note[0], in_use = note[1], frame_row = note[3];
        const uint32_t row = (uint32_t) (((t % PER_TILE) * (4 / CBW) + rw) * 32 + r32), own = min(row, in_use - 1);
        uint32_t from[SLOTS];
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) from[s] = s == 0 ? first + own : frame_row + (uint32_t) B.row_nb[(size_t) (first + own) * B.nb_stride + (s - 1)];
        v16f big, small;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const v4f b4 = *reinterpret_cast<const v4f*>(b_lds + cb * 32 + g * 8 + h * 4);
#pragma unroll
            for (int v = 0; v < 4; ++v) big[g * 4 + v] = b4[v], small[g * 4 + v] = 0.0f;
        }
        v4f ring[DEEP][2];
        auto request = [&](int c) { /* c counts the steps of all stages */
            const int stage = c / CHUNKS, s = c % CHUNKS >> 1, j = c & 1;
            const float* const p = in + (size_t) from[s] * C + stage * SC + j * 16 + h * 8;
            ring[c % DEEP][0] = *reinterpret_cast<const v4f*>(p), ring[c % DEEP][1] = *reinterpret_cast<const v4f*>(p + 4);
        };
#pragma unroll
        for (int c = 0; c < DEEP; ++c) request(c);
        static_for<STAGES * CHUNKS>([&](auto chunk) {
            constexpr int c = decltype(chunk)::value, stage = c / CHUNKS, s = c % CHUNKS >> 1, j = c & 1;
            v4u x[3];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const Parts p = split_pair(ring[c % DEEP][q >> 1][(q & 1) * 2], ring[c % DEEP][q >> 1][(q & 1) * 2 + 1]);
                x[0][q] = p.high, x[1][q] = p.middle, x[2][q] = p.low;
            }
            if constexpr (c + DEEP < STAGES * CHUNKS) request(c + DEEP);
            v4u low = {0, 0, 0, 0};
            if constexpr (s >= LOW_FROM) low = low_lds[((stage * (SLOTS - LOW_FROM) + s - LOW_FROM) * 2 + j) * 64];
            static_for<6>([&](auto kind_tag) {
                constexpr int kind = decltype(kind_tag)::value;
                const v8bf a = __builtin_bit_cast(v8bf, s >= LOW_FROM && kind == 4 ? low : w[stage][s][j][WP[kind]]);
                v16f& acc = kind == 5 ? big : small;
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(v8bf, x[XP[kind]]), acc, 0, 0, 0);
            });
        });
        if (row < in_use) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                v4f o;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float sum = big[g * 4 + v] + small[g * 4 + v];
                    o[v] = ACT == VMHIP_SELU ? selu(sum) : fmaxf(sum, 0.0f);
                }
                *reinterpret_cast<v4f*>(out + (size_t) (first + row) * C + cb * 32 + g * 8 + h * 4) = o;
            }
        }
    }
}

template <int ACT>
int launch_x3(const VmBatchDev& B, const VmLayerDev& L, const float* in, float* out, hipStream_t stream) {
    auto kernel = vm_conv_x3_kernel<ACT>;
    static std::atomic<bool> configured{false}; /* engines on several host threads may get here together */
    if (!configured) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(LDS_BYTES)) != hipSuccess) {
            (void) hipGetLastError();
            return -1;
        }
        configured = true;
    }
    /* one block of four waves per CU; the kernel reads the number of half tiles in use on the device */
    hipLaunchKernelGGL(kernel, dim3(256), dim3(256), LDS_BYTES, stream, B, L, in, out);
    return 0;
}

}  // namespace

/* Weight layout the kernel consumes: [column block cb][stage][slot][step j][part: h, m, l][lane = half * 32 + o][e = 0..7] bf16 of
 * W[slot * 64 + stage * 32 + j * 16 + half * 8 + e][cb * 32 + o] */
size_t vm_x3_weight_bytes(void) { return size_t(SLOTS) * C * C * 3 * 2; }
void vm_x3_permute_weights(const float* w, void* wp) {
    uint16_t* dst = reinterpret_cast<uint16_t*>(wp);
    for (int cb = 0; cb < CBW; ++cb)
        for (int c = 0; c < STAGES; ++c)
            for (int s = 0; s < SLOTS; ++s)
                for (int j = 0; j < 2; ++j)
                    for (int lane = 0; lane < 64; ++lane)
                        for (int e = 0; e < 8; ++e) {
                            float v = w[size_t(s * C + c * SC + j * 16 + (lane >> 5) * 8 + e) * C + cb * 32 + (lane & 31)];
                            for (int p = 0; p < 3; ++p) {
                                const uint16_t part = bf16_round(v);
                                dst[(((((size_t(cb) * STAGES + c) * SLOTS + s) * 2 + j) * 3 + p) * 64 + lane) * 8 + e] = part;
                                v -= bf16_value(part);
                            }
                        }
}

bool vm_x3_supported(int c_in, int c_out, int slots, int activation) {
    return c_in == C && c_out == C && slots == SLOTS && (activation == VMHIP_SELU || activation == VMHIP_RELU);
}

int vm_launch_conv_x3(const VmBatchDev& B, const VmLayerDev& L, const float* in, float* out, hipStream_t stream, const char** kernel_name) {
    if (B.n_row_tiles <= 0) return 0;
    if (!B.row_nbl_h || !B.tile_note_h || !B.active_h || !L.w_x3 || !vm_x3_supported(L.c_in, L.c_out, L.slots, L.activation)) return -1;
    if (kernel_name) *kernel_name = vm_kernel_name("conv_x3", L.c_in, L.c_out, L.slots);
    return L.activation == VMHIP_SELU ? launch_x3<VMHIP_SELU>(B, L, in, out, stream) : launch_x3<VMHIP_RELU>(B, L, in, out, stream);
}
