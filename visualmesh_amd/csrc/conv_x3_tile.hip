/*
 * conv_x3_tile.hip - fp32 graph-convolution layers with 16 or 32 input channels and 32 output channels on the bf16 matrix
 * instructions, with every fp32 factor split into three bf16 parts (conv_x3.hip says what that computes and for which networks): neighbour
 * gather + dense + bias + activation in one kernel (reference engine/cpu/engine.hpp:213-264, apply_activation.hpp:34-84).
 *
 * A block is eight waves, two per SIMD, and works on a row tile (256 rows, through the tile-local tables): wave w on rows 32 w .. 32 w + 31
 * and all output channels. It keeps the high and middle parts of all weights in registers (112 a lane for 32 channels and seven
 * slots), the low parts in LDS. The tile's rows and its halo rows arrive in LDS as fp32 by buffer_load ... lds; each wave splits those that it
 * has brought in itself into three planes of bf16 and requests the next tile's rows into the places they leave; then a barrier, and
 * the matrix work, whose operands come from the planes, while the next tile is under way. Activation and stores of a tile are pieces
 * of side work between the matrix instructions of the one after. The two waves of a SIMD fill each other's gaps; the splitting (a sixth
 * of a tile's time) is not overlapped, there being no room for a second set of planes.
 *
 * What bounds it: a tile's phases one after the other. By counters the matrix pipe is busy for 37 % of the cycles at 32 -> 32 and 28 % at 16 -> 32,
 * the clock is 2.1 to 2.3 GHz and the 291 MB of a 32 -> 32 launch move at 2.8 TB/s: neither the pipe nor memory is at its limit. 1.05
 * million rows by rocprofv3's trace, fp32 products / so: 32 -> 32 132 / 102 us, 16 -> 32 80 / 62; by events 32 -> 16 95 / 110 and
 * 16 -> 16, 71 000 rows, 9.2 / 10.8, where half of the columns are padding: they stay with the fp32 instructions. Sixteen frames' pass
 * through 4-16-32-32-32-32-32-16-3: 814 -> 686 us. Distance of that network's probabilities from float64: 4.0e-7 -> 2.1e-7 (root mean square).
 *
 * A tile with more than 192 halo rows, for which there is no room at 32 channels (the neighbourhood kernel lists them), is computed
 * from memory at the end, with the same parts, instructions and order: which rows were staged does not show in the results.
 */
#include <atomic>

#include "conv_x3.h"

namespace {

constexpr int NT = 512, WAVES = NT / 64;
constexpr int C_OUT = 32, SLOTS = 7, NN = SLOTS - 1;
constexpr int N_SLICES = 20, N_STORES = 4; /* of a wave's finished rows: 16 activations, 4 stores */
constexpr int SLOT_WORDS = 4 + 32;         /* a wave's note of a tile: the descriptor, the halo rows it brings in */

__host__ __device__ constexpr int staged_halo(int c_in) { return c_in > 16 ? VM_X3_TILE_HALO : VMHIP_HALO_MAX; }
__host__ __device__ constexpr int staged_rows(int c_in) { return VMHIP_TILE + staged_halo(c_in); }
__host__ __device__ constexpr int steps(int c_in) { return SLOTS * (c_in / 16); }
__host__ __device__ constexpr size_t tile_lds_bytes(int c_in) {
    return size_t(staged_rows(c_in)) * c_in * (3 * 2 + 4) + WAVES * (32 * 16 + SLOT_WORDS * 4) + 32 * 4 + size_t(steps(c_in)) * 1024;
}

template <int C_IN, int ACT>
__global__ __launch_bounds__(NT) void vm_conv_x3_tile_kernel(VmBatchDev B, VmLayerDev L, const float* __restrict__ in, float* __restrict__ out) {
    constexpr int HALO = staged_halo(C_IN), ROWS = staged_rows(C_IN);
    constexpr int ROWB = C_IN * 4, OUTB = C_OUT * 4, PR = C_IN * 2, PART = ROWS * PR;
    constexpr int J = C_IN / 16, CHUNKS = SLOTS * J;  /* steps of 16 values per slot, and of all slots */
    constexpr int UNIT = 1024 / ROWB, LPR = 64 / UNIT; /* rows that a wave brings in with one load, lanes to a row */
    constexpr int OWN_U = VMHIP_TILE / UNIT / WAVES, HALO_U = HALO / UNIT / WAVES, UNITS = OWN_U + HALO_U;
    static_assert(NN <= VMHIP_NBL_STRIDE && (C_IN == 16 || C_IN == 32), "shapes of this kernel");
    static_assert(HALO_U * UNIT + 4 <= SLOT_WORDS && OWN_U * UNIT * WAVES == VMHIP_TILE && HALO_U * UNIT * WAVES == HALO, "the units cover the staged rows");

    extern __shared__ float4 lds4[];
    char* const lds = reinterpret_cast<char*>(lds4);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
    const int h = lane >> 5, r32 = lane & 31;
    char* const planes = lds;
    char* const landing = planes + 3 * PART + wave * (UNITS * 1024);
    char* const nbl_lds = planes + 3 * PART + ROWS * ROWB + wave * (32 * 16);
    uint32_t* const slot = reinterpret_cast<uint32_t*>(planes + 3 * PART + ROWS * ROWB + WAVES * 32 * 16) + wave * SLOT_WORDS;
    float* const b_lds = reinterpret_cast<float*>(planes + 3 * PART + ROWS * ROWB + WAVES * (32 * 16 + SLOT_WORDS * 4));
    v4u* const low_lds = reinterpret_cast<v4u*>(b_lds + 32) + lane;

    const int n_tiles = vm_row_tiles(B);
    const int per_xcd = (n_tiles + 7) >> 3;
    /* Few tiles: two blocks to a tile, each with half of the waves contracting, one per SIMD (a network 3-16-32-32-32-32-32-16-3 on
     * 4 000 rows: 90.5 us a pass with whole tiles, 84.4 so) */
    const bool halves = per_xcd * 2 <= (int) (gridDim.x >> 3);
    const int xcd = blockIdx.x & 7, lb = (int) (blockIdx.x >> 3) >> (halves ? 1 : 0), gx = (int) (gridDim.x >> 3) >> (halves ? 1 : 0);
    const bool contracts = !halves || (wave >> 2) == (int) (blockIdx.x >> 3 & 1);
    const int t_end = min(n_tiles, (xcd + 1) * per_xcd);
    const int tile0 = xcd * per_xcd + lb;
    const int count = tile0 < t_end ? (t_end - tile0 + gx - 1) / gx : 0; /* tiles of this block: tile0 + k * gx, k < count */
    const int n_far = min(*B.n_far_tiles, B.n_row_tiles);
    if (count == 0 && (int) blockIdx.x >= n_far) return; /* the whole block leaves before any barrier or LDS load */

    const uint32_t total_rows = (uint32_t) B.n_row_tiles * VMHIP_TILE;
    const v4u desc_rsrc = raw_rsrc(B.tile_desc, (uint64_t) n_tiles * 16), halo_rsrc = raw_rsrc(B.tile_halo, (uint64_t) n_tiles * VMHIP_HALO_MAX * 4);
    const v4u nbl_rsrc = raw_rsrc(B.row_nbl, (uint64_t) total_rows * VMHIP_NBL_STRIDE * 2);
    auto tile_of = [&](int k) { return tile0 + k * gx; };
    /* the descriptor of tile t and the halo rows that this wave brings in, into its slot */
    auto request_note = [&](int t, bool live) {
        if (lane < HALO_U * UNIT)
            load_to_lds_b32(halo_rsrc, lds_address(slot + 4), live ? (uint32_t) (t * VMHIP_HALO_MAX + ((lane / UNIT) * WAVES + wave) * UNIT + lane % UNIT) * 4u : OOR);
        if (lane < 4) load_to_lds_b32(desc_rsrc, lds_address(slot), live ? (uint32_t) (t * 4 + lane) * 4u : OOR);
    };
    auto read_note = [&]() {
        const v4u d = *reinterpret_cast<const v4u*>(slot);
        return make_int4(__builtin_amdgcn_readfirstlane((int) d.x), __builtin_amdgcn_readfirstlane((int) d.y),
                         __builtin_amdgcn_readfirstlane((int) d.z), __builtin_amdgcn_readfirstlane((int) d.w));
    };
    /* the wave's rows of the neighbour table */
    auto request_nbl = [&](const int4& d, bool live) {
        if (lane < 32) load_to_lds_b128(nbl_rsrc, lds_address(nbl_lds), live ? (uint32_t) (d.x + wave * 32 + lane) * (VMHIP_NBL_STRIDE * 2) : OOR);
    };
    /* Unit u of the wave: rows (8 u + wave) UNIT .. of the tile, then of its halo. Offsets are relative to the frame's first row: a
     * frame's rows fit 32 bits (the host sees to it), a batch's need not. */
    auto request_rows = [&](int u, const int4& d, const v4u& rsrc, bool live) {
        const int row = ((u < OWN_U ? u : u - OWN_U) * WAVES + wave) * UNIT + lane / LPR;
        uint32_t off = OOR;
        if (u < OWN_U) off = live ? (uint32_t) (d.x - d.w + row) * ROWB + (uint32_t) (lane % LPR) * 16 : OOR;
        else if (live && row < d.z) off = (slot[4 + (u - OWN_U) * UNIT + lane / LPR] - (uint32_t) d.w) * ROWB + (uint32_t) (lane % LPR) * 16;
        load_to_lds_b128(rsrc, lds_address(landing) + (uint32_t) (u * 1024), off);
    };
    auto frame_rows = [&](const int4& d) { return raw_rsrc(reinterpret_cast<const char*>(in) + (size_t) (uint32_t) d.w * ROWB, (uint64_t) (total_rows - (uint32_t) d.w) * ROWB); };
    /* Piece q (eight channels, 16 bytes) of row R of a part lies at R * PR + (q ^ swizzle(R)) * 16: sixteen lanes that read the same piece
     * of sixteen consecutive rows meet no bank twice. */
    auto swizzle = [](uint32_t R) { return C_IN == 32 ? (R >> 2) & 3u : (R >> 3) & 1u; };

    v16f done;
    constexpr uint32_t NOWHERE = 0x80000000u; /* past every tile's results, also with a piece's offset added */
    uint32_t done_first = 0, done_at = NOWHERE;
    auto finish_slice = [&](int i, const __amdgpu_buffer_rsrc_t& rs) {
        if (i < 16) {
            done[i] = ACT == VMHIP_SELU ? selu(done[i]) : fmaxf(done[i], 0.0f);
        }
        else if (i < N_SLICES) {
            const int g = i - 16; /* two lanes write 32 bytes of a row with one instruction */
            __builtin_amdgcn_raw_buffer_store_b128(v4u{__float_as_uint(done[g * 4]), __float_as_uint(done[g * 4 + 1]), __float_as_uint(done[g * 4 + 2]), __float_as_uint(done[g * 4 + 3])}, rs,
                                                   done_at + (uint32_t) (g * 32), 0, 0);
        }
    };
    auto out_window = [&]() {
        return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<char*>(out) + (size_t) done_first * OUTB, 0, VMHIP_TILE * OUTB, 0x00020000);
    };
    auto start_sums = [&](v16f& big, v16f& small) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const v4f b4 = *reinterpret_cast<const v4f*>(b_lds + g * 8 + h * 4);
#pragma unroll
            for (int v = 0; v < 4; ++v) big[g * 4 + v] = b4[v], small[g * 4 + v] = 0.0f;
        }
    };

    /* the first tile on its way, the note of the second requested; the weights come meanwhile */
    int4 d_next = make_int4(0, 0, 0, 0);
    if (count > 0) {
        request_note(tile_of(0), true);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        d_next = read_note();
        const v4u rsrc = frame_rows(d_next);
#pragma unroll
        for (int u = 0; u < UNITS; ++u) request_rows(u, d_next, rsrc, true);
        request_nbl(d_next, true);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the slot has been read: it may be written again */
        request_note(tile_of(min(1, count - 1)), 1 < count);
    }

    /* weights: [step][h, m, l][lane] 16 bytes each */
    v4u w[CHUNKS][2];
    {
        const v4u* const wp = reinterpret_cast<const v4u*>(L.w_x3) + lane;
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) w[c][0] = wp[(c * 3 + 0) * 64], w[c][1] = wp[(c * 3 + 1) * 64];
        for (int c = wave; c < CHUNKS; c += WAVES) low_lds[c * 64] = wp[(c * 3 + 2) * 64];
    }
    if (threadIdx.x < C_OUT) b_lds[threadIdx.x] = L.b[threadIdx.x];
    /* every load the compiler knows of has returned before the tile loop, whose waits count */
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) asm volatile("" : "+v"(w[c][0]), "+v"(w[c][1]));

    if (count > 0) {
#pragma unroll
        for (int v = 0; v < 16; ++v) done[v] = 0.0f;
        for (int k = 0; k < count; ++k) {
            /* my loads of this tile have landed once nothing but the stores issued after them can be in flight (vector memory
             * operations complete in order); before the first stores: once nothing is */
            if (k == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_STORES) : "memory");
            __syncthreads(); /* everyone has read the last of the planes */
            const int4 d_cur = d_next;
            d_next = read_note();
            const bool more = k + 1 < count;
            const v4u nbl = *reinterpret_cast<const v4u*>(nbl_lds + r32 * 16);
            {
                const v4u rsrc = frame_rows(d_next);
                v4f raw[UNITS];
#pragma unroll
                for (int u = 0; u < UNITS; ++u) raw[u] = *reinterpret_cast<const v4f*>(landing + u * 1024 + lane * 16);
#pragma unroll
                for (int u = 0; u < UNITS; ++u) {
                    const uint32_t R = (uint32_t) ((u < OWN_U ? 0 : VMHIP_TILE) + ((u < OWN_U ? u : u - OWN_U) * WAVES + wave) * UNIT + lane / LPR);
                    const Parts a = split_pair(raw[u][0], raw[u][1]), b = split_pair(raw[u][2], raw[u][3]);
                    char* const p = planes + R * PR + (((uint32_t) (lane % LPR) >> 1) ^ swizzle(R)) * 16 + (lane & 1) * 8;
                    *reinterpret_cast<uint2*>(p) = make_uint2(a.high, b.high);
                    *reinterpret_cast<uint2*>(p + PART) = make_uint2(a.middle, b.middle);
                    *reinterpret_cast<uint2*>(p + 2 * PART) = make_uint2(a.low, b.low);
                    request_rows(u, d_next, rsrc, more);
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the neighbour table's rows and the slot have been read */
            request_nbl(d_next, more);
            request_note(tile_of(min(k + 2, count - 1)), k + 2 < count);
            __syncthreads(); /* every part is in its plane */

            if (!contracts) continue; /* the block's only tile */
            const bool far_tile = d_cur.z > VM_X3_TILE_HALO || d_cur.z >= B.halo_cap; /* as the neighbourhood kernel lists them */
            const int own_at = wave * 32 + r32;
            const bool valid = own_at < d_cur.y && !far_tile;
            const uint32_t own = (uint32_t) max(0, min(own_at, d_cur.y - 1)); /* lanes past the rows in use redo the last one and store nothing */
            v16f big, small;
            start_sums(big, small);
            const __amdgpu_buffer_rsrc_t rs = out_window();
            v4u x[2][3];
            uint32_t at = 0; /* where the lane's piece of the slot's row lies; the second step is an exclusive or away */
            auto gather = [&](int c) {
                const int s = c / J, j = c % J;
                if (j == 0) {
                    uint32_t li = s == 0 || own_at >= d_cur.y ? own : nbl_entry(nbl, s - 1);
                    li = li >= (uint32_t) ROWS ? 0u : li; /* not staged: the tile is computed again below */
                    at = li * PR + (((uint32_t) h ^ swizzle(li)) * 16u);
                }
                const char* const p = planes + (at ^ (uint32_t) (j * 32));
#pragma unroll
                for (int t = 0; t < 3; ++t) x[c % 2][t] = *reinterpret_cast<const v4u*>(p + t * PART);
            };
            gather(0);
            static_for<CHUNKS>([&](auto chunk) {
                constexpr int c = decltype(chunk)::value;
                const v4u low = low_lds[c * 64];
                static_for<6>([&](auto kind_tag) {
                    constexpr int kind = decltype(kind_tag)::value, m = c * 6 + kind;
                    const v8bf a = __builtin_bit_cast(v8bf, kind == 4 ? low : w[c][WP[kind] & 1]);
                    v16f& acc = kind == 5 ? big : small;
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(v8bf, x[c % 2][XP[kind]]), acc, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (kind == 1 && c + 1 < CHUNKS) gather(c + 1);
                    if constexpr (m % 2 == 1 && m / 2 < N_SLICES) finish_slice(m / 2, rs);
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* every operand has been read */
            done_first = (uint32_t) d_cur.x;
            done_at = valid ? own * OUTB + (uint32_t) (h * 4) * 4 : NOWHERE;
#pragma unroll
            for (int v = 0; v < 16; ++v) done[v] = big[v] + small[v];
        }
        /* the last tile's results; and no LDS load may outlive the wave */
        {
            const __amdgpu_buffer_rsrc_t rs = out_window();
#pragma unroll
            for (int i = 0; i < N_SLICES; ++i) finish_slice(i, rs);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    else {
        __syncthreads(); /* biases and low parts are in LDS */
    }

    /* tiles with more halo rows than are staged: every neighbour straight from memory, the operands of DEEP steps under way at once */
    constexpr int DEEP = 4;
    for (int t = blockIdx.x; t < n_far; t += gridDim.x) {
        const int4 d = B.tile_desc[B.far_tiles[t]];
        const uint32_t first = (uint32_t) d.x, in_use = (uint32_t) d.y, frame_row = (uint32_t) d.w;
        const uint32_t row = (uint32_t) (wave * 32 + r32), own = min(row, in_use - 1);
        uint32_t from[SLOTS];
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) from[s] = s == 0 ? first + own : frame_row + (uint32_t) B.row_nb[(size_t) (first + own) * B.nb_stride + (s - 1)];
        v16f big, small;
        start_sums(big, small);
        v4f ring[DEEP][2];
        auto request = [&](int c) {
            const float* const p = in + (size_t) from[c / J] * C_IN + (c % J) * 16 + h * 8;
            ring[c % DEEP][0] = *reinterpret_cast<const v4f*>(p), ring[c % DEEP][1] = *reinterpret_cast<const v4f*>(p + 4);
        };
#pragma unroll
        for (int c = 0; c < DEEP; ++c) request(c);
        static_for<CHUNKS>([&](auto chunk) {
            constexpr int c = decltype(chunk)::value;
            v4u x[3];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const Parts p = split_pair(ring[c % DEEP][q >> 1][(q & 1) * 2], ring[c % DEEP][q >> 1][(q & 1) * 2 + 1]);
                x[0][q] = p.high, x[1][q] = p.middle, x[2][q] = p.low;
            }
            if constexpr (c + DEEP < CHUNKS) request(c + DEEP);
            const v4u low = low_lds[c * 64];
            static_for<6>([&](auto kind_tag) {
                constexpr int kind = decltype(kind_tag)::value;
                const v8bf a = __builtin_bit_cast(v8bf, kind == 4 ? low : w[c][WP[kind] & 1]);
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
                *reinterpret_cast<v4f*>(out + (size_t) (first + row) * C_OUT + g * 8 + h * 4) = o;
            }
        }
    }
}

template <int C_IN, int ACT>
int launch_x3_tile(const VmBatchDev& B, const VmLayerDev& L, const float* in, float* out, hipStream_t stream) {
    constexpr size_t lds = tile_lds_bytes(C_IN);
    static_assert(lds <= 160 * 1024, "the block must fit the CU's LDS");
    auto kernel = vm_conv_x3_tile_kernel<C_IN, ACT>;
    static std::atomic<bool> configured{false}; /* engines on several host threads may get here together */
    if (!configured) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)) != hipSuccess) {
            (void) hipGetLastError();
            return -1;
        }
        configured = true;
    }
    /* one block per CU; the kernel reads the number of tiles in use on the device */
    hipLaunchKernelGGL(kernel, dim3(256), dim3(NT), lds, stream, B, L, in, out);
    return 0;
}

}  // namespace

/* Weight layout the kernel consumes: [step c = slot * c_in / 16 + j][part: h, m, l][lane = half * 32 + o][e = 0..7] bf16 of
 * W[slot * c_in + j * 16 + half * 8 + e][o] */
size_t vm_x3_tile_weight_bytes(int c_in) { return size_t(steps(c_in)) * 3 * 64 * 16; }
void vm_x3_tile_permute_weights(const float* w, int c_in, void* wp) {
    uint16_t* dst = reinterpret_cast<uint16_t*>(wp);
    for (int c = 0; c < steps(c_in); ++c)
        for (int lane = 0; lane < 64; ++lane)
            for (int e = 0; e < 8; ++e) {
                float v = w[(size_t(c) * 16 + (lane >> 5) * 8 + e) * C_OUT + (lane & 31)];
                for (int p = 0; p < 3; ++p) {
                    const uint16_t part = bf16_round(v);
                    dst[((size_t(c) * 3 + p) * 64 + lane) * 8 + e] = part;
                    v -= bf16_value(part);
                }
            }
}

bool vm_x3_tile_supported(int c_in, int c_out, int slots, int activation) {
    return (c_in == 16 || c_in == 32) && c_out == C_OUT && slots == SLOTS && (activation == VMHIP_SELU || activation == VMHIP_RELU);
}

int vm_launch_conv_x3_tile(const VmBatchDev& B, const VmLayerDev& L, const float* in, float* out, hipStream_t stream, const char** kernel_name) {
    if (B.n_row_tiles <= 0) return 0;
    if (!B.row_nbl || !B.tile_halo || !B.tile_desc || !B.far_tiles || !L.w_x3 || !vm_x3_tile_supported(L.c_in, L.c_out, L.slots, L.activation)) return -1;
    if (kernel_name) *kernel_name = vm_kernel_name("conv_x3_tile", L.c_in, L.c_out, L.slots);
    const bool selu = L.activation == VMHIP_SELU;
    if (L.c_in == 16) return selu ? launch_x3_tile<16, VMHIP_SELU>(B, L, in, out, stream) : launch_x3_tile<16, VMHIP_RELU>(B, L, in, out, stream);
    return selu ? launch_x3_tile<32, VMHIP_SELU>(B, L, in, out, stream) : launch_x3_tile<32, VMHIP_RELU>(B, L, in, out, stream);
}
