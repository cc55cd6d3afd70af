// vcsr_tile_row.hip - the tile-stationary SpMM on single-row tiles (gfx950).
// See vcsr_tile.hip for the view and the other tile heights.
//
// A wave takes MERGE consecutive work items of the view, at most PE*MERGE
// entries (PE the view's largest piece, 64 or 128) and 32*MERGE pieces (a piece is a row, or a part of a very long
// one).  The wave is S = 64/LPE streams of LPE lanes; each stream takes an
// equal run of the wave's entries, and one load instruction fetches one
// entry's B slice (LPE*VEC columns) for every stream.
//  1. Staging, lane per entry: the entry records (value, B row, and whether
//     the entry ends its piece) and the pieces' destinations are read with
//     all loads in flight at once.  The records go to LDS as (B-row byte
//     offset, value), each stream's run padded with "no row" entries of value
//     0 to the common length, so that the loop needs no index check; the end
//     marks become bit masks, from whose prefix counts every stream knows its
//     first piece without a search.
//  2. Blocks of U loads back to back, then their FMAs; where an entry ends
//     its piece the sum is stored and cleared.
//  3. A piece cut between runs is finished by the stream that began it, from
//     the later streams' partial sums in LDS, added in stream order.
// B is read with raw buffer loads whose range check turns "no row" offsets
// into zeros; a B of 2 GB or more is read at 64-bit addresses and "no row"
// entries select zero.  A row holds only entries it has, so a non-finite B
// needs no second pass.
// Bound by L2 misses (one 128-byte line per random B slice at narrow B, the
// slices themselves at wide B) and by the waves' chain of loads on smaller
// matrices.  Against one kernel with a path for several pieces and one for a
// long piece, and a piece table of 16 bytes per piece read after the entries:
// 39 instead of 55 registers at O = 8, 21 instead of 29 bytes of view per
// two-entry row, one round of loads, no bounds test per entry, and 16-byte
// lanes at any width.  Three formats in turn, us per SpMM: power-law 322K, O
// = 8 24.0 -> 22.2; 100K, O = 20 / 47 / 257 18.3 / 23.4 / 121 -> 15.5 / 20.9 /
// 85; uniform 27K x 14, O = 12 10.0 -> 6.1; banded 60K x 30, O = 50 32.8 ->
// 25.1; uniform 102K x 6, O = 200 107 -> 88; C += A*B, power-law 100K, O = 47
// 34.2 -> 29.2.
#include <type_traits>

#include "../host/tile_view.hpp"
#include "common.hpp"
#include "launch.hpp"
#include "vecops.hpp"

namespace vcsr {
namespace {

constexpr int kWaves = 2;

template <int VEC, int LPE, int MERGE, int PE>
struct RowShape {
    static constexpr int S = 64 / LPE;                          // streams
    static constexpr int EMAX = PE * MERGE;                     // entries per wave
    static constexpr int PMAX = kTileChunkPieces * MERGE;       // pieces per wave
    static constexpr int UT = 2;                                // runs are multiples of this
    static constexpr int IE = EMAX / 64, IP = (PMAX + 63) / 64;
    // Entries from one stream's run to the next in LDS: two more than the
    // run, so that the streams' reads fall into different banks.
    static constexpr int LIST = EMAX + S * (UT + 2);
    static_assert(EMAX / S % UT == 0, "S runs fit into EMAX entries");
    static constexpr int WORDS = EMAX / 32 + 2;
};

template <int VEC, int LPE, int MERGE, int PE>
struct RowLds {
    using Sh = RowShape<VEC, LPE, MERGE, PE>;
    __align__(16) uint2 ent[Sh::LIST];        // (B-row byte offset, value bits)
    typename VecT<VEC>::T xs[Sh::S > 1 ? 64 : 1];  // partial sums of pieces begun earlier
    int32_t dest[Sh::PMAX];                   // row, or ~partial row
    uint32_t ends[Sh::WORDS];                 // bit i: entry i ends its piece
    int32_t first[Sh::S];                     // first piece of each stream's run ...
    int32_t carry[Sh::S];                     // ... and whether it began in an earlier run
};

template <int VEC, int LPE, int MERGE, int PE, bool BUF, bool ACC>
__global__ __launch_bounds__(64 * kWaves)
void vcsr_row_kernel(
    int32_t n_items, int32_t O, int32_t ld, uint32_t b_bytes,
    const int2* __restrict__ items, const int32_t* __restrict__ dest,
    const float2* __restrict__ ent, const float* __restrict__ B, float* __restrict__ C,
    float* __restrict__ partials) {
    using V = typename VecT<VEC>::T;
    using Sh = RowShape<VEC, LPE, MERGE, PE>;
    constexpr int S = Sh::S, UT = Sh::UT, IE = Sh::IE, IP = Sh::IP;
    // Loads per block: 8; 4 where the rows of C are loaded with them (8 cost
    // two waves per SIMD: uniform 395K x 5, O = 32 65.8 / 74.1 us, power-law
    // 322K, O = 128 167.5 / 178.0; without C's rows 4 are 0-3% slower).
    constexpr int U = ACC && VEC == 4 ? 4 : 8;
    __shared__ RowLds<VEC, LPE, MERGE, PE> s_lds[kWaves];

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    const int32_t w = (int32_t)(xcd_remap(blockIdx.x, gridDim.x) * kWaves) + wave;
    const int32_t c0 = w * MERGE;
    if (c0 >= n_items) return;
    const int32_t c1 = min(n_items, c0 + MERGE);
    RowLds<VEC, LPE, MERGE, PE>& L = s_lds[wave];
    // Items are {first entry, first piece}.
    const int32_t e0 = uniform(items[c0].x), ne = uniform(items[c1].x) - e0;
    const int32_t p0 = uniform(items[c0].y), np = uniform(items[c1].y) - p0;
    // Entries per stream.
    const int32_t run = ((ne + S - 1) / S + UT - 1) / UT * UT;

    float2 rec[IE];
    int32_t ds[IP];
#pragma unroll
    for (int it = 0; it < IE; ++it) rec[it] = ent[(int64_t)e0 + min(it * 64 + lane, ne - 1)];
#pragma unroll
    for (int it = 0; it < IP; ++it) ds[it] = dest[(int64_t)p0 + min(it * 64 + lane, np - 1)];

    const uint32_t row_bytes = (uint32_t)ld * 4u;
    // i / run for i < 1024 by multiplication (exact: run < 1024).
    const uint32_t inv = (1u << 20) / (uint32_t)run + 1u;
    int32_t before = 0, last = 1;  // ends before this round; whether the entry before it is one
#pragma unroll
    for (int it = 0; it < IE; ++it) {
        const int32_t i = it * 64 + lane;
        if (it * 64 >= S * run) break;  // S*run <= EMAX
        const bool in = i < ne;
        const uint32_t word = in ? __builtin_bit_cast(uint32_t, rec[it].y) : 0u;
        const uint64_t m = __ballot(word >> 31);
        if (i < S * run) {
            const uint32_t br = word & 0x7fffffffu;
            const bool real = in && br != (uint32_t)kTileNoRow;
            const int32_t s = (int32_t)(((uint32_t)i * inv) >> 20), j = i - s * run;
            uint2 x;
            x.x = real ? (BUF ? br * row_bytes : br) : kNoRow;
            x.y = in ? __builtin_bit_cast(uint32_t, rec[it].x) : 0u;
            L.ent[s * (run + 2) + j] = x;
            if (j == 0) {
                const uint32_t prev = lane == 0 ? (uint32_t)last : (uint32_t)(m >> ((lane - 1) & 63)) & 1u;
                L.first[s] = before + (int32_t)__builtin_amdgcn_mbcnt_hi(
                                          (uint32_t)(m >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                L.carry[s] = in && prev == 0u;
            }
        }
        if (lane < 2) L.ends[2 * it + lane] = (uint32_t)(m >> (32 * lane));
        before += __popcll(m);
        last = (int32_t)(m >> 63);
    }
#pragma unroll
    for (int it = 0; it < IP; ++it) {
        const int32_t i = it * 64 + lane;
        if (i < np) L.dest[i] = ds[it];
    }
    wave_sync();

    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), (short)0, (int)b_bytes,
                                          kRawBufferFlags);
    const int sub = lane / LPE, kl = lane % LPE;
    const int32_t k = kl * VEC;
    const bool kok = k < O;
    const uint32_t koff = (uint32_t)vec_col<VEC>(k, O) * 4u;
    const uint2* le = L.ent + sub * (run + 2);
    const int32_t tb = sub * run;

    auto load_b = [&](uint32_t off) -> V {
        if constexpr (BUF) {
            return load_b_buf<VEC>(rsrc, off + koff);
        } else {
            const bool real = off != kNoRow;
            const V b = load_mem(B + (int64_t)(real ? off : 0u) * ld + koff / 4, V());
            return real ? b : zero_vec(V());
        }
    };
    const int32_t kc = vec_col<VEC>(k, O);
    auto load_c = [&](int32_t p) -> V {
        const int32_t d = L.dest[p];
        return d >= 0 ? load_mem(C + (int64_t)d * ld + kc, V()) : zero_vec(V());
    };
    // Stores the sum x of piece p; c are the row's values in C.
    auto store_piece = [&](int32_t p, V x, const V& c) {
        const int32_t d = L.dest[p];
        if (!kok) return;
        if (d >= 0) {
            if constexpr (ACC) x = add_vec(c, x);
            store_cols<VEC, true>(C + (int64_t)d * ld, k, O, x, false);
        } else {
            store_cols<VEC, false>(partials + (int64_t)~d * O, k, O, x, false);
        }
    };

    int32_t p = L.first[sub];
    bool carry = S > 1 && L.carry[sub] != 0;
    V acc = zero_vec(V());
    auto block = [&](auto n_c, int32_t i0) {
        constexpr int NU = decltype(n_c)::value;
        uint2 r[NU];
        V b[NU];
#pragma unroll
        for (int u = 0; u < NU; u += 2) {
            const uint4 x = *reinterpret_cast<const uint4*>(le + i0 + u);
            r[u] = make_uint2(x.x, x.y);
            r[u + 1] = make_uint2(x.z, x.w);
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) b[u] = load_b(r[u].x);
        // End bits of entries tb + i0 .. + NU - 1.
        const int32_t t = tb + i0;
        const uint32_t bits = __builtin_amdgcn_alignbit(L.ends[(t >> 5) + 1], L.ends[t >> 5], t & 31);
        // C += A*B: the rows that end in this block are read with its B
        // slices, so that a row's end does not wait for memory.
        V c[ACC ? NU : 1];
        if constexpr (ACC) {
#pragma unroll
            for (int u = 0; u < NU; ++u)
                if (bits & (1u << u)) c[u] = load_c(p + __popc(bits & ((1u << u) - 1u)));
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            fma_vec(acc, __builtin_bit_cast(float, r[u].y), b[u]);
            if (bits & (1u << u)) {
                if (S > 1 && carry) {
                    // The end of a piece begun in an earlier run.
                    L.xs[lane] = acc;
                    carry = false;
                } else {
                    store_piece(p, acc, c[ACC ? u : 0]);
                }
                acc = zero_vec(V());
                ++p;
            }
        }
    };
    int32_t i0 = 0;
    for (; i0 + U <= run; i0 += U) block(std::integral_constant<int, U>(), i0);
    if (i0 + U / 2 <= run) {
        block(std::integral_constant<int, U / 2>(), i0);
        i0 += U / 2;
    }
    if constexpr (U / 4 >= UT)
        if (i0 + U / 4 <= run) block(std::integral_constant<int, U / 4>(), i0);

    if constexpr (S > 1) {
        // A run that ends inside a piece: its owner adds the following runs'
        // partial sums; a run that lies wholly inside one leaves its own.
        if (carry) L.xs[lane] = acc;
        wave_sync();
        const bool open = sub + 1 < S && L.carry[sub + 1 < S ? sub + 1 : sub] != 0;
        if (open && !carry) {
            for (int s2 = sub + 1; s2 < S && L.carry[s2] != 0 && L.first[s2] == p; ++s2)
                acc = add_vec(acc, L.xs[s2 * LPE + kl]);
            store_piece(p, acc, ACC ? load_c(p) : zero_vec(V()));
        }
    }
}

template <int VEC, int LPE, int MERGE, int PE, bool BUF>
hipError_t launch_shape(const DeviceFmt& d, const float* B, int32_t O, int32_t ld, float* C,
                        int32_t accumulate, uint32_t b_bytes, float* partials, hipStream_t st) {
    constexpr int per = MERGE * kWaves;
    const dim3 grid((unsigned)(((int64_t)d.tv_n_chunks + per - 1) / per)), block(64 * kWaves);
    auto go = [&](auto acc) {
        hipLaunchKernelGGL((vcsr_row_kernel<VEC, LPE, MERGE, PE, BUF, decltype(acc)::value>), grid,
                           block, 0, st, d.tv_n_chunks, O, ld, b_bytes,
                           reinterpret_cast<const int2*>(d.tv_items), d.tv_dest,
                           reinterpret_cast<const float2*>(d.tv_val), B, C, partials);
        return hipGetLastError();
    };
    return accumulate ? go(std::true_type()) : go(std::false_type());
}

template <int X>
using I = std::integral_constant<int, X>;

}  // namespace

hipError_t launch_vcsr_row_tiles(const DeviceFmt& d, const float* B, int32_t O, int32_t ld,
                                 float* C, int32_t accumulate, uint64_t b_bytes, float* partials,
                                 hipStream_t st) {
    if (d.tv_n_chunks <= 0) return hipSuccess;
    if (b_bytes >= kBufferLimit) {
        constexpr int PE = tile_piece_entries(1);
        if (O < 4)
            return launch_shape<1, 64, 1, PE, false>(d, B, O, ld, C, accumulate, 0u, partials, st);
        return launch_shape<4, 64, 1, PE, false>(d, B, O, ld, C, accumulate, 0u, partials, st);
    }
    auto go_pe = [&](auto vec, auto lpe, auto merge, auto pe) {
        return launch_shape<decltype(vec)::value, decltype(lpe)::value, decltype(merge)::value,
                            decltype(pe)::value, true>(d, B, O, ld, C, accumulate,
                                                       (uint32_t)b_bytes, partials, st);
    };
    auto go = [&](auto vec, auto lpe, auto merge) {
        return d.tv_piece > kTileRowPiece ? go_pe(vec, lpe, merge, I<tile_piece_entries(1)>())
                                          : go_pe(vec, lpe, merge, I<kTileRowPiece>());
    };
    // Work items per wave.  us per SpMM, three formats in turn (the view comes
    // from beyond L2), 1 / 2 / 4 items:
    //  - O <= 32: as many as leave 4 waves per SIMD.  Power-law 322K rows (57K
    //    items), O = 8 29.6 / 24.6 / 22.8; 100K rows (17K), O = 8 14.1 / 13.4 /
    //    12.9; uniform 27K x 14 (13K), O = 12 7.7 / 6.2 / 6.8; uniform 20K x 10
    //    (7K), O = 16 5.1 / 5.3 / 6.3; 8 items 27.4 on the first.
    //  - wider: 2 where the items mostly hold one piece (rows of more than 16
    //    entries), else 1.  Banded 60K x 30, O = 50 / 64 30.7 / 24.9 / 24.9 and
    //    29.2 / 22.6 / 22.5; uniform 137K x 11, O = 64 54.9 / 57.4 / 56.9;
    //    power-law 100K, O = 47 22.0 / 24.7 / 25.3, 322K, O = 128 109.7 / 113.6
    //    / 126.4 (longer waves leave the XCD's range of B later).
    const int64_t items = d.tv_n_chunks, simds = 4 * (int64_t)device_cus(d.device);
    const bool single = (int64_t)d.tv_n_pieces < 2 * items;
    auto narrow = [&](auto vec, auto lpe) {
        return items >= 16 * simds  ? go(vec, lpe, I<4>())
               : items >= 8 * simds ? go(vec, lpe, I<2>())
                                    : go(vec, lpe, I<1>());
    };
    auto wide = [&](auto lpe) {
        return single && items >= 8 * simds ? go(I<4>(), lpe, I<2>()) : go(I<4>(), lpe, I<1>());
    };
    if (O <= 8) return narrow(I<1>(), I<8>());
    // 8 lanes of 2 floats: power-law 100K / 322K, O = 16 13.3 / 26.4 us against
    // 14.6 / 28.4 with 16 lanes of 1 (half the load instructions).
    if (O <= 16) return narrow(I<2>(), I<8>());
    if (O <= 32) return narrow(I<4>(), I<8>());
    if (O <= 64) return wide(I<16>());
    if (O <= 128) return wide(I<32>());
    return wide(I<64>());
}

}  // namespace vcsr
