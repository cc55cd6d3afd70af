// vcsr_tile_row.hip - the tile-stationary SpMM on single-row tiles (gfx950).
// See vcsr_tile.hip for the view and the other tile heights.
//
// A wave takes MERGE consecutive work items of the view, at most PE*MERGE
// entries (PE the view's largest piece, 64 or 128) and 32*MERGE pieces (a piece
// is a row, or a part of a very long one).  The wave is S = 64/LPE streams of
// LPE lanes; each stream takes an equal run of the wave's entries, and one load
// instruction fetches one entry's B slice (LPE*VEC columns) for every stream.
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
//     the later streams' partial sums in LDS, added in stream order; their
//     number comes from one ballot.  A wave of one piece adds its streams'
//     sums in a butterfly instead and has neither masks nor a step for ends
//     (banded 8K x 25, O = 16 / 64 4.1 / 5.5 us with the masks, 3.9 / 5.0; 30K x
//     40, O = 12 9.3 / 8.5).
// B is read with raw buffer loads whose range check turns "no row" offsets
// into zeros; a B of 2 GB or more is read at 64-bit addresses and "no row"
// entries select zero.  A row holds only entries it has, so a non-finite B
// needs no second pass.
// Bound by L2 misses (one 128-byte line per random B slice at narrow B, the
// slices themselves at wide B) and by the waves' chain of loads on smaller
// matrices: the runs' sums read one after the other, each behind two reads
// that said whether to go on, cost more than the loop there (banded 8K x 20, O
// = 8 / 32 5.2 / 5.7 us, 3.6 / 3.7 with the ballot and the butterfly).
// Against one kernel with a path for several pieces and one for a long piece,
// and a piece table of 16 bytes per piece read after the entries: 38 instead of
// 55 registers at O = 8, 21 instead of 29 bytes of view per two-entry row, one
// round of loads, no bounds test per entry, and 16-byte lanes at any width.
// Three formats in turn, us per SpMM: power-law 322K, O = 8 24.0 -> 21.7; 100K,
// O = 20 / 47 / 257 18.2 / 23.2 / 121 -> 14.4 / 20.7 / 87; banded 60K x 30, O =
// 50 32.8 -> 24.7; uniform 102K x 6, O = 200 107 -> 87; C += A*B, power-law
// 100K, O = 47 34.2 -> 28.6.
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

// What becomes of C: written (C = A*B), or added to (C += A*B), whose rows are
// then read ahead of their pieces' ends, so that an end does not wait for
// memory: a block's rows together with its B slices where pieces are short,
// each piece's row where the piece begins where they are long (one row in
// registers instead of one per entry of a block); or at the piece's end, where
// other waves or streams work meanwhile (launch_shape).
enum RowOut { kRowWrite, kRowAddShort, kRowAddLong, kRowAddLate };

// Stores a piece's sum x, columns k and on, to row d of C or partial row ~d; c
// are the row's values in C.
template <int VEC, RowOut OUT, class V>
__device__ __forceinline__ void store_row(float* C, float* partials, int32_t ld, int32_t O,
                                          int32_t k, int32_t d, V x, V c) {
    if (d >= 0) {
        float* row = C + (int64_t)d * ld;
        if constexpr (OUT == kRowAddLate) c = load_mem(row + vec_col<VEC>(k, O), V());
        if constexpr (OUT != kRowWrite) x = add_vec(c, x);
        store_cols<VEC, true>(row, k, O, x, false);
    } else {
        store_cols<VEC, false>(partials + (int64_t)~d * O, k, O, x, false);
    }
}

template <int VEC, int LPE, int MERGE, int PE, bool BUF, RowOut OUT>
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
    // 322K, O = 128 167.5 / 178.0; without C's rows 4 are 0-3% slower), and
    // where a row of C is held for short runs (banded 120K x 20, O = 64 38.9 / 37.6).
    constexpr int U = VEC == 4 && (OUT == kRowAddShort || (OUT == kRowAddLong && LPE <= 16)) ? 4 : 8;
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
    // Writes the staged lists to LDS; `one`: the wave holds one piece, which
    // needs no masks and no first pieces.
    auto stage = [&](auto one) {
        constexpr bool ONE = decltype(one)::value;
        int32_t before = 0, last = 1;  // ends before this round; whether the entry before it is one
#pragma unroll
        for (int it = 0; it < IE; ++it) {
            const int32_t i = it * 64 + lane;
            if (it * 64 >= S * run) break;  // S*run <= EMAX
            const bool in = i < ne;
            const uint32_t word = in ? __builtin_bit_cast(uint32_t, rec[it].y) : 0u;
            const uint64_t m = ONE ? 0u : __ballot(word >> 31);
            if (i < S * run) {
                const uint32_t br = word & 0x7fffffffu;
                const bool real = in && br != (uint32_t)kTileNoRow;
                const int32_t s = (int32_t)(((uint32_t)i * inv) >> 20), j = i - s * run;
                uint2 x;
                x.x = real ? (BUF ? br * row_bytes : br) : kNoRow;
                x.y = in ? __builtin_bit_cast(uint32_t, rec[it].x) : 0u;
                L.ent[s * (run + 2) + j] = x;
                if (!ONE && j == 0) {
                    const uint32_t prev =
                        lane == 0 ? (uint32_t)last : (uint32_t)(m >> ((lane - 1) & 63)) & 1u;
                    L.first[s] = before + (int32_t)__builtin_amdgcn_mbcnt_hi(
                                              (uint32_t)(m >> 32),
                                              __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                    L.carry[s] = in && prev == 0u;
                }
            }
            if constexpr (!ONE) {
                if (lane < 2) L.ends[2 * it + lane] = (uint32_t)(m >> (32 * lane));
                before += __popcll(m);
                last = (int32_t)(m >> 63);
            }
        }
        if constexpr (!ONE) {
#pragma unroll
            for (int it = 0; it < IP; ++it) {
                const int32_t i = it * 64 + lane;
                if (i < np) L.dest[i] = ds[it];
            }
        }
        wave_sync();
    };

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
    auto load_c = [&](int32_t d) -> V {
        return d >= 0 ? load_mem(C + (int64_t)d * ld + kc, V()) : zero_vec(V());
    };
    auto store_to = [&](int32_t d, V x, V c) {
        if (kok) store_row<VEC, OUT>(C, partials, ld, O, k, d, x, c);
    };
    auto store_piece = [&](int32_t p, V x, V c) { store_to(L.dest[p], x, c); };

    int32_t p = 0;       // the stream's piece ...
    bool carry = false;  // ... and whether it began in an earlier run
    V acc = zero_vec(V());
    V c_next = zero_vec(V());  // a row of C read ahead of its piece's end
    // Entries i0 .. i0 + NU - 1 of every stream's run; `ends`: pieces may end
    // among them.
    auto block = [&](auto n_c, auto ends, int32_t i0) {
        constexpr int NU = decltype(n_c)::value;
        constexpr bool ENDS = decltype(ends)::value;
        uint32_t off[NU];
        float a[NU];
        V b[NU];
#pragma unroll
        for (int u = 0; u < NU; u += 2) {
            const uint4 x = *reinterpret_cast<const uint4*>(le + i0 + u);
            off[u] = x.x, a[u] = __builtin_bit_cast(float, x.y);
            off[u + 1] = x.z, a[u + 1] = __builtin_bit_cast(float, x.w);
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) b[u] = load_b(off[u]);
        // End bits of entries tb + i0 .. + NU - 1.
        const int32_t t = tb + i0;
        const uint32_t bits =
            ENDS ? __builtin_amdgcn_alignbit(L.ends[(t >> 5) + 1], L.ends[t >> 5], t & 31) : 0u;
        V c[OUT == kRowAddShort ? NU : 1];
        if constexpr (ENDS && OUT == kRowAddShort) {
            int32_t d[NU];
#pragma unroll
            for (int u = 0; u < NU; ++u)
                d[u] = L.dest[min(p + (int32_t)__popc(bits & ((1u << u) - 1u)), np - 1)];
#pragma unroll
            for (int u = 0; u < NU; ++u)
                if (bits & (1u << u)) c[u] = load_c(d[u]);
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            fma_vec(acc, a[u], b[u]);
            if (ENDS && (bits & (1u << u))) {
                if (S > 1 && carry) {
                    // The end of a piece begun in an earlier run.
                    L.xs[lane] = acc;
                    carry = false;
                } else {
                    store_piece(p, acc, OUT == kRowAddShort ? c[u] : c_next);
                }
                acc = zero_vec(V());
                ++p;
                if constexpr (OUT == kRowAddLong) {
                    if (p < np) c_next = load_c(L.dest[p]);
                }
            }
        }
    };
    auto walk = [&](auto ends) {
        int32_t i0 = 0;
        for (; i0 + U <= run; i0 += U) block(std::integral_constant<int, U>(), ends, i0);
        if (i0 + U / 2 <= run) {
            block(std::integral_constant<int, U / 2>(), ends, i0);
            i0 += U / 2;
        }
        if constexpr (U / 4 >= UT)
            if (i0 + U / 4 <= run) block(std::integral_constant<int, U / 4>(), ends, i0);
    };

    if constexpr (MERGE == 1 && S > 1) {
        // One piece in the wave: nothing ends before the last entry, and the
        // streams' sums meet in a butterfly.
        if (np == 1) {
            stage(std::true_type());
            const int32_t d = uniform(ds[0]);
            V c = zero_vec(V());
            if (OUT != kRowWrite && OUT != kRowAddLate && sub == 0) c = load_c(d);
            walk(std::false_type());
#pragma unroll
            for (int sh = LPE; sh < 64; sh <<= 1) acc = add_vec(acc, shfl_xor_vec(acc, sh));
            if (sub == 0) store_to(d, acc, c);
            return;
        }
    }
    stage(std::false_type());
    p = L.first[sub];
    carry = S > 1 && L.carry[sub] != 0;

    // The row of C of the piece that this stream begins and the next run opens
    // with (the stream finishes it below), or of its first piece.
    const int32_t p_first = p;
    const int nsub = sub + 1 < S ? sub + 1 : sub;
    if constexpr (OUT == kRowAddShort && S > 1) {
        const int32_t p_open = L.first[nsub];
        if (nsub > sub && L.carry[nsub] != 0 && !(carry && p_open == p_first))
            c_next = load_c(L.dest[p_open]);
    }
    if constexpr (OUT == kRowAddLong) {
        if (!carry && p < np) c_next = load_c(L.dest[p]);
    }
    walk(std::true_type());

    if constexpr (S > 1) {
        // A piece cut between runs: its owner adds the following runs' partial
        // sums, in stream order, up to the run in which it ends (a run that
        // lies wholly inside one leaves its own sum).  Their number comes from
        // one ballot, so that the sums are read without waiting in between.
        if (carry) L.xs[lane] = acc;
        const uint64_t ended = __ballot(p != p_first);
        wave_sync();
        if (nsub > sub && L.carry[nsub] != 0 && !carry) {
            const int more = __builtin_ctzll(ended >> (nsub * LPE)) / LPE;  // runs after the next one
            acc = add_vec(acc, L.xs[nsub * LPE + kl]);
            if (more > 0) {
                V x[S];
#pragma unroll
                for (int j = 1; j < S - 1; ++j) x[j] = L.xs[min(nsub + j, S - 1) * LPE + kl];
#pragma unroll
                for (int j = 1; j < S - 1; ++j)
                    if (j <= more) acc = add_vec(acc, x[j]);
            }
            store_piece(p, acc, c_next);
        }
    }
}

template <int VEC, int LPE, int MERGE, int PE, bool BUF>
hipError_t launch_shape(const DeviceFmt& d, const float* B, int32_t O, int32_t ld, float* C,
                        int32_t accumulate, uint32_t b_bytes, float* partials, hipStream_t st) {
    constexpr int per = MERGE * kWaves;
    const dim3 grid((unsigned)(((int64_t)d.tv_n_chunks + per - 1) / per)), block(64 * kWaves);
    auto go = [&](auto out) {
        hipLaunchKernelGGL((vcsr_row_kernel<VEC, LPE, MERGE, PE, BUF, decltype(out)::value>), grid,
                           block, 0, st, d.tv_n_chunks, O, ld, b_bytes,
                           reinterpret_cast<const int2*>(d.tv_items), d.tv_dest,
                           reinterpret_cast<const float2*>(d.tv_val), B, C, partials);
        return hipGetLastError();
    };
    if (!accumulate) return go(std::integral_constant<RowOut, kRowWrite>());
    // C += A*B, us per SpMM:
    //  - pieces of more than 16 entries on average: a row of C ahead of each piece
    //    (banded 30K x 40, O = 256 50.1 with a block's rows, 48.7 so); late where
    //    narrow waves hold several pieces, some streams of which end while others
    //    load (ahead / late: 30K x 40, O = 4 / 24 8.6 / 8.1 and 12.2 / 10.9; 60K x
    //    30, O = 16 / 64 14.8 / 13.5 and 25.4 / 24.7; 120K x 20, O = 24 25.7 / 23.8).
    //  - shorter ones: a block's rows with its B slices (power-law 322K, O = 47
    //    91.2 late, 75.5 so); late in narrow waves of one or two items (uniform
    //    20K x 10, O = 4 4.4 / 4.1; 100K x 5 8.5 / 7.1; with four, power-law 322K
    //    25.2 / 26.8).
    const bool long_pieces = d.tv_n_entries > 16 * (int64_t)d.tv_n_pieces;
    constexpr RowOut LONG = BUF && MERGE > 1 && VEC * LPE <= 64 ? kRowAddLate : kRowAddLong;
    constexpr RowOut SHORT = BUF && MERGE <= 2 && VEC * LPE == 8 ? kRowAddLate : kRowAddShort;
    return long_pieces ? go(std::integral_constant<RowOut, LONG>())
                       : go(std::integral_constant<RowOut, SHORT>());
}

template <int X>
using I = std::integral_constant<int, X>;

}  // namespace

// Whether the work items mostly hold one piece (rows of more than 16 entries).
static bool single_pieces(const DeviceFmt& d) {
    return (int64_t)d.tv_n_pieces < 2 * (int64_t)d.tv_n_chunks;
}

// Floats per lane.  Fewer floats on more lanes halve or quarter the streams that
// a piece is cut between, and so make one piece a wave cheap, but take more load
// instructions an entry: where items are single pieces, unless there are many
// and short ones, which then share waves.  us per SpMM, 1 float / several:
//  - 9 to 16 columns (16 lanes / 8 of 2), O = 16: banded 4K x 30 2.9 / 3.5, 30K x
//    40 8.6 / 9.2, 45K x 50 18.2 / 18.5, 60K x 70 23.3 / 24.7, 60K x 30 17.4 /
//    13.4, 120K x 20 30.3 / 18.6; items of several pieces: uniform 50K x 10 9.0 /
//    7.9, power-law 322K 26.4 / 24.1.
//  - 17 to 31 (32 / 8 of 4), O = 17 / 31: banded 8K x 25 4.3 / 4.9 and 4.4 / 5.4,
//    16K x 60 8.5 / 9.5 and 9.8 / 11.1, 24K x 50 13.0 / 14.8 and 14.7 / 16.6, 60K
//    x 30 16.7 / 14.8 and 18.3 / 17.7.  32 fill the 8 lanes (9K x 40 6.7 / 5.5).
//  - 33 to 63 that are no whole vectors of 4, short pieces (64 / 16 of 4), O = 47 /
//    63: 4K x 30 4.3 / 4.6 and 4.4 / 4.7, 15K x 30 8.2 / 8.7 and 8.9 / 9.3, 9K x 40
//    7.3 / 7.1; not C += A*B (4K x 30, O = 47 4.7 / 4.3).
int row_tiles_vec(const DeviceFmt& d, int32_t O) {
    if (O <= 8) return 1;
    const bool few = d.tv_n_chunks < 32 * (4 * (int64_t)device_cus(d.device));
    const bool mean32 = d.tv_n_entries > 32 * (int64_t)d.tv_n_pieces;
    const bool narrow = single_pieces(d) && (O < 32 ? few || mean32 : few && !mean32);
    if (O <= 16) return narrow ? 1 : 2;
    return narrow && (O < 32 || (O < 64 && O % 4 != 0)) ? 1 : 4;
}

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
    // Work items per wave: as many as still leave every SIMD its waves, fewer
    // where long waves leave the XCD's range of B late.  us per SpMM, two
    // formats in turn, 1 / 2 / 4 items:
    //  - several pieces an item: uniform 20K x 10 (7K items), O = 1 / 32 4.0 / 3.5
    //    / 4.2 and 5.1 / 4.7 / 5.7; power-law 100K (17K), O = 1 10.9 / 10.4 / 10.6;
    //    322K (57K), O = 1 / 8 / 32 23.6 / 19.3 / 18.1, 25.5 / 21.8 / 21.2 and
    //    31.2 / 28.6 / 30.1; wider always 1: power-law 100K, O = 47 21.0 / 22.8 /
    //    23.7, 322K, O = 128 107 / 111 / 125.
    //  - one piece an item: banded 8K x 60, O = 8 / 64 4.1 / 4.6 / 5.5 and 7.0 /
    //    7.4 / 8.1; 20K x 25, O = 8 5.9 / 5.8 / 5.1; 9K x 40, O = 32 5.1 / 5.4 / 5.5;
    //    30K x 40, O = 32 / 64 11.4 / 10.5 / 10.0 and 16.4 / 15.8 / 16.2; 120K x 20, O = 8 / 64 27.8 / 20.4 /
    //    15.9 and 39.3 / 32.3 / 42.6; O = 128: 45K x 50 47.5 / 48.3, 120K x 20 56.6
    //    / 53.4; O = 256: 120K x 20 137 / 133.
    const int64_t items = d.tv_n_chunks, simds = 4 * (int64_t)device_cus(d.device);
    const bool single = single_pieces(d);
    // Short pieces, up to 7 entries on average (2 to 6 in the matrices measured).
    const bool ends = d.tv_n_entries <= 7 * (int64_t)d.tv_n_pieces;
    // 9 to 32 columns, several pieces an item, us per SpMM at 1 / 2 / 4 items:
    // uniform 50K x 4, O = 16 / 20 / 27 4.0 / 4.4 / 5.1, 4.7 / 5.2 / 6.0 and 7.0 /
    // 8.1 / 7.8; 100K x 5, O = 20 11.7 / 13.1 / 13.4; 200K x 4, O = 27 30.9 / 34.1 /
    // 34.2; power-law 100K, O = 27 16.4 / 17.8 / 18.1, 200K, O = 12 20.4 / 19.3 /
    // 20.4; 40K x 8, O = 32 6.2 / 5.7 / 6.0; 60K x 14, O = 16 12.1 / 9.8 / 9.1; 100K
    // x 12, C += A*B, O = 12 21.7 / 15.0 / 13.7.
    const int many = items < (ends ? 32 : 5) * simds                                          ? 1
                     : items >= 24 * simds && d.tv_n_entries > 8 * (int64_t)d.tv_n_pieces ? 4
                                                                                               : 2;
    if (O <= 8) {
        // C += A*B on short pieces, O = 4: uniform 100K x 5, 1 / 2 items 7.0 / 7.9, 50K
        // x 4 4.1 / 4.4, power-law 60K 9.4 / 10.1; 40K x 8 4.9 / 4.8.
        const int64_t four = single ? 16 : 24;
        return items >= four * simds ? go(I<1>(), I<8>(), I<4>())
               : !single && !(accumulate && ends) && items >= 5 * simds
                   ? go(I<1>(), I<8>(), I<2>())
                   : go(I<1>(), I<8>(), I<1>());
    }
    if (O <= 16) {
        if (row_tiles_vec(d, O) == 1) return go(I<1>(), I<16>(), I<1>());
        return single || many == 4 ? go(I<2>(), I<8>(), I<4>())
               : many == 2         ? go(I<2>(), I<8>(), I<2>())
                                   : go(I<2>(), I<8>(), I<1>());
    }
    const bool narrow = row_tiles_vec(d, O) == 1;
    if (O < 32 && narrow) return go(I<1>(), I<32>(), I<1>());
    if (O < 64 && narrow && !accumulate) return go(I<1>(), I<64>(), I<1>());
    if (O <= 32)
        return (single ? items >= 16 * simds : many == 4) ? go(I<4>(), I<8>(), I<4>())
               : !single && many == 2                     ? go(I<4>(), I<8>(), I<2>())
                                                          : go(I<4>(), I<8>(), I<1>());
    if (O <= 64)
        return single && items >= 16 * simds ? go(I<4>(), I<16>(), I<2>())
                                             : go(I<4>(), I<16>(), I<1>());
    if (O <= 128)
        return single && items >= 48 * simds ? go(I<4>(), I<32>(), I<2>())
                                             : go(I<4>(), I<32>(), I<1>());
    return single && items >= 64 * simds ? go(I<4>(), I<64>(), I<2>())
                                         : go(I<4>(), I<64>(), I<1>());
}

}  // namespace vcsr
