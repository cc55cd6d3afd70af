// vcsr_tile_tall.hip - the tile-stationary SpMM on tiles of 2, 3, 4 or 8 rows
// (gfx950).  See vcsr_tile.hip for the view and the other tile heights.
//
// A wave takes G consecutive pieces of the view (a piece is a whole tile, or
// a part of a very long one), 64/G lanes each.  The lanes of a piece are S
// streams of LPE lanes; one load instruction fetches one entry's B slice
// (LPE*VEC columns) for every stream of every piece.
//  1. Staging: the piece's entries (B row and R values) are read lane per
//     entry, all loads of a segment in flight at once, and written to the
//     piece's LDS list as (values, B-row byte offset), padded with "no row"
//     entries of value 0 so that all streams of the wave run the same number
//     of steps: the loop has no per-load index clamp and no branch.
//  2. Entries t = sub + S*i: blocks of U loads back to back, then their FMAs
//     into the piece's R accumulator rows.
//  3. The streams' sums are added by an xor butterfly inside the piece's
//     lanes, and stream s stores rows s, s + S, ... .
// Bound by the L2-to-CU path (one B slice per entry) at wide B, by the view's
// arrival and the loads' latency at narrow B.  Against one kernel for all
// tile heights that packed several tiles per wave in stream mode: only this
// path's registers are held (54 instead of 94 at 3 rows and O = 128: 8 waves
// per SIMD instead of 5), a wave waits for one record and one round of entry
// loads instead of up to four loads in sequence, and short tiles share a wave
// without a per-entry test for the piece's end.  Banded 62K matrix, three
// formats in turn, O = 8 / 32 / 128 / 512: 17.3 / 22.9 / 34.5 / 151 -> 8.4 /
// 12.8 / 31.8 / 146 us; 30K rows of 6-row blocks, O = 50: 27.4 -> 13.2.
// Rows absent from an entry are updated with a zero value, which is exact for
// finite B; a piece with a non-finite sum is recomputed with the presence
// bits before it is stored.
#include <type_traits>

#include "../host/tile_view.hpp"
#include "common.hpp"
#include "launch.hpp"
#include "vecops.hpp"

namespace vcsr {
namespace {

constexpr int kWaves = 2;

// U loads per block.
template <int LPE, int S, int R, int U>
struct TallShape {
    static constexpr int TL = LPE * S;      // lanes per piece
    static constexpr int G = 64 / TL;       // pieces per wave
    static constexpr int UT = 2;            // the list is padded to S*UT entries
    // Entries staged at a time; longer pieces (8-row tiles) take several
    // rounds, which keeps the LDS list small.
    static constexpr int SEG = R == 2 ? 64 : R == 3 ? 96 : 128;
    static constexpr int VF = R <= 4 ? 4 : 8;  // value floats of a staged entry
    // Up to 3 rows the offset takes the values' padding slot: one 16-byte LDS
    // read gives the whole entry.
    static constexpr bool REC = R <= 3;
    static constexpr int IT = (SEG + TL - 1) / TL;
    static_assert(SEG % (S * UT) == 0, "padded list fits");
};

template <int LPE, int S, int R, int U>
struct TallLds {
    using Sh = TallShape<LPE, S, R, U>;
    // The lists of a wave's pieces start S entries further on in the banks.
    __align__(16) float val[Sh::G][(Sh::SEG + (Sh::G > 1 ? S : 0)) * Sh::VF];
    uint32_t off[Sh::REC ? 1 : Sh::G][Sh::REC ? 1 : Sh::SEG + (Sh::G > 1 ? S : 0)];
};

// What becomes of C: written (C = A*B), or added to (C += A*B), whose rows are
// then read ahead of everything else, or just before they are stored.
enum TallOut { kTallWrite, kTallAdd, kTallAddLate };

template <int VEC, int LPE, int S, int R, int U, bool BUF, TallOut OUT>
__global__ __launch_bounds__(64 * kWaves)
__attribute__((amdgpu_waves_per_eu(R <= 3 ? 5 : 1, 8)))
void vcsr_tall_kernel(
    int32_t n_pieces, int32_t O, int32_t ld, uint32_t b_bytes,
    const int4* __restrict__ pieces, const int32_t* __restrict__ ent_brow,
    const uint16_t* __restrict__ ent_mask, const float* __restrict__ ent_val,
    const float* __restrict__ B, float* __restrict__ C, float* __restrict__ partials) {
    using V = typename VecT<VEC>::T;
    using Sh = TallShape<LPE, S, R, U>;
    constexpr int TL = Sh::TL, G = Sh::G, UT = Sh::UT, SEG = Sh::SEG, VF = Sh::VF;
    constexpr int RS = tile_slot_stride(R);      // value floats per entry of the view
    constexpr bool FOLD = tile_dev_folds_brow(R);
    __shared__ TallLds<LPE, S, R, U> s_lds[kWaves];

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    const int32_t w = (int32_t)(xcd_remap(blockIdx.x, gridDim.x) * kWaves) + wave;
    if (w * G >= n_pieces) return;
    const int grp = G == 1 ? 0 : lane / TL, tl = lane % TL, sub = tl / LPE, kl = tl % LPE;

    // The piece: {first row, rows, first entry, partial row or -1}; its
    // entries end where the next piece's begin.
    int4 pc;
    int32_t ne;
    if constexpr (G == 1) {
        pc = make_int4(uniform(pieces[w].x), uniform(pieces[w].y), uniform(pieces[w].z),
                       uniform(pieces[w].w));
        ne = uniform(pieces[w + 1].z) - pc.z;
    } else {
        const int32_t p = w * G + grp, pp = min(p, n_pieces - 1);
        pc = pieces[pp];
        ne = pieces[pp + 1].z - pc.z;
        if (p >= n_pieces) ne = pc.y = 0;
    }
    const int64_t e0 = pc.z;
    int32_t ne_max = ne;
#pragma unroll
    for (int sh = TL; sh < 64; sh <<= 1) ne_max = max(ne_max, __shfl_xor(ne_max, sh));
    if constexpr (G > 1) ne_max = uniform(ne_max);

    const uint32_t row_bytes = (uint32_t)ld * 4u;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), (short)0, (int)b_bytes,
                                          kRawBufferFlags);
    const int32_t k = kl * VEC;
    const bool kok = k < O;
    const uint32_t koff = (uint32_t)vec_col<VEC>(k, O) * 4u;
    float* lv = s_lds[wave].val[grp];
    uint32_t* lo = s_lds[wave].off[Sh::REC ? 0 : grp];

    auto entry_brow = [&](int64_t e) -> uint32_t {
        return FOLD ? __builtin_bit_cast(uint32_t, ent_val[e * RS + RS - 1]) : (uint32_t)ent_brow[e];
    };
    auto load_b = [&](uint32_t off) -> V {
        if constexpr (BUF) return load_b_buf<VEC>(rsrc, off + koff);
        else return load_mem(B + (int64_t)off * ld + koff / 4, V());
    };

    // C += A*B: this stream's rows of C.
    constexpr int CR = (R + S - 1) / S;
    V c[OUT == kTallWrite ? 1 : CR];
    auto load_c = [&] {
#pragma unroll
        for (int i = 0; i < CR; ++i) {
            const int r = i * S + sub;
            c[i] = r < pc.y && pc.w < 0
                       ? load_mem(C + (int64_t)(pc.x + r) * ld + vec_col<VEC>(k, O), V())
                       : zero_vec(V());
        }
    };
    if constexpr (OUT == kTallAdd) load_c();

    V acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = zero_vec(V());

    for (int32_t s0 = 0; s0 < ne_max; s0 += SEG) {
        const int32_t steps = (min(ne_max - s0, SEG) + S * UT - 1) / (S * UT) * UT;  // per stream
        if (s0 > 0) wave_sync();
        {
            float a[Sh::IT][VF];
            uint32_t br[Sh::IT];
#pragma unroll
            for (int it = 0; it < Sh::IT; ++it) {
                const int64_t e = e0 + min(s0 + it * TL + tl, max(ne - 1, 0));
                if constexpr (RS == 2) {
                    const float2 x = *reinterpret_cast<const float2*>(ent_val + e * RS);
                    a[it][0] = x.x, a[it][1] = x.y, a[it][2] = 0.f, a[it][3] = 0.f;
                } else {
#pragma unroll
                    for (int q = 0; q < VF; q += 4) {
                        const float4 x = *reinterpret_cast<const float4*>(ent_val + e * RS + q);
                        a[it][q] = x.x, a[it][q + 1] = x.y, a[it][q + 2] = x.z, a[it][q + 3] = x.w;
                    }
                }
                br[it] = FOLD ? __builtin_bit_cast(uint32_t, a[it][VF - 1]) : (uint32_t)ent_brow[e];
            }
#pragma unroll
            for (int it = 0; it < Sh::IT; ++it) {
                const int32_t i = it * TL + tl;
                if (i < steps * S) {
                    const bool in = s0 + i < ne;
                    const bool real = in && br[it] != (uint32_t)kTileNoEntry;
                    const uint32_t off = BUF ? (real ? br[it] * row_bytes : kNoRow)
                                             : (real ? br[it] : 0u);
#pragma unroll
                    for (int q = 0; q < VF; ++q) a[it][q] = in ? a[it][q] : 0.f;
                    if constexpr (Sh::REC) a[it][3] = __builtin_bit_cast(float, off);
                    else lo[i] = off;
#pragma unroll
                    for (int q = 0; q < VF; q += 4)
                        *reinterpret_cast<float4*>(lv + i * VF + q) =
                            make_float4(a[it][q], a[it][q + 1], a[it][q + 2], a[it][q + 3]);
                }
            }
        }
        wave_sync();

        auto block = [&](auto n_c, int32_t i0) {
            constexpr int NU = decltype(n_c)::value;
            V b[NU];
            if constexpr (Sh::REC) {
                float4 rec[NU];
#pragma unroll
                for (int u = 0; u < NU; ++u)
                    rec[u] = *reinterpret_cast<const float4*>(lv + (sub + S * (i0 + u)) * VF);
#pragma unroll
                for (int u = 0; u < NU; ++u) b[u] = load_b(__builtin_bit_cast(uint32_t, rec[u].w));
#pragma unroll
                for (int u = 0; u < NU; ++u)
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        fma_vec(acc[r], reinterpret_cast<const float*>(&rec[u])[r], b[u]);
            } else {
#pragma unroll
                for (int u = 0; u < NU; ++u) b[u] = load_b(lo[sub + S * (i0 + u)]);
#pragma unroll
                for (int u = 0; u < NU; ++u) {
                    float4 x[VF / 4];
#pragma unroll
                    for (int q = 0; q < VF / 4; ++q)
                        x[q] = *reinterpret_cast<const float4*>(lv + (sub + S * (i0 + u)) * VF + 4 * q);
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        fma_vec(acc[r], reinterpret_cast<const float*>(x)[r], b[u]);
                }
            }
        };
        int32_t i0 = 0;
        for (; i0 + U <= steps; i0 += U) block(std::integral_constant<int, U>(), i0);
        if constexpr (U / 2 >= UT) {
            if (i0 + U / 2 <= steps) {
                block(std::integral_constant<int, U / 2>(), i0);
                i0 += U / 2;
            }
        }
        if constexpr (U / 4 >= UT) {
            if (i0 + U / 4 <= steps) {
                block(std::integral_constant<int, U / 4>(), i0);
                i0 += U / 4;
            }
        }
        if constexpr (U / 8 >= UT) {
            if (i0 + U / 8 <= steps) block(std::integral_constant<int, U / 8>(), i0);
        }
    }

#pragma unroll
    for (int sh = LPE; sh < TL; sh <<= 1) {
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = add_vec(acc[r], shfl_xor_vec(acc[r], sh));
    }
    // Finite exactly when every accumulator is (x * 0 is NaN for inf and NaN).
    float z = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) z = fma_zero_acc(acc[r], z);
    const uint64_t bad = __ballot(!__builtin_isfinite(z) && kok);
    if (bad != 0) {
        // In entry order, skipping the rows an entry does not have; every
        // stream of the piece computes the same sums.
        const uint64_t mine = TL == 64 ? ~0ull : ((1ull << (TL & 63)) - 1ull) << (grp * (TL & 63));
        if ((bad & mine) != 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] = zero_vec(V());
            for (int32_t t = 0; t < ne; ++t) {
                const uint32_t br = entry_brow(e0 + t), m = ent_mask[e0 + t];
                if (m == 0) continue;
                const V b = load_b(BUF ? br * row_bytes : br);
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if ((m >> r) & 1u) fma_vec(acc[r], ent_val[(e0 + t) * RS + r], b);
            }
        }
    }
    if (!kok) return;
    if constexpr (OUT == kTallAddLate) load_c();
#pragma unroll
    for (int i = 0; i < CR; ++i) {
        const int r = i * S + sub;
        if (r < R && r < pc.y) {
            V x = acc[0];
#pragma unroll
            for (int q = 1; q < R; ++q)
                if (q == r) x = acc[q];
            if constexpr (OUT != kTallWrite) x = add_vec(c[i], x);
            if (pc.w < 0)
                store_cols<VEC, true>(C + (int64_t)(pc.x + r) * ld, k, O, x, false);
            else
                store_cols<VEC, false>(partials + (int64_t)(pc.w + r) * O, k, O, x, false);
        }
    }
}

template <int VEC, int LPE, int S, int R, int U, bool BUF>
hipError_t launch_shape(const DeviceFmt& d, const float* B, int32_t O, int32_t ld, float* C,
                        int32_t accumulate, uint32_t b_bytes, float* partials, hipStream_t st) {
    constexpr int per = TallShape<LPE, S, R, U>::G * kWaves;
    const dim3 grid((unsigned)(((int64_t)d.tv_n_pieces + per - 1) / per)), block(64 * kWaves);
    auto go = [&](auto out) {
        hipLaunchKernelGGL((vcsr_tall_kernel<VEC, LPE, S, R, U, BUF, decltype(out)::value>), grid,
                           block, 0, st, d.tv_n_pieces, O, ld, b_bytes,
                           reinterpret_cast<const int4*>(d.tv_pieces), d.tv_brow, d.tv_mask,
                           d.tv_val, B, C, partials);
        return hipGetLastError();
    };
    if (!accumulate) return go(std::integral_constant<TallOut, kTallWrite>());
    // C is read ahead, except where the registers that its rows take cost waves
    // (2 and 3 rows, O > 128: 6 instead of 8 per SIMD at 3) that more waves than
    // are resident at once would fill, and where B and C fit into the 256 MB MALL
    // with room, so that a late read waits for little.  us per SpMM, ahead / late:
    // blocks of 2 rows, O = 256 62K x 24 58 / 44, 90K x 24 84 / 61; of 3 rows 62K x
    // 64 70 / 62, 120K x 24, O = 200 69 / 54; few waves: 12K x 64, 3 rows, O = 200
    // 13.5 / 14.5; B and C of 246 MB: 120K x 64, 3 rows, O = 256 132 / 149.
    if constexpr (VEC == 4 && LPE == 64 && R <= 3 && BUF) {
        const uint64_t c_bytes = (uint64_t)d.tv_n_pieces * R * (uint64_t)ld * 4u;
        if (d.tv_n_pieces > 32 * (int64_t)device_cus(d.device) && b_bytes + c_bytes <= (192ull << 20))
            return go(std::integral_constant<TallOut, kTallAddLate>());
    }
    return go(std::integral_constant<TallOut, kTallAdd>());
}

template <int X>
using I = std::integral_constant<int, X>;

template <int R>
hipError_t launch_rows(const DeviceFmt& d, const float* B, int32_t O, int32_t ld, float* C,
                       int32_t accumulate, uint64_t b_bytes, float* partials, hipStream_t st) {
    if (b_bytes >= kBufferLimit) {
        if (O < 4)
            return launch_shape<1, 64, 1, R, 8, false>(d, B, O, ld, C, accumulate, 0u, partials, st);
        return launch_shape<4, 64, 1, R, 8, false>(d, B, O, ld, C, accumulate, 0u, partials, st);
    }
    const uint32_t bb = (uint32_t)b_bytes;
    // The shape <floats per lane, lanes per entry, streams per piece, loads
    // per block> by width, and by the pieces' mean entry count where that
    // decides how many lanes a piece can feed.  us per SpMM on banded
    // matrices of 62K rows, three formats in turn (so that the view comes
    // from beyond L2), blocks of 3 / 6 / 4 / 2 rows with 64 / 60 / 40 / 40
    // entries a row and 120K rows of 3-row blocks with 24:
    //  O = 8   <1,8,4,8> 8.4 / 9.7 / 7.1 / 7.8 / 8.8;   <1,8,8,4> 9.4 (3 rows)
    //  O = 16  <1,16,4,8> 10.3 / 10.5 / 7.7 / 10.9 / 12.7
    //          <1,16,2,8> 10.4 / 11.5 / 8.2 / 8.8 / 10.4
    //  O = 32  <4,8,4,4> 12.2 / 15.0 / 10.1 / 12.4 / 12.9
    //          <1,32,2,16> 13.1 / 13.2 / 9.3 / 11.9 / 14.7
    //  O = 64  <4,16,4,4> 18.1 / 18.1 / 13.2 / 17.3 / 20.0
    //          <4,16,2,4> 18.9 / 19.7 / 13.6 / 17.4 / 17.8
    //  O = 128 <4,32,2,4> 30.3 / 26.2 / 20.4 / 28.3 / 29.7
    //          <4,32,1,8> 31.5 / 30.1 / 20.8 / 29.6 / 34.2
    const int64_t mean = d.tv_n_entries / d.tv_n_pieces;
    auto go = [&](auto vec, auto lpe, auto s, auto u) {
        return launch_shape<decltype(vec)::value, decltype(lpe)::value, decltype(s)::value, R,
                            decltype(u)::value, true>(d, B, O, ld, C, accumulate, bb, partials, st);
    };
    if (O <= 8) return go(I<1>(), I<8>(), I<4>(), I<8>());
    if (O <= 16)
        return mean > 48 ? go(I<1>(), I<16>(), I<4>(), I<8>()) : go(I<1>(), I<16>(), I<2>(), I<8>());
    if (O <= 32) {
        if constexpr (R >= 4) return go(I<1>(), I<32>(), I<2>(), I<16>());
        else return go(I<4>(), I<8>(), I<4>(), I<4>());
    }
    if (O <= 64)
        return mean > 32 ? go(I<4>(), I<16>(), I<4>(), I<4>()) : go(I<4>(), I<16>(), I<2>(), I<4>());
    if (O <= 128) return go(I<4>(), I<32>(), I<2>(), I<4>());
    return go(I<4>(), I<64>(), I<1>(), I<8>());
}

}  // namespace

hipError_t launch_vcsr_tall(const DeviceFmt& d, const float* B, int32_t O, int32_t ld, float* C,
                            int32_t accumulate, uint64_t b_bytes, float* partials,
                            hipStream_t st) {
    if (d.tv_n_pieces <= 0) return hipSuccess;
    switch (d.tv_R) {
        case 2: return launch_rows<2>(d, B, O, ld, C, accumulate, b_bytes, partials, st);
        case 3: return launch_rows<3>(d, B, O, ld, C, accumulate, b_bytes, partials, st);
        case 4: return launch_rows<4>(d, B, O, ld, C, accumulate, b_bytes, partials, st);
        case 8: return launch_rows<8>(d, B, O, ld, C, accumulate, b_bytes, partials, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace vcsr
