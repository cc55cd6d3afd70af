// csr_wave.hip - wave-per-row CSR SpMM on plain CSR arrays, the ASpT-style
// competitor (src/aspt.cu:38-142): rows are spread over the lanes of a
// wavefront, each row's (column, value) pairs are read once by the lanes and
// shared with the row's other lanes, every lane accumulates its columns of
// C in registers, and C is written once (C = A*B).  No format build.
//
// gfx950 form: a row is a stream of LPE lanes holding VEC consecutive
// columns each, so a wave computes S = 64/LPE rows at once; the reference's
// warp computes one row per 64-column chunk with 4-byte loads and needs
// O % 64 == 0, this kernel takes any O and any alignment.  Every column of C
// is one chain of fused multiply-adds in the row's entry order (the CPU
// loop's bits), so a row's entries cannot be split between lanes.
//  - Rows of up to kLongRow entries: a stream stages CH of its row's entries
//    at a time (B-row byte offset and value) in the wave's LDS (one row a
//    wave: in its lanes' registers), the next ones' loads in flight meanwhile,
//    and applies them in blocks of U loads issued back to back; B is read with
//    raw buffer loads whose range check returns zeros past the row's end.
//    Bound by the waves' chain of loads (row, entries, B rows) where rows are
//    short, by the L2-to-CU path where they are not: as little as possible
//    stands before the first load, and the registers leave 7 or 8 waves per
//    SIMD.
//  - Longer rows bound the kernel by their own latency (8 loads in flight a
//    stream), so the block's four waves take them together afterwards: the
//    waves take turns of LU entries each, all of a turn's B rows loaded ahead
//    while the other waves have their turns, and hand the running sums on
//    through LDS.
// us per SpMM, three matrices in turn, before the long rows' turns, the
// entries' prefetch and the 16-byte lanes at any width, and now: power-law
// 100K rows (longest 1.7K), O = 8 / 47 / 64 136 / 118 / 138 -> 27 / 34 / 34;
// 322K (5.2K), O = 128 539 -> 206; banded 62K, O = 8 / 47 24.8 / 58.4 -> 14.4 /
// 38.5; 16K rows of 9 16x16 blocks, O = 66 67.7 -> 36.0; uniform 1M x 16, O =
// 256 2,737 -> 2,732.
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "vecops.hpp"

namespace vcsr {
namespace {

// Waves per block: 4 (with 8, power-law 100K, O = 64 52 against 37 us).
constexpr int kWaveRowsWaves = 4;
// 64 instead of 128 changes nothing measurable.
constexpr int32_t kLongRow = 128;

// Long rows: columns per lane (64 lanes a row) and entries per turn: 32
// loads of 4 bytes a lane in flight (64: the same times, 16: 10% slower).
template <int VEC, int LPE>
struct LongShape {
    static constexpr int LV = VEC * LPE <= 64 ? 1 : VEC * LPE <= 128 ? 2 : 4;
    static constexpr int LU = 32 / LV;
};

template <int VEC, int LPE, bool BUF>
__global__ __launch_bounds__(64 * kWaveRowsWaves) void csr_wave_kernel(int32_t M, int32_t N, int32_t O,
                                                       uint32_t b_bytes,
                                                       const int32_t* __restrict__ rowptr,
                                                       const int32_t* __restrict__ col,
                                                       const float* __restrict__ val,
                                                       const float* __restrict__ B,
                                                       float* __restrict__ C) {
    using V = typename VecT<VEC>::T;
    constexpr int S = 64 / LPE;                   // rows per wave
    constexpr int NR = kWaveRowsWaves * S;        // ... and block
    constexpr int U = 8;                          // loads per block
    constexpr int NC = LPE >= 32 ? 1 : 32 / LPE;  // entries a lane stages at a time
    constexpr int CH = LPE * NC;                  // ... and a stream
    constexpr int LS = CH + 4;                    // keeps the streams' reads in different banks
    __shared__ __align__(16) uint32_t s_off[kWaveRowsWaves][S * LS];
    __shared__ __align__(16) float s_val[kWaveRowsWaves][S * LS];
    __shared__ __align__(16) float s_sum[64 * 4];

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63), sub = lane / LPE, kl = lane % LPE;
    const int64_t row0 = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * NR;
    // The block's rows, one a lane, read by every wave for itself beside its
    // own: a block without long rows has no barrier.  Rows past M repeat the
    // last one.
    const int32_t rows = (int32_t)min((int64_t)NR, M - row0), slot = wave * S + sub;
    const bool rowok = slot < rows;
    const int32_t* ra = rowptr + row0 + min(slot, rows - 1);
    const int32_t* rb = rowptr + row0 + min(lane & (NR - 1), rows - 1);
    const int32_t p0 = ra[0], p1 = ra[1], bp = rb[0], bn = rb[1] - bp;
    const uint64_t longs = __ballot(bn > kLongRow) & ((2ull << (rows - 1)) - 1ull);
    // The block takes its long rows together only if few rows stand out:
    // otherwise the rows' streams, side by side, are the faster way (16x16
    // blocks, 51 a row, O = 100 all together 708 us, side by side 222).
    bool together = false;
    if (longs != 0) {
        constexpr int FEW = S >= 4 ? 4 : 2;
        int32_t most = lane < rows ? bn : 0, sum = min(most, 1 << 24);
#pragma unroll
        for (int sh = 1; sh < 64; sh <<= 1) {
            most = max(most, __shfl_xor(most, sh));
            sum += __shfl_xor(sum, sh);
        }
        together = uniform(sum) / FEW <= uniform(most);
    }
    // One row a wave: the block's waves start their rows together, so that
    // neighbouring rows find each other's B rows in the L1 (banded 120K
    // matrix with 24 entries a row, O = 256 153.4 -> 149.3 us).
    if constexpr (LPE == 64) __syncthreads();
    const int32_t limit = together ? kLongRow : INT32_MAX;
    const bool mine = rowok && p1 - p0 <= limit;  // this stream's row, unless the block takes it
    const int32_t n = mine ? p1 - p0 : 0;
    int32_t nmax = 0;
#pragma unroll
    for (int i = 0; i < S; ++i) {
        const int32_t x = __builtin_amdgcn_readlane(bn, wave * S + i);
        nmax = max(nmax, x <= limit ? x : 0);
    }
    uint32_t* lo = s_off[wave] + sub * LS;
    float* lv = s_val[wave] + sub * LS;
    const uint32_t row_bytes = (uint32_t)O * 4u;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), (short)0, (int)b_bytes,
                                          kRawBufferFlags);
    // B-row offset (index off the buffer path) of column cj; a column outside
    // [0, N) reads nothing.
    auto b_off = [&](int32_t cj) -> uint32_t {
        return (uint32_t)cj < (uint32_t)N ? (BUF ? (uint32_t)cj * row_bytes : (uint32_t)cj) : kNoRow;
    };

    // Narrower shapes hold all columns at once: no loop, whose invariants
    // (addresses) would be kept in registers.
    const int32_t kend = LPE == 64 ? O : LPE * VEC;
    for (int32_t k0 = 0; k0 < kend; k0 += LPE * VEC) {
        const int32_t k = k0 + kl * VEC;
        const bool kok = k < O;
        const int32_t kc = vec_col<VEC>(k, O);
        // Lanes past O read their row's last vector once more.  Masking them
        // with offsets past the end of B costs twice the time of the loads
        // (banded 62K matrix, O = 1 / 7 / 9: 19.8 / 22.2 / 34.0 us so masked,
        // 10.8 / 13.0 / 15.1 now).
        auto load_b = [&](uint32_t off, int32_t c) -> V {
            if constexpr (BUF) return load_b_buf<VEC>(rsrc, off + (uint32_t)c * 4u);
            else return off != kNoRow ? load_mem(B + (int64_t)off * O + c, V()) : zero_vec(V());
        };
        V acc = zero_vec(V());
        int32_t cj[NC];
        float a[NC];
        auto fetch = [&](int32_t c0) {
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                if (q > 0 && c0 + q * LPE >= nmax) break;
                const int32_t i = c0 + q * LPE + kl;
                cj[q] = i < n ? col[p0 + i] : -1;
                a[q] = i < n ? val[p0 + i] : 0.f;
            }
        };
        fetch(0);
        if constexpr (LPE == 64) {
            // One row a wave: the entries stay in its lanes' registers.
            for (int32_t c0 = 0; c0 < nmax; c0 += CH) {
                const uint32_t off = b_off(cj[0]);
                const float av = off == kNoRow ? 0.f : a[0];
                if (c0 + CH < nmax) fetch(c0 + CH);
                const int32_t cnt = min(CH, nmax - c0);
                for (int32_t j0 = 0; j0 < cnt; j0 += U) {
                    uint32_t o[U];
                    float x[U];
                    V b[U];
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        o[u] = (uint32_t)__builtin_amdgcn_readlane((int)off, j0 + u);
#pragma unroll
                    for (int u = 0; u < U; ++u) b[u] = load_b(o[u], kc);
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        x[u] = __builtin_bit_cast(
                            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, av), j0 + u));
#pragma unroll
                    for (int u = 0; u < U; ++u) fma_vec(acc, x[u], b[u]);
                }
            }
        } else {
            for (int32_t c0 = 0; c0 < nmax; c0 += CH) {
#pragma unroll
                for (int q = 0; q < NC; ++q) {
                    if (q > 0 && c0 + q * LPE >= nmax) break;
                    const uint32_t off = b_off(cj[q]);
                    lo[q * LPE + kl] = off;
                    lv[q * LPE + kl] = off == kNoRow ? 0.f : a[q];
                }
                if (c0 + CH < nmax) fetch(c0 + CH);
                wave_sync();
                const int32_t cnt = min(CH, nmax - c0);
                for (int32_t j0 = 0; j0 < cnt; j0 += U) {  // CH is a multiple of U
                    uint32_t o[U];
                    float x[U];
                    V b[U];
#pragma unroll
                    for (int u = 0; u < U; u += 4)
                        *reinterpret_cast<uint4*>(o + u) = *reinterpret_cast<const uint4*>(lo + j0 + u);
#pragma unroll
                    for (int u = 0; u < U; ++u) b[u] = load_b(o[u], kc);
#pragma unroll
                    for (int u = 0; u < U; u += 4)
                        *reinterpret_cast<float4*>(x + u) = *reinterpret_cast<const float4*>(lv + j0 + u);
#pragma unroll
                    for (int u = 0; u < U; ++u) fma_vec(acc, x[u], b[u]);
                }
                wave_sync();
            }
        }
        if (mine && kok)
            store_cols<VEC, false>(C + (row0 + wave * S) * O + sub * O, k, O, acc, false);
    }

    // Long rows.
    if (!together) return;
    constexpr int LV = LongShape<VEC, LPE>::LV, LU = LongShape<VEC, LPE>::LU;
    using W = typename VecT<LV>::T;
    for (uint64_t left = longs; left != 0; left &= left - 1) {
        const int slot = __builtin_ctzll(left);  // of the block's rows
        const int32_t nl = __builtin_amdgcn_readlane(bn, slot);
        const int32_t pl = __builtin_amdgcn_readlane(bp, slot), turns = (nl + LU - 1) / LU;
        for (int32_t k0 = 0; k0 < O; k0 += 64 * LV) {
            const int32_t k = k0 + lane * LV;
            const bool kok = k < O;
            const int32_t kc = vec_col<LV>(k, O);  // O >= LV
            // This wave's turn (B rows in b, values in lanes' av) and the
            // entries of the one after it.
            // (Loads at clamped indices: a branch around them makes the
            // compiler wait for them before the barrier.)
            W b[LU];
            float av, vnext;
            int32_t cnext;
            auto fetch_entries = [&](int32_t t) {
                const int32_t i = pl + min(t * LU + (lane % LU), nl - 1);
                cnext = col[i];
                vnext = val[i];
            };
            auto fetch_rows = [&](int32_t t) {
                const uint32_t off = t * LU + (lane % LU) < nl ? b_off(cnext) : kNoRow;
                av = off == kNoRow ? 0.f : vnext;
#pragma unroll
                for (int u = 0; u < LU; ++u) {
                    const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)off, u);
                    if constexpr (BUF) {
                        b[u] = load_b_buf<LV>(rsrc, o + (uint32_t)kc * 4u);
                    } else {
                        b[u] = o != kNoRow ? load_mem(B + (int64_t)o * O + kc, W()) : zero_vec(W());
                    }
                }
                fetch_entries(t + kWaveRowsWaves);
            };
            fetch_entries(wave);
            fetch_rows(wave);
            // Every wave meets `turns` barriers, one at the end of each turn.
            int32_t met = 0;
            for (int32_t t = wave; t < turns; t += kWaveRowsWaves) {
                for (; met < t; ++met) __syncthreads();
                W acc = zero_vec(W());
                if (t > 0) acc = *reinterpret_cast<const W*>(s_sum + lane * LV);
#pragma unroll
                for (int u = 0; u < LU; ++u)
                    fma_vec(acc, __builtin_bit_cast(float, __builtin_amdgcn_readlane(
                                                               __builtin_bit_cast(int, av), u)),
                            b[u]);
                if (t + 1 < turns) {
                    *reinterpret_cast<W*>(s_sum + lane * LV) = acc;
                } else if (kok) {
                    store_cols<LV, false>(C + (row0 + slot) * O, k, O, acc, false);
                }
                __syncthreads();
                ++met;
                fetch_rows(t + kWaveRowsWaves);
            }
            for (; met < turns; ++met) __syncthreads();
        }
    }
}

template <int VEC, int LPE>
hipError_t launch_lpe(int32_t M, const int32_t* rowptr, const int32_t* col, const float* val,
                      const float* B, int32_t N, int32_t O, float* C, hipStream_t st) {
    constexpr int rows = 64 / LPE * kWaveRowsWaves;
    const dim3 grid((unsigned)(((int64_t)M + rows - 1) / rows)), block(64 * kWaveRowsWaves);
    const uint64_t b_bytes = (uint64_t)N * (uint64_t)O * 4u;
    if (b_bytes >= kBufferLimit)
        hipLaunchKernelGGL((csr_wave_kernel<VEC, LPE, false>), grid, block, 0, st, M, N, O, 0u,
                           rowptr, col, val, B, C);
    else
        hipLaunchKernelGGL((csr_wave_kernel<VEC, LPE, true>), grid, block, 0, st, M, N, O,
                           (uint32_t)b_bytes, rowptr, col, val, B, C);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_csr_wave(int32_t M, const int32_t* rowptr, const int32_t* col, const float* val,
                           const float* B, int32_t N, int32_t O, float* C, hipStream_t st) {
    if (M <= 0 || O <= 0) return hipSuccess;
    if (O <= 8) return launch_lpe<1, 8>(M, rowptr, col, val, B, N, O, C, st);
    if (O <= 16) return launch_lpe<1, 16>(M, rowptr, col, val, B, N, O, C, st);
    if (O <= 32) return launch_lpe<4, 8>(M, rowptr, col, val, B, N, O, C, st);
    if (O <= 64) return launch_lpe<4, 16>(M, rowptr, col, val, B, N, O, C, st);
    if (O <= 128) return launch_lpe<4, 32>(M, rowptr, col, val, B, N, O, C, st);
    return launch_lpe<4, 64>(M, rowptr, col, val, B, N, O, C, st);
}

}  // namespace vcsr
