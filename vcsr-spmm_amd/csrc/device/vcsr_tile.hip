// vcsr_tile.hip - tile-stationary SpMM over the VCSR slots (gfx950).
//
// The arithmetic is the VCSR one: every nonzero is a packed slot s of the
// format, contributing val[s] * B[seg_base + lcol[s], :] to its row.  The
// schedule is the one that suits MI355X: a wavefront owns whole C rows and
// writes them once with plain stores (no FP32 atomics, which cost about ten
// plain stores each here), and rows that share columns are processed
// together as a tile, so each B row slice is loaded once per tile and
// applied to up to R rows held in registers.  On block-structured matrices
// (FEM: the rows of a node's block row have the same columns) this divides
// the B-row traffic through the vector memory pipe, the limiting resource of
// a row-stationary SpMM, by the block height.
//
// This file holds the matrix-core kernel of 16-row tiles, the reduce of split
// tiles and the launcher; single-row tiles are in vcsr_tile_row.hip, tiles of
// 2 to 8 rows in vcsr_tile_tall.hip.
//
// The host launcher runs one launch per column slice of at most 256 columns
// (128 when B is over 512 MB) for tiles of up to 8 rows, and for 16-row tiles
// when some are split (their partial rows are one slice wide).
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "../host/tile_view.hpp"
#include "common.hpp"
#include "launch.hpp"
#include "vecops.hpp"

namespace vcsr {

// Compute units of a device (256 on MI355X), read once per device.
int device_cus(int device) {
    static std::atomic<int> cus[64];
    if (device < 0 || device >= 64) return 256;
    int n = cus[device].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
            n <= 0)
            n = 256;
        cus[device].store(n, std::memory_order_relaxed);
    }
    return n;
}

namespace {

// Column slices (launch_vcsr_tile): at most kTileWideCols columns per
// launch, and kTileSliceCols when B is over twice the MALL's 256 MB.
constexpr int32_t kTileWideCols = 256;
constexpr int32_t kTileSliceCols = 128;
constexpr uint64_t kTileSliceBytes = 512ull << 20;

// Adds the piece partials of the rows of split tiles into C.  split: {row,
// first partial row, stride, pieces}, in decreasing piece count.  Lanes
// work in groups of cl lanes (the smallest power of two covering the row's
// column vectors, at most 64): lane c of group g sums column vector c of
// partials g, g + groups, ... .
//  - The first n_heavy rows (the most pieces) take a block of 256 threads
//    each (eight loads in flight for 16-byte vectors, four otherwise: cfg3
//    O = 128 1% faster with eight, O = 8 1% slower), whose groups are added
//    in LDS, so a row split into many pieces costs a few load latencies
//    instead of one per piece.
//  - The other rows take one wave each, four per block, whose groups are
//    added with lane shuffles: no LDS and no block barrier.  Most split rows
//    have a few pieces (power-law 322K matrix: 2,740 rows, most with 2 to 8);
//    as a block each they left most of the block idle behind its barriers.
// Each row's sum has a fixed order (the same bits on every call).
template <int VEC>
__global__ __launch_bounds__(256) void vcsr_tile_reduce(int32_t O, int32_t ld, int32_t accumulate,
                                                        int32_t n_heavy, int32_t n_split,
                                                        const int4* __restrict__ split,
                                                        const float* __restrict__ partials,
                                                        float* __restrict__ C) {
    using V = typename VecT<VEC>::T;
    __shared__ V red[256];
    const int32_t nvec = (O + VEC - 1) / VEC;
    int32_t cl = 1;
    while (cl < nvec && cl < 64) cl <<= 1;
    auto part = [&](const int4& s, int32_t j, int32_t cv) {
        return load_mem(partials + (int64_t)s.y * O + (int64_t)j * ((int64_t)s.z * O) +
                            vec_col<VEC>(cv * VEC, O),
                        V());
    };
    // acc += partials g, g + groups, ... of column vector cv of row s.
    auto sum_group = [&](const int4& s, int32_t g, int32_t groups, int32_t cv, V acc) {
        int32_t j = g;
        if constexpr (VEC == 4) {
            for (; j + 7 * groups < s.w; j += 8 * groups) {
                const V x0 = part(s, j, cv), x1 = part(s, j + groups, cv);
                const V x2 = part(s, j + 2 * groups, cv), x3 = part(s, j + 3 * groups, cv);
                const V x4 = part(s, j + 4 * groups, cv), x5 = part(s, j + 5 * groups, cv);
                const V x6 = part(s, j + 6 * groups, cv), x7 = part(s, j + 7 * groups, cv);
                acc = add_vec(acc, add_vec(add_vec(add_vec(x0, x1), add_vec(x2, x3)),
                                           add_vec(add_vec(x4, x5), add_vec(x6, x7))));
            }
        }
        for (; j + 3 * groups < s.w; j += 4 * groups) {
            const V x0 = part(s, j, cv), x1 = part(s, j + groups, cv);
            const V x2 = part(s, j + 2 * groups, cv), x3 = part(s, j + 3 * groups, cv);
            acc = add_vec(acc, add_vec(add_vec(x0, x1), add_vec(x2, x3)));
        }
        for (; j < s.w; j += groups) acc = add_vec(acc, part(s, j, cv));
        return acc;
    };
    auto store = [&](const int4& s, int32_t cv, const V& x) {
        store_cols<VEC, false>(C + (int64_t)s.x * ld, cv * VEC, O, x, accumulate);
    };
    if ((int32_t)blockIdx.x < n_heavy) {
        const int4 s = split[blockIdx.x];
        const int32_t groups = 256 / cl;
        const int32_t tid = (int32_t)threadIdx.x, c = tid % cl, g = tid / cl;
        for (int32_t c0 = 0; c0 < nvec; c0 += cl) {
            const int32_t cv = c0 + c;
            red[tid] = cv < nvec ? sum_group(s, g, groups, cv, zero_vec(V())) : zero_vec(V());
            __syncthreads();
            for (int32_t h = groups / 2; h >= 1; h >>= 1) {
                if (g < h) red[tid] = add_vec(red[tid], red[tid + h * cl]);
                __syncthreads();
            }
            if (g == 0 && cv < nvec) store(s, cv, red[tid]);
            __syncthreads();
        }
        return;
    }
    // Light rows: wave w of block b takes row n_heavy + 4 (b - n_heavy) + w.
    const int32_t i = n_heavy + ((int32_t)blockIdx.x - n_heavy) * 4 + (int32_t)(threadIdx.x >> 6);
    if (i >= n_split) return;
    const int4 s = split[i];
    const int32_t lane = (int32_t)(threadIdx.x & 63u), groups = 64 / cl;
    const int32_t c = lane % cl, g = lane / cl;
    for (int32_t c0 = 0; c0 < nvec; c0 += cl) {
        const int32_t cv = c0 + c;
        V acc = cv < nvec ? sum_group(s, g, groups, cv, zero_vec(V())) : zero_vec(V());
        for (int32_t h = cl; h < 64; h <<= 1) acc = add_vec(acc, shfl_xor_vec(acc, h));
        if (g == 0 && cv < nvec) store(s, cv, acc);
    }
}

// ---------------------------------------------------------------------------
// 16-row tiles on the matrix cores (view height kTileMmaRows).
//
// v_mfma_f32_16x16x4f32 computes D[i][j] += sum_k A[i][k] * B[k][j] for a
// 16 x 4 A and a 4 x 16 B, with A[i][k] in lane 16k + i, B[k][j] in lane
// 16k + j and D[4q + v][j] in register v of lane 16q + j (checked on the
// device).  Here A is the tile's values for four entries (k) and its 16 rows
// (i), and B the four entries' B-row slices: lane 16k + j holds VEC columns
// c0 + VEC*j .. + VEC-1 of entry k's B row, and MFMA number c takes
// component c, so D_c[i][j] is C[row i][c0 + VEC*j + c].  A group of 16
// entries is four k-steps; the view stores its values in operand order, so
// lane l reads the A operands of all four as one 16-byte load.
//
// Rows of B and C need not be aligned to VEC floats: a lane whose columns
// would reach past O takes the last VEC of the row and stores its own ones
// (vec_col, store_cols), so VEC depends on O and the tiles only (tile_mma_vec).
// Block-sparse 16K matrix, O = 65 / 127 / 333: 51.8 / 83.9 / 229 us with the
// 4-byte lanes an odd O used to take, 39.2 / 41.0 / 102 now; O = 100 and 512
// unchanged.
//
// One wave per (piece, column tile of 16*VEC columns).  The grid runs
// column-tile-major with the XCD-aware block order, so each XCD works on one
// column range of B at a time and its L2 holds that slice of B (the B rows a
// block-sparse matrix touches are spread over all of B).  B and C rows are
// ld floats apart (ld > O for one column slice of a wider product); partial
// rows are O floats.
// ---------------------------------------------------------------------------
typedef float mma_acc4 __attribute__((ext_vector_type(4)));
constexpr int kMmaWaves = 4;
constexpr int kMmaPiece = tile_piece_entries(kTileMmaRows);

template <int VEC>
__device__ __forceinline__ float vec_part(const typename VecT<VEC>::T& b, int c) {
    return reinterpret_cast<const float*>(&b)[c];
}

// Operands of NG entry groups of one wave.
template <int VEC, int NUM>
struct MmaGroups {
    static constexpr int NG = NUM;
    float4 a[NG];
    typename VecT<VEC>::T b[NG][4];
};

// How a wave's loads and MFMAs follow each other, GU entry groups (of 16) per
// block of loads.
enum MmaOrder {
    kMmaMixed,  // as the compiler interleaves them: the fewest registers
    kMmaAhead,  // a block's loads ahead of its MFMAs (a scheduling barrier)
    kMmaTwo     // two sets of operands, one multiplied while the other loads
};
template <int VEC, bool BUF, int GU, MmaOrder ORD>
__global__ __launch_bounds__(256) void vcsr_tile_mma_kernel(
    int32_t n_items, int32_t n_ctiles, int32_t O, int32_t ld, int32_t accumulate, uint32_t b_bytes,
    const int4* __restrict__ chunks, const int4* __restrict__ pieces,
    const int32_t* __restrict__ ent_brow, const uint16_t* __restrict__ ent_mask,
    const float* __restrict__ ent_val, const float* __restrict__ B, float* __restrict__ C,
    float* __restrict__ partials) {
    using V = typename VecT<VEC>::T;
    __shared__ uint32_t s_brow[kMmaWaves][kMmaPiece];

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    const int64_t w = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * kMmaWaves + wave;
    if (w >= (int64_t)n_items * n_ctiles) return;
    const int32_t ct = (int32_t)(w / n_items), item = (int32_t)(w - (int64_t)ct * n_items);
    const int32_t e0 = uniform(chunks[item].x), ne = uniform(chunks[item].y) - e0;  // 16 | ne
    const int32_t pidx = uniform(chunks[item].z);
    const int32_t row0 = uniform(pieces[pidx].x), rows = uniform(pieces[pidx].y);
    const int32_t part = uniform(pieces[pidx].w);
    uint32_t* lb = s_brow[wave];

    // Phase 1: B-row byte offsets (row indices without the buffer path) of
    // the piece's entries; placeholders get "no row".
    const uint32_t row_bytes = (uint32_t)ld * 4u;
    for (int32_t i = lane; i < ne; i += 64) {
        const uint32_t br = (uint32_t)ent_brow[e0 + i];
        const bool any = br != (uint32_t)kTileNoEntry;
        lb[i] = BUF ? (any ? br * row_bytes : kNoRow) : (any ? br : kNoRow);
    }
    wave_sync();

    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), (short)0, (int)b_bytes,
                                          kRawBufferFlags);
    const int kq = lane >> 4, jl = lane & 15;  // MFMA k index, column lane
    const int32_t col = ct * 16 * VEC + VEC * jl;
    const bool kok = col < O;
    const uint32_t koff = (uint32_t)vec_col<VEC>(col, O) * 4u;
    // Entry t's B slice for this lane; zeros for "no row" and columns past O.
    auto load_b = [&](int32_t t) -> V {
        if constexpr (BUF) {
            return load_b_buf<VEC>(rsrc, (lb[t] + koff) | (kok ? 0u : kNoRow));
        } else {
            const uint32_t br = lb[t];
            if (br == kNoRow || !kok) return zero_vec(V());
            return load_mem(B + (int64_t)br * ld + koff / 4, V());
        }
    };
    const float* vp = ent_val + (int64_t)e0 * kTileMmaRows + 4 * lane;

    mma_acc4 d[VEC];
#pragma unroll
    for (int c = 0; c < VEC; ++c) d[c] = mma_acc4{0.f, 0.f, 0.f, 0.f};
    auto load = [&](auto& x, int32_t g0) {
#pragma unroll
        for (int gu = 0; gu < x.NG; ++gu) {
            x.a[gu] = *reinterpret_cast<const float4*>(vp + (int64_t)(g0 + gu) * 256);
#pragma unroll
            for (int s = 0; s < 4; ++s) x.b[gu][s] = load_b(16 * (g0 + gu) + 4 * s + kq);
        }
    };
    auto multiply = [&](const auto& x) {
#pragma unroll
        for (int gu = 0; gu < x.NG; ++gu)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int c = 0; c < VEC; ++c)
                    d[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        reinterpret_cast<const float*>(&x.a[gu])[s], vec_part<VEC>(x.b[gu][s], c),
                        d[c], 0, 0, 0);
    };
    auto block = [&](auto n_c, int32_t g0) {
        MmaGroups<VEC, decltype(n_c)::value> x;
        load(x, g0);
        if constexpr (ORD == kMmaAhead) __builtin_amdgcn_sched_barrier(0);
        multiply(x);
    };
    const int32_t ng = ne / kTileMmaGroup;
    int32_t g0 = 0;
    if constexpr (ORD == kMmaAhead) {
        for (; g0 + GU <= ng; g0 += GU) block(std::integral_constant<int, GU>(), g0);
    } else if constexpr (ORD == kMmaTwo) {
        const int32_t nb = ng / GU;
        if (nb > 0) {
            MmaGroups<VEC, GU> x, y;
            load(x, 0);
            int32_t i = 0;
            for (; i + 3 <= nb; i += 2) {
                load(y, (i + 1) * GU);
                __builtin_amdgcn_sched_barrier(0);
                multiply(x);
                __builtin_amdgcn_sched_barrier(0);
                load(x, (i + 2) * GU);
                __builtin_amdgcn_sched_barrier(0);
                multiply(y);
                __builtin_amdgcn_sched_barrier(0);
            }
            // The last two blocks apart: a load past them, though its result
            // goes unused, is waited for before the wave's stores.
            if (i + 2 == nb) {
                load(y, (i + 1) * GU);
                __builtin_amdgcn_sched_barrier(0);
                multiply(x);
                multiply(y);
            } else {
                multiply(x);
            }
            g0 = nb * GU;
        }
    } else {
        // Many waves per SIMD, all resident from the start: the SIMD issues
        // oldest first, so with equal work the first waves of a SIMD finish
        // long before its last (cfg5 O = 512: 84 us for the first of 8 against
        // 134 us for the last, slots busy 78% of the kernel).  The wave's
        // priority falls with the quarter of its groups done, so lagging
        // waves issue first: 111-127 us, slots busy 92%, the SpMM 5% faster
        // (O = 256 and 512).
        int32_t lvl = 3;
        __builtin_amdgcn_s_setprio(3);
        for (; g0 + GU <= ng; g0 += GU) {
            const int32_t nl = 3 - min(3, (4 * g0) / ng);
            if (nl != lvl) {
                lvl = nl;
                if (lvl == 2) __builtin_amdgcn_s_setprio(2);
                else if (lvl == 1) __builtin_amdgcn_s_setprio(1);
                else __builtin_amdgcn_s_setprio(0);
            }
            block(std::integral_constant<int, GU>(), g0);
        }
        __builtin_amdgcn_s_setprio(0);
    }
    for (; g0 < ng; ++g0) block(std::integral_constant<int, 1>(), g0);

    // This lane holds rows 4*kq + v of the tile, columns col .. col+VEC-1.
    bool fin = true;
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int c = 0; c < VEC; ++c)
            if (4 * kq + v < rows) fin = fin && __builtin_isfinite(d[c][v]);
    if (__any(!(fin || !kok))) {
        // A non-finite sum: recompute this lane's rows in entry order on the
        // VALU, skipping the rows an entry does not have (0 * inf must not
        // reach them), like the reference's per-row loop.
        V acc[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[v] = zero_vec(V());
        for (int32_t t = 0; t < ne; ++t) {
            const uint32_t m = ent_mask[e0 + t];
            const V b = load_b(t);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 4 * kq + v;
                if ((m >> r) & 1u)
                    fma_vec(acc[v], ent_val[tile_val_index(kTileMmaRows, (int64_t)e0 + t, r)], b);
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int c = 0; c < VEC; ++c) d[c][v] = reinterpret_cast<const float*>(&acc[v])[c];
    }
    if (!kok) return;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int r = 4 * kq + v;
        if (r >= rows) continue;
        V x;
#pragma unroll
        for (int c = 0; c < VEC; ++c) reinterpret_cast<float*>(&x)[c] = d[c][v];
        if (part < 0)
            store_cols<VEC, true>(C + (int64_t)(row0 + r) * ld, col, O, x, accumulate);
        else
            store_cols<VEC, false>(partials + (int64_t)(part + r) * O, col, O, x, false);
    }
}

template <int VEC, bool BUF, int GU, MmaOrder ORD>
void launch_mma_as(const DeviceFmt& d, dim3 grid, int32_t n_ct, int32_t O, int32_t ld,
                   int32_t accumulate, uint32_t b_bytes, const float* B, float* C, float* partials,
                   hipStream_t st) {
    hipLaunchKernelGGL((vcsr_tile_mma_kernel<VEC, BUF, GU, ORD>), grid, dim3(64 * kMmaWaves), 0, st,
                       d.tv_n_chunks, n_ct, O, ld, accumulate, b_bytes,
                       reinterpret_cast<const int4*>(d.tv_chunks),
                       reinterpret_cast<const int4*>(d.tv_pieces), d.tv_brow, d.tv_mask, d.tv_val,
                       B, C, partials);
}

template <int VEC, bool BUF>
void launch_mma_buf(const DeviceFmt& d, dim3 grid, int64_t waves, int32_t n_ct, int32_t O,
                    int32_t ld, int32_t accumulate, uint32_t b_bytes, const float* B, float* C,
                    float* partials, hipStream_t st) {
    // Few waves per SIMD: each wave's loads in flight bound the time, so they
    // go ahead of the MFMAs; with many, 8 waves per SIMD with interleaved
    // loads hide the latency better.  us per SpMM on the 16K block-sparse
    // matrix (1,024 tiles; 100 MB read per launch at O = 64), by waves per
    // SIMD:
    //  1 (O = 32 / 64): two sets of 2 groups 17.0 / 22.5, of 1 19.6 / 23.3, of
    //    4 18.8 / 26.2; 4 groups ahead 18.5 / 24.4.
    //  2 / 3 (O = 128 / 192): 2 groups ahead 39.1 / 56.7; two sets of 2 42.4 /
    //    63.0, of 1 40.0 / 59.1.
    //  4 / 8 (O = 256 / 512): 8 groups mixed 68.4 / 122 (4 groups 1-4% slower);
    //    two sets of 1 77 / 156.
    const int64_t simds = 4 * (int64_t)device_cus(d.device);
    if (waves <= simds)
        launch_mma_as<VEC, BUF, 2, kMmaTwo>(d, grid, n_ct, O, ld, accumulate, b_bytes, B, C,
                                            partials, st);
    else if (waves <= 3 * simds)
        launch_mma_as<VEC, BUF, 2, kMmaAhead>(d, grid, n_ct, O, ld, accumulate, b_bytes, B, C,
                                              partials, st);
    else
        launch_mma_as<VEC, BUF, 8, kMmaMixed>(d, grid, n_ct, O, ld, accumulate, b_bytes, B, C,
                                              partials, st);
}

// Columns [0, O) of B and C, whose rows are ld floats apart.
template <int VEC>
hipError_t launch_mma(const Vcsr& v, const DeviceFmt& d, const float* B, int32_t O, int32_t ld,
                      float* C, int32_t accumulate, float* partials, hipStream_t st) {
    const int32_t n_ct = (O + 16 * VEC - 1) / (16 * VEC);
    const int64_t waves = (int64_t)d.tv_n_chunks * n_ct;
    const dim3 grid((unsigned)((waves + kMmaWaves - 1) / kMmaWaves));
    // Bytes from B to the end of its last row.
    const uint64_t b_bytes =
        v.N > 0 ? ((uint64_t)(v.N - 1) * (uint64_t)ld + (uint64_t)O) * 4u : 0u;
    if (b_bytes + 64u * 4u * (uint64_t)VEC >= kBufferLimit)
        launch_mma_buf<VEC, false>(d, grid, waves, n_ct, O, ld, accumulate, 0u, B, C, partials, st);
    else
        launch_mma_buf<VEC, true>(d, grid, waves, n_ct, O, ld, accumulate, (uint32_t)b_bytes, B, C,
                                  partials, st);
    return hipGetLastError();
}

// Columns [0, O) of B and C, whose rows are ld floats apart (B and C point
// at the first column; ld > O for one column slice of wider matrices).
template <int VEC>
hipError_t launch_vec(const Vcsr& v, const DeviceFmt& d, const float* B, int32_t O, int32_t ld,
                      float* C, int32_t accumulate, float* partials, hipStream_t st) {
    if (d.tv_n_chunks > 0) {
        // Bytes from B to the end of its last row.
        const uint64_t b_bytes = v.N > 0 ? ((uint64_t)(v.N - 1) * (uint64_t)ld + (uint64_t)O) * 4u : 0u;
        hipError_t e;
        switch (d.tv_R) {
            case 1:
                e = launch_vcsr_row_tiles(d, B, O, ld, C, accumulate, b_bytes, partials, st);
                break;
            case 2:
            case 3:
            case 4:
            case 8: e = launch_vcsr_tall(d, B, O, ld, C, accumulate, b_bytes, partials, st); break;
            case kTileMmaRows:
                e = launch_mma<VEC>(v, d, B, O, ld, C, accumulate, partials, st);
                break;
            default: return hipErrorInvalidValue;
        }
        if (e != hipSuccess) return e;
    }
    if (d.tv_n_split > 0) {
        // Rows whose pieces one wave covers in at most four loads per lane
        // take a wave each, the others (the split rows come in decreasing
        // piece count, so they are the first n_heavy) a block each; at wide B
        // only where there are many split rows, since with few a block's
        // extra loads in flight win.  Power-law 322K matrix (2,700 split
        // rows), O = 47 58.8 -> 53.7 us against a block per row, O = 128 with
        // a wave per row 5.9 against 5.3 us for the reduce; banded 60K matrix
        // with 70 entries a row, all split, O = 50 / 128 99.6 / 149 -> 60.6 /
        // 115 us.
        const int32_t nvec = (O + VEC - 1) / VEC;
        int32_t cl = 1;
        while (cl < nvec && cl < 64) cl <<= 1;
        const int32_t light_max = cl <= 16 || d.tv_n_split > 16384 ? std::max(4, 4 * (64 / cl)) : 0;
        const auto& pc = d.tv_split_pieces;
        const int32_t n_heavy = (int32_t)(std::partition_point(pc.begin(), pc.end(),
                                                               [&](int32_t x) { return x > light_max; }) -
                                          pc.begin());
        const int64_t blocks = (int64_t)n_heavy + ((int64_t)d.tv_n_split - n_heavy + 3) / 4;
        hipLaunchKernelGGL(vcsr_tile_reduce<VEC>, dim3((unsigned)blocks), dim3(256), 0, st, O, ld,
                           accumulate, n_heavy, d.tv_n_split,
                           reinterpret_cast<const int4*>(d.tv_split), partials, C);
        return hipGetLastError();
    }
    return hipSuccess;
}

}  // namespace

// Floats per lane of a 16-row tile's column tile (16 lanes) for w columns of
// any alignment: the narrowest whose one column tile covers w, else 4.  Idle
// lanes are cheaper than a second column tile, which reads every B row and
// all values again: block-sparse 16K matrix, O = 24 16.7 us as one tile of
// 2 floats per lane against 24.6 as two of 1, O = 50 22.7 as one of 4
// against 30.4 as two of 2.
// Four floats a lane give way to two where the launch then takes less than 3/2
// of its rounds of waves (a wave with two takes two thirds of the time), and two
// to one where all waves still fit one round.  A second time, or with three
// rounds for short pieces of very few tiles, only where a row is no whole number
// of vectors, whose moved-back ends cost more than the values read again.
// us per SpMM, 2 / 4 floats: 380 tiles of 320 entries, O = 144 14.5 / 18.2; 768,
// O = 130 / 200 25.1 / 28.4 and 32.2 / 28.5; 512 of 816, O = 128 30.3 / 22.6;
// 1 / 2 / 4: 128 of 96, O = 47 4.1 / 4.9 / 6.1, O = 257 5.6 / 6.5 / 6.3; 128 of
// 400, O = 257 14.8 / 16.6 / 13.1; 256 of 400, O = 47 7.6 / 9.0 / 12.0, O = 64,
// C += A*B 10.0 / 8.7 / 11.8; 512 of 816, O = 33 24.0 / 17.4 / 22.4.
static int tile_mma_vec(const DeviceFmt& d, int32_t w) {
    const int widest = w > 32 ? 4 : w > 16 ? 2 : 1;
    const int64_t simds = 4 * (int64_t)device_cus(d.device), tiles = d.tv_n_chunks;
    const bool tiny = 8 * tiles <= simds && d.tv_n_entries <= 128 * tiles;
    auto rounds = [&](int vec) {
        return (tiles * ((w + 16 * vec - 1) / (16 * vec)) + simds - 1) / simds;
    };
    int vec = widest;
    while (vec > 1) {
        const bool whole = w % vec == 0;
        const int64_t half = rounds(vec / 2);
        const bool better = vec < widest ? !whole && half == 1 : 2 * half < 3 * rounds(vec);
        if (!better && !(tiny && !whole && half <= 3)) break;
        vec /= 2;
    }
    return vec;
}

// Floats per lane of any tiles for w columns of any alignment (the shapes of
// vcsr_tile_row.hip and vcsr_tile_tall.hip); the reduce of their partial rows
// takes the same.
static int tile_vec(const DeviceFmt& d, int32_t w) {
    if (d.tv_R == kTileMmaRows) return tile_mma_vec(d, w);
    if (d.tv_R == 1) return row_tiles_vec(d, w);
    return w > 32 || (w > 16 && d.tv_R < 4) ? 4 : 1;
}

// Column-slice width of a launch over B and C of width O.  Tiles of 1 to 8
// rows: one launch per column slice of at most 256 columns (one column tile
// of a wave), or 128 when B is over 512 MB, so that the B bytes live at a
// time stay small.
// Measured against one launch over all columns: banded 62K matrix, slices of
// 256, O = 512 / 1024 / 2048: same / 16% / 30% faster; slices of 128,
// uniform-random 1M matrix O = 256 (1 GB): 11% faster, power-law 322K
// matrix O = 512 (659 MB): 3% faster, O = 256 (330 MB): 3% slower.
static int32_t tile_slice_width(const Vcsr& v, const DeviceFmt& d, int32_t O) {
    int32_t width = O;
    if (d.tv_R != kTileMmaRows)
        width = std::min(O, (uint64_t)v.N * (uint64_t)O * 4u > kTileSliceBytes ? kTileSliceCols
                                                                               : kTileWideCols);
    // Split tiles write partial rows one slice wide: whatever the tile
    // height, a launch then covers at most the 256 columns the upload sizes
    // the partial rows for, so no O needs more scratch.
    if (d.tv_partial_rows > 0) width = std::min(width, kTileWideCols);
    return width;
}

int64_t tile_partials_floats(const Vcsr& v, const DeviceFmt& d, int32_t O) {
    if (O <= 0 || v.M == 0 || d.tv_partial_rows == 0) return 0;
    return (int64_t)d.tv_partial_rows * tile_slice_width(v, d, O);
}

int64_t tile_partials_upload_floats(const DeviceFmt& d) {
    return (int64_t)d.tv_partial_rows * kTileWideCols;
}

TilePlan tile_launch_plan(const Vcsr& v, const DeviceFmt& d, int32_t O) {
    TilePlan p;
    if (O <= 0 || v.M == 0) return p;
    p.slice_cols = tile_slice_width(v, d, O);
    p.vec = tile_vec(d, p.slice_cols);
    p.slices = (O + p.slice_cols - 1) / p.slice_cols;
    p.matrix_cores = d.tv_R == kTileMmaRows && d.tv_n_chunks > 0;
    p.reduce_launches = d.tv_n_split > 0 ? p.slices : 0;
    p.partial_floats = tile_partials_floats(v, d, O);
    return p;
}

hipError_t launch_vcsr_tile(const Vcsr& v, const DeviceFmt& d, const float* B, int32_t O,
                            float* C, int32_t accumulate, float* partials, hipStream_t st) {
    if (O <= 0 || v.M == 0) return hipSuccess;
    const int32_t width = tile_slice_width(v, d, O);
    for (int32_t c0 = 0; c0 < O; c0 += width) {
        const int32_t w = std::min(width, O - c0);
        hipError_t e;
        switch (tile_vec(d, w)) {
            case 4: e = launch_vec<4>(v, d, B + c0, w, O, C + c0, accumulate, partials, st); break;
            case 2: e = launch_vec<2>(v, d, B + c0, w, O, C + c0, accumulate, partials, st); break;
            default: e = launch_vec<1>(v, d, B + c0, w, O, C + c0, accumulate, partials, st); break;
        }
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

MfmaWork tile_mfma_work(const DeviceFmt& d, int32_t O) {
    MfmaWork w;
    w.flops_per_op = 2 * 16 * 16 * 4;
    if (d.tv_R != kTileMmaRows || O <= 0) return w;
    const int32_t width = d.tv_partial_rows > 0 ? std::min(O, kTileWideCols) : O;
    for (int32_t c0 = 0; c0 < O; c0 += width) {
        const int32_t n = std::min(width, O - c0), vec = tile_mma_vec(d, n);
        w.ops += d.tv_n_entries / 4 * ((n + 16 * vec - 1) / (16 * vec)) * vec;
    }
    return w;
}

}  // namespace vcsr
