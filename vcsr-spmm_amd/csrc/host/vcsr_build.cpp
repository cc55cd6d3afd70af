// vcsr_build.cpp - VCSR format builders (layouts H, S and TC).
//
// The arrays produced are bit-identical to the reference builders:
//   layout H  : csr_to_vcsr_spmm      include/vcsr.hpp:25-109
//   layout S  : csr_to_vcsr_seg/_opt  src/vcsr_seg.cu:24-113, src/vcsr_opt.cu:23-101
//   layout TC : csr_to_vcsr_tc        src/vcsr_tc.cu:26-106 (segw=16, bundle=16)
// Algorithm (the same steps as the reference, kept alike because the row
// permutation is part of the format):
//   1. every nnz goes to segment sid = col / segw with local column col % segw;
//   2. the entries of one (segment, row) are ordered by local column with
//      std::sort (vcsr.hpp:43-48, vcsr_seg.cu:45-50);
//   3. the rows of a segment are ordered by their entry count, descending,
//      with std::sort.  Layout H sorts all M row ids starting from 0..M-1
//      (vcsr.hpp:56-59); layouts S/TC sort the active rows starting from the
//      iteration order of a std::unordered_map<int,...> filled in ascending
//      row order (vcsr_seg.cu:32,40,57-65);
//   4. the sorted rows are cut into bundles of `bundle` lanes; a bundle's depth
//      is its largest count; layout H skips depth-0 bundles (vcsr.hpp:70);
//   5. group_rows holds the row of each lane: layout H keeps the ids of empty
//      rows and uses -1 only past M (vcsr.hpp:76-80), layouts S/TC use -1 past
//      the active rows (vcsr_seg.cu:83-86);
//   6. slots are packed depth-major, lane-minor; a lane with fewer entries
//      than the depth gets (lcol=-1, val=0) (vcsr.hpp:82-96, vcsr_seg.cu:89-107).
// Because std::sort is not stable, ties are ordered by libstdc++'s introsort;
// reproducing them requires the same std::sort over sequences with the same
// comparison outcomes, and the same unordered_map insertion sequence (its
// iteration order depends only on the keys inserted, their order and the
// rehash policy, not on the mapped type).  That is what is done here, with
// flat arrays instead of per-row vectors.
//
// Work is split by segment: each segment's groups depend only on that
// segment's entries, so segments are built in parallel into per-block
// buffers and concatenated in segment order, giving the sequential result.
#include <algorithm>
#include <cstring>
#include <numeric>
#include <string>
#include <unordered_map>

#include "core.hpp"
#include "parallel.hpp"

namespace vcsr {
namespace {

struct SegEntry {
    int32_t row;
    int32_t lcol;
    float v;
};

// A run of entries of one row inside one segment.
struct Run {
    int32_t row;
    int32_t begin;  // index into the segment's entry list
    int32_t len;
};

// Output of a block of consecutive segments.
struct BlockOut {
    std::vector<int32_t> depth, rows, lcol;
    std::vector<float> val;
    std::vector<int32_t> groups_per_seg;
};

// Buckets all nnz by segment, keeping (row ascending, p ascending) order
// inside a segment, the order in which the reference pushes them.  Blocks of
// rows of about equal nnz count their entries per segment and then write them
// at the offsets that follow from the blocks before them, so the result does
// not depend on the number of blocks.
void bucket_by_segment(const Csr& csr, int segw, int S, int nthreads,
                       std::vector<int64_t>& seg_off, std::vector<SegEntry>& ent) {
    seg_off.assign((size_t)S + 1, 0);
    ent.resize((size_t)csr.nnz);
    int64_t nb = std::min<int64_t>(nthreads, 1 + csr.nnz / 65536);
    while (nb > 1 && nb * (int64_t)S > (int64_t)csr.nnz * 2) nb /= 2;
    std::vector<int32_t> row_of((size_t)nb + 1, csr.M);
    for (int64_t b = 0; b < nb; ++b) {
        const int32_t p = (int32_t)((int64_t)csr.nnz * b / nb);
        row_of[(size_t)b] = (int32_t)(std::lower_bound(csr.row_ptr.begin(), csr.row_ptr.end(), p) -
                                      csr.row_ptr.begin());
    }
    row_of[0] = 0;
    std::vector<std::vector<int64_t>> at((size_t)nb);
    parallel_for(nb, 1, nthreads, [&](int64_t bb, int64_t be) {
        for (int64_t b = bb; b < be; ++b) {
            auto& c = at[(size_t)b];
            c.assign((size_t)S, 0);
            const int32_t p1 = csr.row_ptr[row_of[(size_t)b + 1]];
            for (int32_t p = csr.row_ptr[row_of[(size_t)b]]; p < p1; ++p)
                c[(size_t)(csr.col[p] / segw)]++;
        }
    });
    int64_t off = 0;
    for (int s = 0; s < S; ++s) {
        seg_off[(size_t)s] = off;
        for (auto& c : at) {
            const int64_t n = c[(size_t)s];
            c[(size_t)s] = off;
            off += n;
        }
    }
    seg_off[(size_t)S] = off;
    parallel_for(nb, 1, nthreads, [&](int64_t bb, int64_t be) {
        for (int64_t b = bb; b < be; ++b) {
            auto& cur = at[(size_t)b];
            for (int32_t r = row_of[(size_t)b]; r < row_of[(size_t)b + 1]; ++r) {
                for (int32_t p = csr.row_ptr[r]; p < csr.row_ptr[r + 1]; ++p) {
                    const int32_t c = csr.col[p];
                    const int32_t sid = c / segw;
                    ent[(size_t)cur[(size_t)sid]++] = SegEntry{r, c - sid * segw, csr.val[p]};
                }
            }
        }
    });
}

// Splits a segment's entries into per-row runs and orders each run by local
// column with std::sort (the reference sorts a vector<Entry{lcol,v}> with the
// comparator lcol-less; comparing the same lcol values gives the same order).
void make_runs(SegEntry* e, int32_t n, std::vector<Run>& runs) {
    runs.clear();
    int32_t i = 0;
    while (i < n) {
        int32_t j = i + 1;
        while (j < n && e[j].row == e[i].row) ++j;
        runs.push_back(Run{e[i].row, i, j - i});
        if (j - i > 1)
            std::sort(e + i, e + j,
                      [](const SegEntry& a, const SegEntry& b) { return a.lcol < b.lcol; });
        i = j;
    }
}

// Appends one group (rows of `lane_run`, -1 for missing lanes) to `out`.
// lane_row[l] is the row id of lane l (or -1), lane_run[l] the run index
// holding that row's entries (or -1 for a row with no entries here).
void emit_group(BlockOut& out, int bundle, int depth, const int32_t* lane_row,
                const int32_t* lane_run, const std::vector<Run>& runs, const SegEntry* e) {
    out.depth.push_back(depth);
    for (int l = 0; l < bundle; ++l) out.rows.push_back(lane_row[l]);
    for (int d = 0; d < depth; ++d) {
        for (int l = 0; l < bundle; ++l) {
            const int32_t ri = lane_run[l];
            if (ri >= 0 && d < runs[ri].len) {
                const SegEntry& x = e[runs[ri].begin + d];
                out.lcol.push_back(x.lcol);
                out.val.push_back(x.v);
            } else {
                out.lcol.push_back(-1);
                out.val.push_back(0.f);
            }
        }
    }
}

// Layout S / TC groups of one segment.
void build_segment_S(SegEntry* e, int32_t n, int bundle, BlockOut& out,
                     std::vector<Run>& runs, std::vector<int32_t>& order,
                     std::vector<int32_t>& lane_row, std::vector<int32_t>& lane_run) {
    make_runs(e, n, runs);
    // Same insertion sequence as seg_entries[sid][r] over ascending r.
    std::unordered_map<int32_t, int32_t> m;
    for (int32_t i = 0; i < (int32_t)runs.size(); ++i) m[runs[i].row] = i;
    order.clear();
    for (const auto& kv : m) order.push_back(kv.second);
    // vcsr_seg.cu:63-65: entry count descending.
    std::sort(order.begin(), order.end(),
              [&runs](int32_t a, int32_t b) { return runs[a].len > runs[b].len; });
    const int32_t nact = (int32_t)order.size();
    int32_t ngroups = 0;
    for (int32_t start = 0; start < nact; start += bundle) {
        const int32_t end = std::min(start + bundle, nact);
        int depth = 0;
        for (int32_t i = start; i < end; ++i) depth = std::max(depth, runs[order[i]].len);
        if (depth == 0) continue;
        for (int l = 0; l < bundle; ++l) {
            const int32_t ridx = start + l;
            if (ridx < nact) {
                lane_run[l] = order[ridx];
                lane_row[l] = runs[order[ridx]].row;
            } else {
                lane_run[l] = -1;
                lane_row[l] = -1;
            }
        }
        emit_group(out, bundle, depth, lane_row.data(), lane_run.data(), runs, e);
        ++ngroups;
    }
    out.groups_per_seg.push_back(ngroups);
}

// Per-thread scratch of layout H (arrays of length M).
struct HScratch {
    std::vector<int32_t> cnt, run_of_row, rows;
};

// Layout H groups of one segment.
void build_segment_H(SegEntry* e, int32_t n, int32_t M, int bundle, BlockOut& out,
                     std::vector<Run>& runs, HScratch& hs, std::vector<int32_t>& lane_row,
                     std::vector<int32_t>& lane_run) {
    make_runs(e, n, runs);
    for (int32_t i = 0; i < (int32_t)runs.size(); ++i) {
        hs.cnt[runs[i].row] = runs[i].len;
        hs.run_of_row[runs[i].row] = i;
    }
    // vcsr.hpp:56-59: all rows 0..M-1, entry count descending.
    std::iota(hs.rows.begin(), hs.rows.end(), 0);
    const int32_t* cnt = hs.cnt.data();
    std::sort(hs.rows.begin(), hs.rows.end(),
              [cnt](int32_t a, int32_t b) { return cnt[a] > cnt[b]; });
    int32_t ngroups = 0;
    for (int64_t start = 0; start < M; start += bundle) {
        const int64_t end = std::min<int64_t>(start + bundle, M);
        int depth = 0;
        for (int64_t i = start; i < end; ++i) depth = std::max(depth, cnt[hs.rows[i]]);
        if (depth == 0) continue;
        for (int l = 0; l < bundle; ++l) {
            const int64_t ridx = start + l;
            if (ridx < M) {
                const int32_t row = hs.rows[ridx];
                lane_row[l] = row;
                lane_run[l] = cnt[row] > 0 ? hs.run_of_row[row] : -1;
            } else {
                lane_row[l] = -1;
                lane_run[l] = -1;
            }
        }
        emit_group(out, bundle, depth, lane_row.data(), lane_run.data(), runs, e);
        ++ngroups;
    }
    out.groups_per_seg.push_back(ngroups);
    for (const Run& r : runs) hs.cnt[r.row] = 0;
}

}  // namespace

Vcsr build_vcsr(const Csr& csr, int segw, int bundle, int layout, int nthreads) {
    validate_csr(csr);
    if (layout != kLayoutH && layout != kLayoutS && layout != kLayoutTC)
        throw Error(1, "unknown layout " + std::to_string(layout));
    if (layout == kLayoutTC) {  // src/vcsr_tc.cu:27-28
        segw = 16;
        bundle = 16;
    }
    if (segw <= 0) throw Error(1, "segw must be > 0");
    if (bundle <= 0) throw Error(1, "bundle must be > 0");
    if (nthreads <= 0) nthreads = default_threads();

    Vcsr V;
    V.M = csr.M;
    V.N = csr.N;
    V.segw = segw;
    V.bundle = bundle;
    V.layout = layout;
    const int64_t S64 = ((int64_t)csr.N + segw - 1) / segw;
    if (S64 > INT32_MAX) throw Error(5, "too many segments");
    const int32_t S = (int32_t)S64;
    V.num_segments = S;

    std::vector<int64_t> seg_off;
    std::vector<SegEntry> ent;
    bucket_by_segment(csr, segw, S, nthreads, seg_off, ent);

    // Segments per task: layout H does O(M log M) work per segment.
    // Others: several tasks per thread (2,048 segments a task left a matrix of
    // 20,000 columns to 3 of 16 threads).
    const int64_t grain =
        layout == kLayoutH
            ? 8
            : std::min<int64_t>(2048, std::max<int64_t>(16, S / (8 * (int64_t)nthreads)));
    const int64_t nblocks = (S + grain - 1) / grain;
    std::vector<BlockOut> blocks((size_t)nblocks);
    parallel_for(nblocks, 1, nthreads, [&](int64_t bb, int64_t be) {
        std::vector<Run> runs;
        std::vector<int32_t> order, lane_row(bundle), lane_run(bundle);
        HScratch hs;
        if (layout == kLayoutH) {
            hs.cnt.assign((size_t)csr.M, 0);
            hs.run_of_row.assign((size_t)csr.M, -1);
            hs.rows.resize((size_t)csr.M);
        }
        for (int64_t b = bb; b < be; ++b) {
            BlockOut& out = blocks[(size_t)b];
            const int64_t s0 = b * grain, s1 = std::min<int64_t>(S, s0 + grain);
            for (int64_t sid = s0; sid < s1; ++sid) {
                SegEntry* e = ent.data() + seg_off[sid];
                const int32_t n = (int32_t)(seg_off[sid + 1] - seg_off[sid]);
                if (layout == kLayoutH)
                    build_segment_H(e, n, csr.M, bundle, out, runs, hs, lane_row, lane_run);
                else
                    build_segment_S(e, n, bundle, out, runs, order, lane_row, lane_run);
            }
        }
    });

    // Concatenate in segment order.
    int64_t G = 0, P = 0;
    for (const BlockOut& b : blocks) {
        G += (int64_t)b.depth.size();
        P += (int64_t)b.lcol.size();
    }
    if (P > INT32_MAX) throw Error(5, "packed slot count exceeds int32");
    if (G * (int64_t)bundle > INT32_MAX) throw Error(5, "groups*bundle exceeds int32");
    V.group_ptr.resize((size_t)G + 1);
    V.group_depth.resize((size_t)G);
    V.group_seg_base.resize((size_t)G);
    V.group_rows.resize((size_t)(G * bundle));
    V.lcol.resize((size_t)P);
    V.val.resize((size_t)P);
    V.segment_group_start.resize((size_t)S + 1);
    V.segment_group_start[0] = 0;
    std::vector<int64_t> g0((size_t)nblocks + 1, 0), p0((size_t)nblocks + 1, 0);
    for (int64_t b = 0; b < nblocks; ++b) {
        g0[(size_t)b + 1] = g0[(size_t)b] + (int64_t)blocks[(size_t)b].depth.size();
        p0[(size_t)b + 1] = p0[(size_t)b] + (int64_t)blocks[(size_t)b].lcol.size();
    }
    V.group_ptr[(size_t)G] = (int32_t)P;
    parallel_for(nblocks, 1, nthreads, [&](int64_t bb, int64_t be) {
        for (int64_t b = bb; b < be; ++b) {
            const BlockOut& out = blocks[(size_t)b];
            int64_t gi = 0, slot = p0[(size_t)b];
            const int64_t gb = g0[(size_t)b];
            for (size_t k = 0; k < out.groups_per_seg.size(); ++k) {
                const int32_t sid = (int32_t)(b * grain + (int64_t)k);
                for (int32_t q = 0; q < out.groups_per_seg[k]; ++q, ++gi) {
                    V.group_ptr[(size_t)(gb + gi)] = (int32_t)slot;
                    V.group_depth[(size_t)(gb + gi)] = out.depth[(size_t)gi];
                    V.group_seg_base[(size_t)(gb + gi)] = sid * segw;
                    slot += (int64_t)out.depth[(size_t)gi] * bundle;
                }
                V.segment_group_start[(size_t)sid + 1] = (int32_t)(gb + gi);
            }
            std::copy(out.rows.begin(), out.rows.end(), V.group_rows.begin() + gb * bundle);
            std::copy(out.lcol.begin(), out.lcol.end(), V.lcol.begin() + p0[(size_t)b]);
            std::copy(out.val.begin(), out.val.end(), V.val.begin() + p0[(size_t)b]);
            blocks[(size_t)b] = BlockOut();  // release as we go
        }
    });
    return V;
}

}  // namespace vcsr
