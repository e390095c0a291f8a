// hashgrid.hip — multiresolution hash encoding, forward and table gradient.
//
// Forward restates models/encoders.py:82-233 (HashGridEncoder.__call__): the
// reference evaluates it as XLA gather + lerp fusions and materialises [L,N,8]
// index and weight arrays; here each thread computes one (point, level) pair in
// registers: normalise, scale, floor, 8 vertex indices (dense x + y res + z res^2
// below first_hash_level, else x ^ y*2654435761 ^ z*805459861, both mod T, plus the
// level's row offset), trilinear weights, weighted sum of the gathered rows.
// Workgroups are level-affine per XCD (see level_block), so a level's gathers hit one
// L2, whichever layout the output has.
//
// Backward is the VJP of the gather (encoders.py:226) and of the weighted sum
// (encoders.py:231): dtable[idx] += w * g, computed by a counting sort of the
// contributions into row slices that are summed in LDS (no global atomics).
//
// Arithmetic: f32, no contraction (matches the CPU oracle bit for bit on indices
// and weights).  Indices past the last row (only possible when the last level is
// dense) are clamped to the last row, as JAX clamps gather indices.
#include <hip/hip_fp16.h>

#include "ngp_common.h"
#include "hashgrid_device.h"

namespace ngp {
namespace {

constexpr int kBlock = 256;

// Workgroups are dispatched round-robin over the 8 XCDs of the chip (block b runs
// on XCD b % 8), each with its own 4 MiB L2.  An XCD therefore works on one level at a
// time, so that level's rows (at most T * F * 4 B = 4 MiB for T = 2^19, F = 2) stay in
// its L2 for the gathers, instead of every L2 streaming the whole 46.5 MiB table.
// Levels cost differently (2^18 ray samples, one level on every XCD: 16 us for a dense
// or coarse one, whose cells a ray's samples share, 54 us for the finest, f32), so two
// whole levels per XCD left the ones with the finest levels working alone (71 us
// against a mean of 57).  Four pairs of XCDs instead deal the levels in snake order
// from the finest down, each XCD of a pair taking every second group of points: the
// sums of the four sets are within 6% of the mean for ray samples, and random points,
// where all hashed levels cost alike, get 2 or 3 of the 11 per pair.  Fewer levels leave
// some of four sets with nothing or with one level more than the rest, so they are dealt to
// two sets of four XCDs, or one after the other to all eight (level_sets).
constexpr uint32_t kXcds = 8;
constexpr uint64_t kL2Bytes = 4u << 20;
constexpr int kLmPointsPerThread = 2;
constexpr int kPointsPerBlock = kBlock * kLmPointsPerThread;

// 2^18 ray samples, f32, level-major, with 1, 2 and 4 sets: 3 levels 10.5, 9.9 and 16.1 us;
// 5 levels of up to 2^19 rows 20.6, 22.1 and 27.8; 8 levels 23.9, 23.0 and 27.6; 12 levels
// 41.8, 38.8 and 41.0 (32,768 of them 10.8, 9.7 and 8.6); 16 levels 63.0, 58.9 and 56.7.
__host__ __device__ inline uint32_t level_sets(uint32_t L) { return L >= 12 ? 4u : L >= 6 ? 2u : 1u; }

// Point groups (of kPointsPerBlock points) of one XCD and level.
__host__ __device__ inline uint32_t xcd_groups(uint32_t n_points, uint32_t sets) {
    const uint64_t n_pg = ((uint64_t)n_points + kPointsPerBlock - 1) / kPointsPerBlock;
    return (uint32_t)((n_pg * sets + kXcds - 1) / kXcds);
}

struct LevelBlock {
    uint32_t level, point0;
    bool live;
};

__device__ __forceinline__ LevelBlock level_block(uint32_t n_points, uint32_t L) {
    const uint32_t sets = level_sets(L), n_groups = xcd_groups(n_points, sets);
    const uint32_t b = blockIdx.x;
    const uint32_t x = b % kXcds, rest = b / kXcds;
    const uint32_t i = rest % n_groups, phase = rest / n_groups;
    const uint32_t s = x % sets;
    const uint32_t k = phase * sets + ((phase & 1u) ? sets - 1u - s : s);
    const uint64_t point0 = (uint64_t)(kXcds / sets * i + x / sets) * kPointsPerBlock;
    LevelBlock lb;
    lb.level = L - 1u - k;
    lb.point0 = (uint32_t)point0;
    lb.live = k < L && point0 < n_points;
    return lb;
}

inline uint32_t level_grid(uint32_t n_points, uint32_t L) {
    const uint32_t sets = level_sets(L);
    return kXcds * xcd_groups(n_points, sets) * div_up(L, sets);
}

// Forward: each thread takes kLmPointsPerThread points of the block's level, kBlock
// apart, so the gathers of both are in flight together; points past the end load the
// last point and store nothing.  Level-major output is one contiguous run per
// wavefront; point-major output is 8 bytes per point, 128 apart, which costs less than
// giving up the level's residency in L2 did (a wavefront of 4 points x 16 levels).
// kGroups: see GroupedGather.  Measured, 2^18 ray samples: f32 level-major 92 -> 55 us
// (68 with the levels two to an XCD), point-major 109 -> 93; f16 82 -> 46 and 97 -> 76.
template <int F, typename TT, bool kGroups>
__global__ void __launch_bounds__(kBlock)
    hashgrid_fwd_kernel(HashGridDescriptor d, const float *__restrict__ pos, const TT *__restrict__ table,
                           float *__restrict__ enc) {
    constexpr int P = kLmPointsPerThread;
    const LevelBlock lb = level_block(d.n_points, d.L);
    if (!lb.live) return;
    const uint32_t l = lb.level;
    const bool level_major = d.enc_layout == NGP_ENC_LEVEL_MAJOR;
    const size_t point_stride = level_major ? F : (size_t)d.L * F;
    float *const level_out = enc + (size_t)l * (level_major ? (size_t)d.n_points * F : F);
    float at[P][3], q[P][3];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const uint32_t n = lb.point0 + j * kBlock + threadIdx.x;
        const uint32_t np = n < d.n_points ? n : d.n_points - 1;
#pragma unroll
        for (int a = 0; a < 3; ++a) at[j][a] = pos[3 * (size_t)np + a];
    }
    const Divisor two_b = make_divisor(2.0f * d.bound);
#pragma unroll
    for (int j = 0; j < P; ++j) normalise(two_b, d.bound, at[j], q[j]);
    with_rule(l < d.first_hash_level, (d.T & (d.T - 1u)) == 0, [&](auto rule, auto pow2) {
        uint32_t idx[P][8];
        float w[P][8];
#pragma unroll
        for (int j = 0; j < P; ++j)
            level_vertices_t<decltype(rule)::value, decltype(pow2)::value>(
                q[j][0], q[j][1], q[j][2], d.scales[l], d.resolutions[l], l < d.first_hash_level, d.T, d.offsets[l],
                d.n_rows - 1u, idx[j], w[j]);
        if constexpr (kGroups) {
            static_assert(F == 2, "grouped rows hold two features");
            GroupedGather<TT> gg[P];
#pragma unroll
            for (int j = 0; j < P; ++j) gg[j].load(table_buffer(d, table), idx[j]);
#pragma unroll
            for (int j = 0; j < P; ++j) {
                const float2 v = gg[j].sum(idx[j], w[j]);
                const uint32_t n = lb.point0 + j * kBlock + threadIdx.x;
                if (n < d.n_points) *reinterpret_cast<float2 *>(level_out + n * point_stride) = v;
            }
        } else {
#pragma unroll
            for (int j = 0; j < P; ++j) {
                float acc[F];
#pragma unroll
                for (int f = 0; f < F; ++f) acc[f] = 0.0f;
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    const TT *row = table + (size_t)idx[j][c] * F;
#pragma unroll
                    for (int f = 0; f < F; ++f) acc[f] = acc[f] + to_f32<TT>(row[f]) * w[j][c];
                }
                const uint32_t n = lb.point0 + j * kBlock + threadIdx.x;
                if (n < d.n_points) {
                    float *out = level_out + n * point_stride;
#pragma unroll
                    for (int f = 0; f < F; ++f) out[f] = acc[f];
                }
            }
        }
    });
}

// Point-major forward with the levels of a point in neighbouring lanes: its row is written
// in whole lines, and no level stays in an L2.  For levels so large that they would not.
// 2^18 ray samples, f32, against the kernel above: T = 2^22, F = 2 123 and 181 us, T = 2^19,
// F = 8 168 and 254 (2^14: 15 and 19); a level of two L2s, T = 2^20, F = 2: 111 and 113, and at
// random 289 and 182.
template <int F, typename TT>
__global__ void __launch_bounds__(kBlock)
    hashgrid_fwd_points_kernel(HashGridDescriptor d, const float *__restrict__ pos, const TT *__restrict__ table,
                               float *__restrict__ enc) {
    __shared__ LevelTables lt;
    if (threadIdx.x < d.L) {
        lt.scale[threadIdx.x] = d.scales[threadIdx.x];
        lt.res[threadIdx.x] = d.resolutions[threadIdx.x];
        lt.offset[threadIdx.x] = d.offsets[threadIdx.x];
    }
    __syncthreads();
    const uint64_t t = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (t >= (uint64_t)d.n_points * d.L) return;
    const uint32_t n = (uint32_t)(t / d.L), l = (uint32_t)(t % d.L);
    float p[3];
    normalise(make_divisor(2.0f * d.bound), d.bound, pos + 3 * (size_t)n, p);
    uint32_t idx[8];
    float w[8], acc[F];
    level_vertices(p[0], p[1], p[2], lt.scale[l], lt.res[l], l < d.first_hash_level, d.T, (d.T & (d.T - 1u)) == 0,
                   lt.offset[l], d.n_rows - 1u, idx, w);
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const TT *row = table + (size_t)idx[c] * F;
#pragma unroll
        for (int f = 0; f < F; ++f) acc[f] = acc[f] + to_f32<TT>(row[f]) * w[c];
    }
#pragma unroll
    for (int f = 0; f < F; ++f) enc[t * F + f] = acc[f];
}

// [L, n, F] encodings -> [n, L * F], Vec one point's F features: a workgroup takes
// kTransposePoints points, reads each level's run (512 bytes for F = 2) and writes the
// points' rows, both coalesced, through LDS.
constexpr int kTransposePoints = 64;
template <typename Vec>
__global__ void __launch_bounds__(kBlock)
    encodings_to_points_kernel(uint32_t n_points, uint32_t L, const Vec *__restrict__ lm, Vec *__restrict__ pm) {
    __shared__ Vec tile[kTransposePoints * (NGP_HASHGRID_MAX_LEVELS + 1)];
    const uint32_t p0 = blockIdx.x * kTransposePoints;
    const uint32_t n = min((uint32_t)kTransposePoints, n_points - p0), row = L + 1;
    for (uint32_t t = threadIdx.x; t < L * kTransposePoints; t += kBlock) {
        const uint32_t l = t / kTransposePoints, i = t % kTransposePoints;
        if (i < n) tile[i * row + l] = lm[(size_t)l * n_points + p0 + i];
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < n * L; t += kBlock) pm[(size_t)p0 * L + t] = tile[t / L * row + t % L];
}

// [n, L * F] gradients -> [L, n, F], for F = 2: the same the other way.  The level's bucket
// kernel then reads whole lines; point-major it takes 8 bytes of each of 64 lines, and
// every level reads the lines again (2^18 ray samples f32: bucket 97 -> 68 us for 15 here).
__global__ void __launch_bounds__(kBlock)
    gradients_to_levels_kernel(uint32_t n_points, uint32_t L, const float2 *__restrict__ pm, float2 *__restrict__ lm) {
    __shared__ float2 tile[kTransposePoints * (NGP_HASHGRID_MAX_LEVELS + 1)];
    const uint32_t p0 = blockIdx.x * kTransposePoints;
    const uint32_t n = min((uint32_t)kTransposePoints, n_points - p0), row = L + 1;
    for (uint32_t t = threadIdx.x; t < n * L; t += kBlock) tile[t / L * row + t % L] = pm[(size_t)p0 * L + t];
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < L * kTransposePoints; t += kBlock) {
        const uint32_t l = t / kTransposePoints, i = t % kTransposePoints;
        if (i < n) lm[(size_t)l * n_points + p0 + i] = tile[i * row + l];
    }
}

// Backward without global atomics.  Device-scope atomics on this chip (float or
// integer, any scope) retire at ~21-27 G/s for the whole device on scattered
// addresses, two orders of magnitude below the gather rate, so contributions are
// routed to LDS by a deterministic counting sort over row slices of R rows
// (R rows of F floats fill 128 KiB of LDS):
//   1. count:   work item = (level, 2048-point chunk); LDS histogram of the item's
//               contributions per slice, stored slice-major;
//   2. scan:    exclusive scan of the counts -> each item's write offset per slice
//               (per-block sums, then each block adds the sums before its own);
//   3. scatter: the item recomputes its contributions (with dL_dencodings) and
//               writes (row within slice, values) entries at its offsets;
//   4. reduce:  workgroup s sums slice s's contiguous entries with LDS atomics and
//               stores its rows once (so no table zero-fill either).
// Within an item, lanes are 64 consecutive samples of one level; runs of equal rows
// (coarse levels: consecutive samples of a ray share cells) are summed with a
// segmented scan first, so one entry carries a run.
constexpr int kChunk = 2048;         // points per work item
constexpr int kItemThreads = 256;    // 8 points per thread per item
constexpr int kReduceThreads = 1024;
constexpr uint32_t kPart = 65536;    // entries one reduce workgroup sums
constexpr uint32_t kMinPart = 8192;  // of the one-pass form, at least
constexpr uint32_t kFullParts = 768;  // of one batch, at most, while kPart is enough
constexpr uint32_t kMaxSlices = 8192;
constexpr uint32_t kSliceBytes = 131072;
constexpr uint32_t kRunSliceBytes = 65536;  // one-pass form: two reduce workgroups per CU
constexpr int kRunThreads = 512;
constexpr int kScanThreads = 1024;
constexpr int kScanPer = 4;  // elements per thread in the scan kernels

// An entry is (row within slice, F values), padded to a power of two of words so
// that it is written and read with one or two vector accesses.
// Words of one sort entry: the row in its slice, then the F values, as f32 (F = 2:
// 12 bytes, one dwordx3 access) or, for f16 tables with F = 2 or 4, as f16 pairs
// (F = 2: 8 bytes) — the precision path accumulates its table gradient from
// f16-rounded contributions, as half-precision grids are trained in tiny-cuda-nn.
template <int F, bool kHalf>
constexpr int entry_words() {
    return kHalf && F == 2 ? 2 : (kHalf && F == 4 ? 3 : (F == 1 ? 2 : (F == 2 ? 3 : (F == 4 ? 8 : 16))));
}

inline int entry_words_host(uint32_t F, bool half) {
    return half && F == 2 ? 2 : (half && F == 4 ? 3 : (F == 1 ? 2 : (F == 2 ? 3 : (F == 4 ? 8 : 16))));
}

template <int F, bool kHalf>
__device__ __forceinline__ void pack_values(uint32_t *w, const float *v) {
    if constexpr (kHalf && (F == 2 || F == 4)) {
#pragma unroll
        for (int q = 0; q < F / 2; ++q) {
            const __half2 h = __floats2half2_rn(v[2 * q], v[2 * q + 1]);
            w[1 + q] = *reinterpret_cast<const uint32_t *>(&h);
        }
    } else {
#pragma unroll
        for (int f = 0; f < F; ++f) w[1 + f] = __float_as_uint(v[f]);
    }
}

template <int F, bool kHalf>
__device__ __forceinline__ float entry_value(const uint32_t *w, int f) {
    if constexpr (kHalf && (F == 2 || F == 4)) {
        const uint32_t u = w[1 + f / 2];
        const __half2 h = *reinterpret_cast<const __half2 *>(&u);
        return (f & 1) ? __high2float(h) : __low2float(h);
    } else {
        return __uint_as_float(w[1 + f]);
    }
}

// The last row level l's vertices can address: rows are taken modulo T, so a point outside
// the box reaches any of the T rows from the level's offset on, past a dense level's own, as
// the reference's indices do.  Clamped to the table.
inline uint32_t level_last_row(const HashGridDescriptor &d, uint32_t l) {
    return (uint32_t)std::min<uint64_t>((uint64_t)d.offsets[l] + d.T - 1u, (uint64_t)d.n_rows - 1u);
}

// The last one that points of the box address.  A dense level's vertex coordinates reach
// res (a point on the upper face), so its rows run up to res + res^2 + res^3 past the
// level's offset, into the next level's.
inline uint32_t level_last_box_row(const HashGridDescriptor &d, uint32_t l) {
    const uint64_t res = d.resolutions[l];
    const uint64_t local = l < d.first_hash_level ? res + res * res + res * res * res : ~0ull >> 1;
    return (uint32_t)std::min<uint64_t>(d.offsets[l] + local, level_last_row(d, l));
}

// The one-pass table gradient (F <= 2, every level's rows of the box within kStageSlices
// slices): work item = (level, bucket_points consecutive points).  Its entries are kept
// in two arrays, the F values (f32, or one half2 for an f16 table with F = 2) and the
// 16-bit row within the slice: 10 or 6 bytes instead of 12 or 8.
constexpr int kBucketThreads = 512;
// f32 entries: items of 1024 points (two per thread) leave the reducer half as many runs
// (3 us of it at 2^18 points); the smaller f16 entries gain more from the lighter kernel of
// one point per thread (10 us of the bucket kernel).
constexpr int bucket_phases(bool half_values) { return half_values ? 1 : 2; }
constexpr uint32_t bucket_points(bool half_values) { return kBucketThreads * bucket_phases(half_values); }
constexpr uint32_t bucket_entries(bool half_values) { return bucket_points(half_values) * 8; }  // one item's at most
constexpr uint32_t kStageSlices = 1024;                 // slices one level may span inside the box

constexpr uint32_t kStageEntries = 4096;                // entries staged in LDS at a time

template <int F, bool kHalf>
struct EntryValue {
    uint32_t w[kHalf && F == 2 ? 1 : F];
    __device__ __forceinline__ void pack(const float *v) {
        if constexpr (kHalf && F == 2) {
            w[0] = __builtin_bit_cast(uint32_t, __floats2half2_rn(v[0], v[1]));
        } else {
#pragma unroll
            for (int f = 0; f < F; ++f) w[f] = __float_as_uint(v[f]);
        }
    }
    __device__ __forceinline__ float get(int f) const {
        if constexpr (kHalf && F == 2) {
            const __half2 h = __builtin_bit_cast(__half2, w[0]);
            return f ? __high2float(h) : __low2float(h);
        } else {
            return __uint_as_float(w[f]);
        }
    }
};

inline uint32_t value_bytes(uint32_t F, bool half) { return half && F == 2 ? 4 : 4 * F; }

// points (both ways: 77,777 72 and 74 us, 150,000 120 and 105; f16 67 and 70, 116 and 97)
constexpr uint32_t kTransposeFrom = 3u << 15;

struct BwdPlan {
    uint32_t R, n_slices, n_chunks, n_items;
    uint64_t M;             // n_slices * n_items counters
    uint64_t scan_blocks;   // blocks of the counter scan
    uint32_t max_parts;     // upper bound of the reduce grid
    uint64_t counts_off, sums_off, meta_off, parts_off, part_slice_off, partials_off, entries_off, bytes;
    // one-pass path: items of bucket_points points, each level's slices
    // [s_lo[l], s_hi[l]] (all it can reach), per item and slice of its level the run's start
    // and length
    bool bucket;
    bool wide;  // a level reaches more than kStageSlices slices, outside the box
    uint32_t n_bchunks, n_bitems, span_stride;
    uint32_t run_part;  // entries one workgroup of the reducer sums
    uint32_t s_lo[NGP_HASHGRID_MAX_LEVELS], s_hi[NGP_HASHGRID_MAX_LEVELS];
    uint64_t runs_off, slice_np_off, first_part_off, split_off, levels_off, rows_off;
    bool whole;      // no slice can be cut into parts
    bool transpose;  // a point-major gradient is copied level-major first (to partials_off)
};

// Rows of one slice: R rows of F f64 accumulators fill kSliceBytes of LDS.  A power
// of two, so the kernels split a row into (slice, row in slice) with shifts.
template <int F>
constexpr uint32_t slice_rows() {
    static_assert((kSliceBytes / (8 * F) & (kSliceBytes / (8 * F) - 1)) == 0, "slice rows: a power of two");
    return kSliceBytes / (8 * F);
}

// Slices of kRunSliceBytes for the one-pass form where every level then spans at most
// kStageSlices slices for points of the box, else of kSliceBytes; whether either fits.
// box_hi: the levels' last slices for points of the box.
inline bool plan_slices(const HashGridDescriptor &d, uint32_t slice_bytes, BwdPlan &p, uint32_t *box_hi) {
    p.R = slice_bytes / (8 * d.F);
    p.n_slices = div_up(d.n_rows, p.R);
    p.span_stride = 1;
    uint32_t box_span = 1;
    for (uint32_t l = 0; l < d.L; ++l) {
        p.s_lo[l] = d.offsets[l] / p.R;
        p.s_hi[l] = level_last_row(d, l) / p.R;
        p.span_stride = std::max(p.span_stride, p.s_hi[l] - p.s_lo[l] + 1u);
        box_hi[l] = level_last_box_row(d, l) / p.R;
        box_span = std::max(box_span, box_hi[l] - p.s_lo[l] + 1u);
    }
    p.wide = p.span_stride > kStageSlices;
    return d.F <= 2 && box_span <= kStageSlices;
}

inline uint64_t ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

inline BwdPlan make_plan(const HashGridDescriptor &d) {
    auto align = [](uint64_t x) { return (x + 255) / 256 * 256; };
    BwdPlan p{};
    const int ew = entry_words_host(d.F, d.table_dtype == NGP_DTYPE_F16);
    const bool half_values = d.F == 2 && d.table_dtype == NGP_DTYPE_F16;
    p.n_bchunks = std::max<uint32_t>(1, div_up(d.n_points, bucket_points(half_values)));
    // (entry indexes within a level are 32 bits; the small slices of a table past half of
    // kMaxSlices * kSliceBytes would be more than kMaxSlices; the sort below takes kSliceBytes)
    const bool short_index = (uint64_t)p.n_bchunks * bucket_entries(half_values) <= 0xffffffffull;
    uint32_t box_hi[NGP_HASHGRID_MAX_LEVELS];
    p.bucket = short_index && plan_slices(d, kRunSliceBytes, p, box_hi) && p.n_slices <= kMaxSlices;
    if (!p.bucket) p.bucket = plan_slices(d, kSliceBytes, p, box_hi) && short_index;
    if (p.bucket) {
        p.n_bitems = d.L * p.n_bchunks;
        const uint64_t runs = (uint64_t)p.n_bitems * p.span_stride;
        const uint64_t max_entries = (uint64_t)p.n_bitems * bucket_entries(half_values);
        // A batch's entries make at most kFullParts full parts, one and a half to a workgroup
        // that the chip holds: the slices of coarse levels, which hold most entries and whose
        // entries also collide more in the LDS atomics, are cut until the reducer's last round
        // is short, and a part costs its R * F f64 of the workspace.  A hashed level spreads 8
        // contributions a point evenly over its slices; where cutting all of these would only
        // double the parts, a part takes one of them whole, with a quarter to spare.  2^18 points
        // f32, L = 16, T = 2^19, all kernels, along rays and at random: 145 and 213 us; 512 parts
        // 165 and 215, 1,024 139 and 224, 2,048 175 and 318.  T = 2^17, 40,000 at random: 70,
        // with its hashed slices cut 106.  (Parts of 2.5 slices, cut once more where the sums were
        // grouped: T = 2^19 147 and 250, 2^17 213 and 319, 2^22 302 and 680, now 257 and 359.)
        const uint64_t E = 8ull * d.n_points * d.L, mean4 = 32ull * d.n_points * p.R;  // 4 T times the mean
        uint64_t want = ceil_div(E, 1024ull * kFullParts);
        if (mean4 / d.T * 5 <= std::min<uint64_t>(16ull * kPart, 32 * E / kFullParts))
            want = std::max(want, ceil_div(mean4 * 5, 16384ull * d.T));
        p.run_part = (uint32_t)std::min<uint64_t>(kPart, std::max<uint64_t>(kMinPart, want * 1024));
        // Few points: even all contributions of all levels that share kSliceBytes of rows inside
        // the box make one part, so nothing is counted, cut or combined: two launches, not four
        // (2000 ray samples f32: 35 -> 26 us; with every point in a fifth of the box 4000 points
        // take 73 us on either side).
        const uint32_t pair = p.R * d.F * 8 == kSliceBytes ? 0 : 1;
        uint32_t sharing = 0;
        for (uint32_t l = 0; l < d.L; ++l) {
            uint32_t n = 0;
            for (uint32_t k = 0; k < d.L; ++k)
                n += p.s_lo[k] >> pair <= p.s_lo[l] >> pair && box_hi[k] >> pair >= p.s_lo[l] >> pair;
            sharing = std::max(sharing, n);
        }
        p.whole = (uint64_t)d.n_points * 8 * sharing <= kPart;
        // Parts of cut slices: one of t > run_part entries has at most 2 (t - 1) / run_part, and
        // at most 1 + t / run_part.  A bounds E / run_part by what it is before run_part is rounded
        // up, so that a batch of fewer points never needs more workspace.
        const uint64_t A = std::min(ceil_div(E, kMinPart), std::max<uint64_t>(ceil_div(E, kPart), kFullParts));
        p.max_parts = p.whole ? 0 : (uint32_t)std::min(2 * A, p.n_slices + A);
        p.runs_off = 0;
        p.slice_np_off = align(p.runs_off + 4 * runs);
        p.first_part_off = align(p.slice_np_off + 4 * (uint64_t)p.n_slices);
        p.split_off = align(p.first_part_off + 4 * (uint64_t)p.n_slices);
        p.levels_off = align(p.split_off + 4 * (uint64_t)p.n_slices);
        p.meta_off = align(p.levels_off + 4 * (uint64_t)p.n_slices);  // [0] parts, [1] cut slices
        p.part_slice_off = align(p.meta_off + 8);
        p.partials_off = align(p.part_slice_off + 4 * (uint64_t)p.max_parts);
        p.transpose = d.F == 2 && d.enc_layout == NGP_ENC_POINT_MAJOR && !p.whole && d.n_points >= kTransposeFrom;
        const uint64_t lm_bytes = p.transpose ? (uint64_t)d.n_points * d.L * 8 : 0;
        p.entries_off = align(p.partials_off + std::max((uint64_t)p.max_parts * p.R * d.F * 8, lm_bytes));
        p.rows_off = align(p.entries_off + max_entries * value_bytes(d.F, d.table_dtype == NGP_DTYPE_F16));
        p.bytes = p.rows_off + max_entries * sizeof(uint16_t);
        return p;
    }
    p.n_chunks = std::max<uint32_t>(1, div_up(d.n_points, kChunk));
    p.n_items = d.L * p.n_chunks;
    p.M = (uint64_t)p.n_slices * p.n_items;
    p.scan_blocks = (p.M + kScanThreads * kScanPer - 1) / (kScanThreads * kScanPer);
    const uint64_t max_entries = (uint64_t)d.n_points * d.L * 8;
    // a slice with c entries takes max(1, ceil(c / kPart)) parts
    p.max_parts = (uint32_t)(p.n_slices + max_entries / kPart);
    p.counts_off = 0;
    p.sums_off = align(p.counts_off + 4 * p.M);
    p.meta_off = align(p.sums_off + 4 * p.scan_blocks);        // [0] total entries, [1] total parts
    p.parts_off = align(p.meta_off + 8);                          // first part of each slice
    p.part_slice_off = align(p.parts_off + 4 * ((uint64_t)p.n_slices + 1));  // slice of each part
    p.partials_off = align(p.part_slice_off + 4 * (uint64_t)p.max_parts);
    p.entries_off = align(p.partials_off + (uint64_t)p.max_parts * p.R * d.F * 4);
    p.bytes = p.entries_off + max_entries * 4 * ew;
    return p;
}

// Lane shifts on the vector ALU (DPP), no LDS: lanes without a source, or in rows
// the row mask leaves out, get `fill`.
constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118;
constexpr int kWaveShl1 = 0x130, kWaveShr1 = 0x138, kRowBcast15 = 0x142, kRowBcast31 = 0x143;

template <int kCtrl, int kRowMask>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v, uint32_t fill) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)fill, (int)v, kCtrl, kRowMask, 0xf, false);
}

// One step of the segmented inclusive sum: combine with the pair the shift brings
// (0 and flag 0 where there is none, which changes nothing).
template <int kCtrl, int kRowMask, int F>
__device__ __forceinline__ void seg_step(float *v, uint32_t &fl) {
    const uint32_t fin = dpp_u32<kCtrl, kRowMask>(fl, 0u);
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const float vin = __uint_as_float(dpp_u32<kCtrl, kRowMask>(__float_as_uint(v[f]), 0u));
        v[f] = fl ? v[f] : v[f] + vin;
    }
    fl |= fin;
}

// The run-merged contributions of one point per lane at level l: the wavefront's
// 64 lanes hold 64 consecutive points; for each corner, lanes whose row equals the
// previous lane's join its run, and emit(row, v) is called on each run's last lane
// with the run's summed values.  Inactive lanes (past the last point) get keys no
// active lane has, so they form no runs.
template <int F, bool kValues, typename Emit>
__device__ __forceinline__ void point_runs(const HashGridDescriptor &d, uint32_t l, float scale, uint32_t res,
                                           bool dense, bool pow2, const float *xyz, const float *gin, bool active,
                                           Emit emit) {
    const int lane = lane_id();
    float p[3];
    normalise(make_divisor(2.0f * d.bound), d.bound, xyz, p);
    uint32_t idx[8];
    float w[8];
    with_rule(dense, pow2, [&](auto rule, auto p2) {
        level_vertices_t<decltype(rule)::value, decltype(p2)::value>(p[0], p[1], p[2], scale, res, dense, d.T,
                                                                     d.offsets[l], d.n_rows - 1u, idx, w);
    });
    float g[F];
#pragma unroll
    for (int f = 0; f < F; ++f) g[f] = kValues && active ? gin[f] : 0.0f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const uint32_t key = active ? idx[c] : 0xffffffffu - (uint32_t)lane;
        float v[F];
#pragma unroll
        for (int f = 0; f < F; ++f) v[f] = w[c] * g[f];
        const uint32_t prev = dpp_u32<kWaveShr1, 0xf>(key, ~key);  // lane 0: no predecessor
        const bool head = prev != key;
        bool tail = true;
        if (__ballot(!head) != 0) {
            if (kValues) {
                // segmented inclusive sums of runs: (v, flag) pairs combined by
                // (a, fa) + (b, fb) = (fb ? b : a + b, fa | fb), shifts within
                // 16-lane rows, then row 15 -> rows 1 and 3, lane 31 -> rows 2 and 3
                uint32_t fl = head ? 1u : 0u;
                seg_step<kRowShr1, 0xf, F>(v, fl);
                seg_step<kRowShr2, 0xf, F>(v, fl);
                seg_step<kRowShr4, 0xf, F>(v, fl);
                seg_step<kRowShr8, 0xf, F>(v, fl);
                seg_step<kRowBcast15, 0xa, F>(v, fl);
                seg_step<kRowBcast31, 0xc, F>(v, fl);
            }
            const uint32_t next_head = dpp_u32<kWaveShl1, 0xf>(head ? 1u : 0u, 1u);  // lane 63: end of wave
            tail = next_head != 0u;
        }
        if (tail && active) emit(key, v, c);
    }
}

// Visits the run-merged contributions of work item `item` (level l, kChunk
// consecutive points) and calls emit(row, v, corner) on each run's last lane.
// The same inputs always give the same multiset of emitted rows, so counting and
// scattering agree.
template <int F, bool kValues, typename Emit>
__device__ __forceinline__ void item_contributions(const HashGridDescriptor &d, const BwdPlan &p, uint32_t item,
                                                   const float *__restrict__ pos, const float *__restrict__ dL_denc,
                                                   Emit emit) {
    const uint32_t l = item / p.n_chunks, k = item % p.n_chunks;
    const bool pow2 = (d.T & (d.T - 1u)) == 0;
    const bool level_major = d.enc_layout == NGP_ENC_LEVEL_MAJOR;
    const float scale = d.scales[l];
    const uint32_t res = d.resolutions[l];
    const bool dense = l < d.first_hash_level;
    constexpr int kSubs = kChunk / kItemThreads;
    // the inputs of a group of sub-chunks are all loaded before any is used, so
    // the loads overlap; 8 features per level hold half as many in flight (all
    // eight sub-chunks of them would not fit the registers)
    constexpr int kGroup = F >= 8 ? kSubs / 2 : kSubs;
    for (int g0 = 0; g0 < kSubs; g0 += kGroup) {
        float xyz[kGroup][3], gin[kGroup][F];
#pragma unroll
        for (int sub = 0; sub < kGroup; ++sub) {
            const uint32_t n = k * kChunk + (g0 + sub) * kItemThreads + threadIdx.x;
            const uint32_t np = n < d.n_points ? n : d.n_points - 1;
#pragma unroll
            for (int a = 0; a < 3; ++a) xyz[sub][a] = pos[3 * (size_t)np + a];
            if (kValues) {
                const size_t gb =
                    level_major ? ((size_t)l * d.n_points + np) * F : (size_t)np * d.L * F + (size_t)l * F;
#pragma unroll
                for (int f = 0; f < F; ++f) gin[sub][f] = dL_denc[gb + f];
            }
        }
#pragma unroll
        for (int sub = 0; sub < kGroup; ++sub) {
            const uint32_t n = k * kChunk + (g0 + sub) * kItemThreads + threadIdx.x;
            point_runs<F, kValues>(d, l, scale, res, dense, pow2, xyz[sub], gin[sub], n < d.n_points, emit);
        }
    }
}

// 1. per item, entries per slice (slice-major counters)
template <int F>
__global__ void __launch_bounds__(kItemThreads)
    bwd_count_kernel(HashGridDescriptor d, BwdPlan p, const float *__restrict__ pos, uint32_t *__restrict__ counts) {
    constexpr uint32_t R = slice_rows<F>();
    __shared__ uint32_t hist[kMaxSlices];
    for (uint32_t s = threadIdx.x; s < p.n_slices; s += kItemThreads) hist[s] = 0u;
    __syncthreads();
    const uint32_t item = blockIdx.x;
    item_contributions<F, false>(d, p, item, pos, nullptr,
                                 [&](uint32_t row, const float *, int) { atomicAdd(&hist[row / R], 1u); });
    __syncthreads();
    for (uint32_t s = threadIdx.x; s < p.n_slices; s += kItemThreads) counts[(size_t)s * p.n_items + item] = hist[s];
}

// 2a. per-block sums of kScanThreads * kScanPer counters
__global__ void __launch_bounds__(kScanThreads) scan_sums_kernel(uint64_t M, const uint32_t *__restrict__ a,
                                                                 uint32_t *__restrict__ sums) {
    const uint64_t base = (uint64_t)blockIdx.x * kScanThreads * kScanPer;
    uint32_t v = 0;
#pragma unroll
    for (int q = 0; q < kScanPer; ++q) {
        const uint64_t i = base + (uint64_t)q * kScanThreads + threadIdx.x;
        if (i < M) v += a[i];
    }
    __shared__ uint32_t ws[kScanThreads / kWave];
    v = wave_sum(v);
    if (lane_id() == 0) ws[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int w = 0; w < kScanThreads / kWave; ++w) t += ws[w];
        sums[blockIdx.x] = t;
    }
}

// 2b. exclusive scan inside each block plus the block's prefix (the sum of the
// block sums before it, added by the workgroup itself), in place; the last block
// writes the total entries into meta[0]
__global__ void __launch_bounds__(kScanThreads) scan_apply_kernel(uint64_t M, uint32_t *__restrict__ a,
                                                                  const uint32_t *__restrict__ sums,
                                                                  uint32_t *__restrict__ meta) {
    __shared__ uint32_t ws[kScanThreads / kWave];
    __shared__ uint32_t prefix;
    uint32_t v = 0;
    for (uint32_t j = threadIdx.x; j < blockIdx.x; j += kScanThreads) v += sums[j];
    v = wave_sum(v);
    if (lane_id() == 0) ws[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int w = 0; w < kScanThreads / kWave; ++w) t += ws[w];
        prefix = t;
    }
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * kScanThreads * kScanPer;
    uint32_t carry = prefix;
    for (int q = 0; q < kScanPer; ++q) {
        const uint64_t i = base + (uint64_t)q * kScanThreads + threadIdx.x;
        const uint32_t x = i < M ? a[i] : 0u;
        uint32_t tot;
        const uint32_t ex = block_exclusive_scan<kScanThreads>(x, &tot);
        if (i < M) a[i] = carry + ex;
        carry += tot;
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) meta[0] = carry;
}

__device__ __forceinline__ uint32_t slice_begin(const BwdPlan &p, const uint32_t *offsets, const uint32_t *meta,
                                                uint32_t s) {
    return s < p.n_slices ? offsets[(size_t)s * p.n_items] : meta[0];
}

// 2d. one workgroup: parts per slice (kPart entries each, at least one) and their
// prefix, and the slice of every part; parts[n_slices] and meta[1] hold the total.
__global__ void __launch_bounds__(kScanThreads) plan_parts_kernel(BwdPlan p, const uint32_t *__restrict__ offsets,
                                                                  uint32_t *__restrict__ meta,
                                                                  uint32_t *__restrict__ parts,
                                                                  uint32_t *__restrict__ part_slice) {
    uint32_t carry = 0;
    for (uint32_t c = 0; c < p.n_slices; c += kScanThreads) {
        const uint32_t s = c + threadIdx.x;
        uint32_t k = 0;
        if (s < p.n_slices) {
            const uint32_t cnt = slice_begin(p, offsets, meta, s + 1) - slice_begin(p, offsets, meta, s);
            k = cnt == 0 ? 1u : (cnt + kPart - 1) / kPart;
        }
        uint32_t tot;
        const uint32_t ex = block_exclusive_scan<kScanThreads>(k, &tot);
        if (s < p.n_slices) {
            parts[s] = carry + ex;
            for (uint32_t j = 0; j < k; ++j) part_slice[carry + ex + j] = s;
        }
        carry += tot;
    }
    if (threadIdx.x == 0) {
        parts[p.n_slices] = carry;
        meta[1] = carry;
    }
}

// 3. entries at each item's offsets
template <int F, bool kHalf>
__global__ void __launch_bounds__(kItemThreads)
    bwd_scatter_kernel(HashGridDescriptor d, BwdPlan p, const float *__restrict__ pos, const float *__restrict__ dL_denc,
                       const uint32_t *__restrict__ offsets, uint32_t *__restrict__ entries) {
    constexpr int EW = entry_words<F, kHalf>();
    constexpr uint32_t R = slice_rows<F>();
    __shared__ uint32_t cursor[kMaxSlices];
    const uint32_t item = blockIdx.x;
    for (uint32_t s = threadIdx.x; s < p.n_slices; s += kItemThreads) cursor[s] = offsets[(size_t)s * p.n_items + item];
    __syncthreads();
    item_contributions<F, true>(d, p, item, pos, dL_denc, [&](uint32_t row, const float *v, int) {
        const uint32_t s = row / R;
        const uint32_t at = atomicAdd(&cursor[s], 1u);
        uint32_t w[EW];
#pragma unroll
        for (int k = 0; k < EW; ++k) w[k] = 0u;
        w[0] = row - s * R;
        pack_values<F, kHalf>(w, v);
        uint4 *e = reinterpret_cast<uint4 *>(entries + (size_t)at * EW);
        if constexpr (EW == 2) {
            *reinterpret_cast<uint2 *>(entries + (size_t)at * EW) = make_uint2(w[0], w[1]);
        } else if constexpr (EW == 3) {
            *reinterpret_cast<uint3 *>(entries + (size_t)at * EW) = make_uint3(w[0], w[1], w[2]);
        } else {
#pragma unroll
            for (int q = 0; q < EW / 4; ++q) e[q] = make_uint4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
        }
    });
}


// Item (l, k)'s run of the sl-th slice of level l: start within the item's region and
// length (both at most bucket_entries, 2^13) in one word.  Slice-major, so a reducer
// reads the runs of one slice side by side.
static_assert(bucket_entries(false) < 0x10000u, "run starts and lengths fit 16 bits");
__device__ __forceinline__ uint32_t pack_run(uint32_t start, uint32_t n) { return start | n << 16; }
__device__ __forceinline__ uint32_t run_start(uint32_t r) { return r & 0xffffu; }
__device__ __forceinline__ uint32_t run_length(uint32_t r) { return r >> 16; }
__device__ __forceinline__ size_t run_index(const BwdPlan &p, uint32_t l, uint32_t sl, uint32_t k) {
    return ((size_t)l * p.span_stride + sl) * p.n_bchunks + k;
}

// The wavefront's runs of consecutive points in one cell, as lane masks: `head` bit i is
// set where lane i starts a run, `keep[s]` where lane i takes nothing in step s of the
// segmented sum (its own run starts within the lanes step s would add).  Computed on the
// scalar unit once per point, for all corners and features.
struct CellRuns {
    uint64_t head, keep[6];
};

__device__ __forceinline__ CellRuns cell_runs(uint64_t head) {
    constexpr uint64_t kRow1 = 0x0001000100010001ull, kRow2 = 0x0003000300030003ull, kRow4 = 0x000f000f000f000full,
                       kRow8 = 0x00ff00ff00ff00ffull, kRows13 = 0xffff0000ffff0000ull, kRows23 = 0xffffffff00000000ull;
    CellRuns r;
    r.head = head;
    uint64_t f = head;  // lane i: a run starts within the lanes summed so far
    r.keep[0] = f;
    f |= (f << 1) & ~kRow1;
    r.keep[1] = f;
    f |= (f << 2) & ~kRow2;
    r.keep[2] = f;
    f |= (f << 4) & ~kRow4;
    r.keep[3] = f;
    f |= (f << 8) & ~kRow8;
    r.keep[4] = f | ~kRows13;
    f |= ((f >> 15) & 1ull) * 0x00000000ffff0000ull | ((f >> 47) & 1ull) * 0xffff000000000000ull;
    r.keep[5] = f | ~kRows23;
    return r;
}

// The last lane of each run (a lane past the last point starts a run of its own, so the
// last point's lane ends one).
__device__ __forceinline__ uint64_t run_ends(const CellRuns &r) { return r.head >> 1 | 1ull << 63; }

constexpr uint32_t kNoEntry = 0xffffffffu;

template <int kCtrl, int N>
__device__ __forceinline__ void run_step(float *v, uint64_t keep) {
    if (~keep == 0ull) return;  // uniform: no lane has anything to take in this step
    const bool k = __builtin_amdgcn_inverse_ballot_w64(keep);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float in = v[i] + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v[i]), kCtrl, 0xf, 0xf, true));
        v[i] = k ? v[i] : in;
    }
}

// Sums N values over each run; a run's last lane ends with its total.  Shifts within
// 16-lane rows, then row 15 -> rows 1 and 3, lane 31 -> rows 2 and 3.  Steps that no
// run reaches are skipped, so the finest levels, where consecutive samples lie in
// different cells, do none.
template <int N>
__device__ __forceinline__ void sum_runs(float *v, const CellRuns &r) {
    run_step<kRowShr1, N>(v, r.keep[0]);
    run_step<kRowShr2, N>(v, r.keep[1]);
    run_step<kRowShr4, N>(v, r.keep[2]);
    run_step<kRowShr8, N>(v, r.keep[3]);
    run_step<kRowBcast15, N>(v, r.keep[4]);
    run_step<kRowBcast31, N>(v, r.keep[5]);
}

// One-pass table gradient, part 1 (F <= 2).  Block = item (level l, bucket_points
// consecutive points, one per thread and phase).  The item's contributions are computed
// once and kept in registers: a wavefront's 64 lanes hold 64 consecutive points, and
// runs of points in the same cell (all eight corners alike) are summed into the run's
// last lane, which takes each corner's rank within its slice from an LDS counter.  An
// exclusive scan of the counters places each slice's run in the item's own region of
// the entry buffer (bucket_entries), the entries go to run start + rank, and
// the run's start and length are stored for the reducers.  Within a run, entries are in
// LDS-atomic order; the reducer's sums do not depend on it beyond f64 rounding.
// 2^18 ray samples: f32 110 -> 68 us, f16 90 -> 55 us.  It was bound by the run merge
// (each corner found its own runs: 626 vector instructions a wavefront and level) and,
// once that was cheaper (86 us), by 17 M scattered 12-byte stores.  kSlices: counters for as
// many slices as a level can reach; the last of them, kMaxSlices, take 32 KiB of LDS.
template <int F, bool kHalf, uint32_t R, uint32_t kSlices>
__global__ void __launch_bounds__(kBucketThreads)
    bwd_bucket_kernel(HashGridDescriptor d, BwdPlan p, const float *__restrict__ pos,
                      const float *__restrict__ dL_denc, uint32_t *__restrict__ runs_out,
                      EntryValue<F, kHalf> *__restrict__ values, uint16_t *__restrict__ rows_out,
                      uint32_t *__restrict__ meta) {
    typedef EntryValue<F, kHalf> Value;
    constexpr int kBucketPhases = bucket_phases(kHalf);
    constexpr uint32_t kBucketPoints = bucket_points(kHalf), kBucketEntries = bucket_entries(kHalf);
    static_assert(R <= 0x10000u, "rows within a slice fit 16 bits");
    constexpr int kPer = kSlices / kBucketThreads;
    static_assert(kPer * kBucketThreads == kSlices, "whole slice counters per thread");
    __shared__ uint32_t cnt[kSlices];
    __shared__ __align__(16) Value stage_v[kStageEntries];
    __shared__ __align__(16) uint16_t stage_r[kStageEntries];
    const uint32_t item = blockIdx.x;
    if (item == 0 && threadIdx.x < 2) meta[threadIdx.x] = 0u;  // for bwd_slice_parts_kernel
    const uint32_t l = item / p.n_bchunks, k = item % p.n_bchunks;
    const uint32_t s_lo = p.s_lo[l];
    const uint32_t span = p.s_hi[l] - s_lo + 1u;  // <= kSlices (host check)
    const bool pow2 = (d.T & (d.T - 1u)) == 0;
    const bool level_major = d.enc_layout == NGP_ENC_LEVEL_MAJOR;
    const float scale = d.scales[l];
    // all phases' inputs are loaded up front, so only the first phase waits on memory
    float xyz_all[kBucketPhases][3], gin_all[kBucketPhases][F];
#pragma unroll
    for (int ph = 0; ph < kBucketPhases; ++ph) {
        const uint32_t n = k * kBucketPoints + ph * kBucketThreads + threadIdx.x;
        const uint32_t np = n < d.n_points ? n : d.n_points - 1;
#pragma unroll
        for (int q = 0; q < 3; ++q) xyz_all[ph][q] = pos[3 * (size_t)np + q];
        const size_t gb = level_major ? ((size_t)l * d.n_points + np) * F : (size_t)np * d.L * F + (size_t)l * F;
#pragma unroll
        for (int f = 0; f < F; ++f) gin_all[ph][f] = dL_denc[gb + f];
    }
#pragma unroll
    for (int q = 0; q < kPer; ++q) cnt[kPer * threadIdx.x + q] = 0u;
    __syncthreads();  // counters cleared
    uint32_t rows[kBucketPhases][8], rank[kBucketPhases][8];
    float vals[kBucketPhases][8 * F];
    const Divisor two_b = make_divisor(2.0f * d.bound);
#pragma unroll
    for (int ph = 0; ph < kBucketPhases; ++ph) {
        const uint32_t n = k * kBucketPoints + ph * kBucketThreads + threadIdx.x;
        const uint64_t active = __ballot(n < d.n_points);
        float q[3], w[8];
        normalise(two_b, d.bound, xyz_all[ph], q);
        with_rule(l < d.first_hash_level, pow2, [&](auto rule, auto p2) {
            level_vertices_t<decltype(rule)::value, decltype(p2)::value>(
                q[0], q[1], q[2], scale, d.resolutions[l], l < d.first_hash_level, d.T, d.offsets[l], d.n_rows - 1u,
                rows[ph], w);
        });
        // a lane continues the previous lane's run if both points lie in one cell (a NaN
        // position is in none); points past the end are runs of their own.  The lane shifts
        // come before any comparison: a shift reads nothing from a lane that is masked off.
        float cell[3], before[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            cell[a] = floorf(q[a] * scale + 0.5f);
            before[a] = __uint_as_float(dpp_u32<kWaveShr1, 0xf>(__float_as_uint(cell[a]), 0x7fc00000u));
        }
        const bool same = (n < d.n_points) & (cell[0] == before[0]) & (cell[1] == before[1]) & (cell[2] == before[2]);
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int f = 0; f < F; ++f) vals[ph][c * F + f] = w[c] * gin_all[ph][f];
        // f16 values are rounded once per entry, so there a row that neighbouring points of
        // different cells share by a hash collision is one entry too: its wavefront (rare)
        // finds the runs of each corner
        bool clash = false;
        if constexpr (kHalf) {
#pragma unroll
            for (int c = 0; c < 8; ++c) clash |= rows[ph][c] == dpp_u32<kWaveShr1, 0xf>(rows[ph][c], ~rows[ph][c]);
            clash = clash & !same & (n < d.n_points);
        }
        if (kHalf && __ballot(clash) != 0ull) {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const bool eq = rows[ph][c] == dpp_u32<kWaveShr1, 0xf>(rows[ph][c], ~rows[ph][c]);
                const CellRuns runs = cell_runs(~__ballot(eq & (n < d.n_points)));
                sum_runs<F>(vals[ph] + c * F, runs);
                rank[ph][c] = kNoEntry;
                if (__builtin_amdgcn_inverse_ballot_w64(run_ends(runs) & active))
                    rank[ph][c] = atomicAdd(&cnt[rows[ph][c] / R - s_lo], 1u);
            }
        } else {
            const CellRuns runs = cell_runs(~__ballot(same));
            sum_runs<8 * F>(vals[ph], runs);
#pragma unroll
            for (int c = 0; c < 8; ++c) rank[ph][c] = kNoEntry;
            if (__builtin_amdgcn_inverse_ballot_w64(run_ends(runs) & active)) {
#pragma unroll
                for (int c = 0; c < 8; ++c) rank[ph][c] = atomicAdd(&cnt[rows[ph][c] / R - s_lo], 1u);
            }
        }
    }
    __syncthreads();
    uint32_t mine[kPer], sum = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        mine[q] = cnt[kPer * threadIdx.x + q];
        sum += mine[q];
    }
    uint32_t total;
    uint32_t ex = block_exclusive_scan<kBucketThreads>(sum, &total);
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const uint32_t sl = kPer * threadIdx.x + q;
        cnt[sl] = ex;  // from here on, the start of slice sl's run
        if (sl < span) runs_out[run_index(p, l, sl, k)] = pack_run(ex, mine[q]);
        ex += mine[q];
    }
    __syncthreads();
    // rank becomes the entry's place in the item's region
#pragma unroll
    for (int ph = 0; ph < kBucketPhases; ++ph) {
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (rank[ph][c] != kNoEntry) rank[ph][c] += cnt[rows[ph][c] / R - s_lo];
    }
    // the region, kStageEntries at a time through LDS: each 64-byte request to the L2
    // carries whole neighbouring entries (scattered entry by entry, 17 M requests of 12
    // bytes took the L2 channels longer than everything else here)
    const size_t region = (size_t)item * kBucketEntries;
    for (uint32_t e0 = 0; e0 < total; e0 += kStageEntries) {
        if (e0 > 0) __syncthreads();  // the stage is read out
#pragma unroll
        for (int ph = 0; ph < kBucketPhases; ++ph) {
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const uint32_t at = rank[ph][c] - e0;
                if (at < kStageEntries) {
                    Value v;
                    v.pack(vals[ph] + c * F);
                    stage_v[at] = v;
                    stage_r[at] = (uint16_t)(rows[ph][c] % R);
                }
            }
        }
        __syncthreads();
        const uint32_t n = min(total - e0, kStageEntries);
        // whole 16-byte vectors; the last may reach past n, within the item's region
        constexpr uint32_t kV = 16 / sizeof(Value), kR = 16 / sizeof(uint16_t);
        uint4 *const gv = reinterpret_cast<uint4 *>(values + region + e0);
        uint4 *const gr = reinterpret_cast<uint4 *>(rows_out + region + e0);
        for (uint32_t t = threadIdx.x; t < (n + kV - 1) / kV; t += kBucketThreads)
            gv[t] = reinterpret_cast<const uint4 *>(stage_v)[t];
        for (uint32_t t = threadIdx.x; t < (n + kR - 1) / kR; t += kBucketThreads)
            gr[t] = reinterpret_cast<const uint4 *>(stage_r)[t];
    }
}

// One-pass table gradient, part 2: the number of parts of slice s, run_part entries each in
// (level, chunk) order of the items, from the run lengths of every item whose level reaches
// it, and for a slice of several a slot for each and its place in the list of cut slices.
// Also the levels that have entries in s: outside the box a dense level reaches many slices,
// inside few.
__global__ void __launch_bounds__(256)
    bwd_slice_parts_kernel(HashGridDescriptor d, BwdPlan p, const uint32_t *__restrict__ runs,
                           uint32_t *__restrict__ meta, uint32_t *__restrict__ slice_np,
                           uint32_t *__restrict__ first_part, uint32_t *__restrict__ part_slice,
                           uint32_t *__restrict__ split, uint32_t *__restrict__ slice_levels) {
    const uint32_t s = blockIdx.x;
    uint32_t own = 0, levels = 0;
    for (uint32_t l = 0; l < d.L; ++l) {
        if (s < p.s_lo[l] || s > p.s_hi[l]) continue;
        const uint32_t before = own;
        for (uint32_t k = threadIdx.x; k < p.n_bchunks; k += 256)
            own += run_length(runs[run_index(p, l, s - p.s_lo[l], k)]);
        if (__ballot(own != before) != 0ull) levels |= 1u << l;
    }
    __shared__ uint32_t ws[2][256 / kWave];
    own = wave_sum(own);
    if (lane_id() == 0) {
        ws[0][threadIdx.x / kWave] = own;
        ws[1][threadIdx.x / kWave] = levels;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t t = 0;
        uint32_t m = 0;
        for (int w = 0; w < 256 / kWave; ++w) {
            t += ws[0][w];
            m |= ws[1][w];
        }
        slice_levels[s] = m;
        const uint32_t n = t == 0 ? 1u : (uint32_t)((t + p.run_part - 1) / p.run_part);
        slice_np[s] = n;
        if (n > 1) {  // which slot a part gets does not matter to its sums
            const uint32_t at = atomicAdd(meta, n);
            first_part[s] = at;
            for (uint32_t j = 0; j < n; ++j) part_slice[at + j] = s;
            split[atomicAdd(meta + 1, 1u)] = s;
        }
    }
}

template <int EW>
__device__ __forceinline__ void load_entry(const uint32_t *__restrict__ src, uint32_t *w) {
    if constexpr (EW == 2) {
        const uint2 q = *reinterpret_cast<const uint2 *>(src);
        w[0] = q.x;
        w[1] = q.y;
    } else if constexpr (EW == 3) {
        const uint3 q = *reinterpret_cast<const uint3 *>(src);
        w[0] = q.x;
        w[1] = q.y;
        w[2] = q.z;
    } else {
#pragma unroll
        for (int q = 0; q < EW / 4; ++q) {
            const uint4 u = reinterpret_cast<const uint4 *>(src)[q];
            w[4 * q] = u.x;
            w[4 * q + 1] = u.y;
            w[4 * q + 2] = u.z;
            w[4 * q + 3] = u.w;
        }
    }
}

// 4. workgroup b sums part b's entries in LDS.  A slice of one part writes its
// rows of the gradient; a slice of several writes partial rows, summed in order
// by combine_kernel.  The LDS sums are f64 (each row rounded to f32 once at the
// end): f64 LDS atomics run several times faster than f32 ones here, and they
// keep full relative precision whatever the magnitudes, with inf and NaN
// propagating as in a float sum.
template <int F, bool kHalf>
__global__ void __launch_bounds__(kReduceThreads)
    bwd_reduce_kernel(HashGridDescriptor d, BwdPlan p, const uint32_t *__restrict__ offsets,
                      const uint32_t *__restrict__ meta, const uint32_t *__restrict__ parts,
                      const uint32_t *__restrict__ part_slice, const uint32_t *__restrict__ entries,
                      float *__restrict__ partials, float *__restrict__ dtable) {
    constexpr int EW = entry_words<F, kHalf>();
    extern __shared__ double acc[];
    const uint32_t b = blockIdx.x;
    if (b >= meta[1]) return;
    const uint32_t s = part_slice[b];
    const uint32_t part = b - parts[s];
    const uint32_t n_parts = parts[s + 1] - parts[s];
    const uint32_t s_begin = slice_begin(p, offsets, meta, s), s_end = slice_begin(p, offsets, meta, s + 1);
    const uint32_t begin = s_begin + part * kPart;
    const uint32_t end = min(s_end, begin + kPart);
    const uint32_t rows = min(d.n_rows - s * p.R, p.R);
    // feature f of local row r at acc[f * R + r]: one atomic instruction's rows
    // spread over all banks
    for (uint32_t t = threadIdx.x; t < p.R * F; t += kReduceThreads) acc[t] = 0.0;
    __syncthreads();
    // kU entries in flight per thread: the loads are unconditional (indices past the
    // part clamp to its last entry and are dropped afterwards), so they issue back
    // to back instead of each waiting in its own branch
    constexpr int kU = 8;
    for (uint32_t e0 = begin; e0 < end; e0 += kU * kReduceThreads) {
        uint32_t w[kU][EW];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const uint32_t e = min(e0 + u * kReduceThreads + threadIdx.x, end - 1u);
            load_entry<EW>(entries + (size_t)e * EW, w[u]);
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const bool in = e0 + u * kReduceThreads + threadIdx.x < end;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const float v = entry_value<F, kHalf>(w[u], f);
                if (in && v != 0.0f) atomicAdd(&acc[f * p.R + w[u][0]], (double)v);
            }
        }
    }
    __syncthreads();
    float *out = n_parts == 1 ? dtable + (size_t)s * p.R * F : partials + (size_t)b * p.R * F;
    for (uint32_t t = threadIdx.x; t < rows * F; t += kReduceThreads) out[t] = (float)acc[(t % F) * p.R + t / F];
}

// One-pass table gradient, part 3: a workgroup sums one part of slice s, as
// bwd_reduce_kernel does, from the runs of the items whose level reaches s.  The first
// kSplitBlocks workgroups take the parts of cut slices, the others a whole slice each.
// The LDS atomics set the time (about 31 cycles of a CU per 64-lane f64 add, however many
// of its lanes are masked off), so a wavefront reads its runs as one sequence with every
// lane filled: lane i of wavefront w loads the run of item w + i * kWaves, a prefix sum of
// the lengths places the runs in the sequence, and 64 entries at a time find their runs by
// pushing each run's lane number to the lane of its first entry and a running maximum
// (RunSequence).  kSteps such groups are loaded before the previous ones are added.  A
// whole slice (nearly all of them) needs no barrier between its runs; a part of a cut
// slice first finds its items by the prefixes of their run lengths: those that start within
// it.  Its sums stay f64 until the parts are added, so the result does not depend on the cut.
// With kAdam, a slice summed in one part is not stored: its rows take the optimizer
// step in place (params, m, v), and bwd_combine_runs does the same for the others.
// 2^18 ray samples, f32: 82 -> 67 us, of which the atomics themselves need 27 (34 M f64
// adds at 1.27 T/s); slices of 64 KiB, two workgroups to a CU, so that one clears or
// stores its rows while the other adds (128 KiB slices: 80 us); 1,024 points: 29 -> 17.
// All four kernels: f32 190 -> 145 us (68 + 5 + 67 + 5), f16 176 -> 130 (55 + 7 + 64 + 5);
// 1,024 points, two kernels: 44 -> 25.
struct RunSequence {
    uint32_t *marks;        // 64 words of LDS of the wavefront's own, tags below `tag`
    uint32_t tag;           // of the latest group of 64 places
    uint32_t start, total;  // this lane's run: first place in the sequence; places in all
    uint32_t shift;         // entry index of a place of this lane's run, less the place
    uint32_t last;          // lane number + 1 of the run the previous group ended in
    bool any;               // this lane's run is not empty

    // `entry0`: index of the run's first entry
    __device__ __forceinline__ void init(uint32_t len, uint32_t entry0) {
        const uint32_t incl = wave_inclusive_scan(len);
        start = incl - len;
        total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        shift = entry0 - start;
        any = len > 0;
        last = 0;
    }
    // The entry at place t0 + lane (the last one past the end), for t0 = 0, 64, ...
    __device__ __forceinline__ uint32_t entry(uint32_t t0) {
        const uint32_t lane = lane_id(), to = start - t0;
        ++tag;
        if (any && to < (uint32_t)kWave) marks[to] = tag << 8 | (lane + 1u);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const uint32_t m = marks[lane];
        uint32_t r = m >> 8 == tag ? m & 0xffu : 0u;  // a run of this group starts here
        r = max(r, dpp_u32<kRowShr1, 0xf>(r, 0u));
        r = max(r, dpp_u32<kRowShr2, 0xf>(r, 0u));
        r = max(r, dpp_u32<kRowShr4, 0xf>(r, 0u));
        r = max(r, dpp_u32<kRowShr8, 0xf>(r, 0u));
        r = max(r, dpp_u32<kRowBcast15, 0xf>(r, 0u));
        r = max(r, dpp_u32<kRowBcast31, 0xf>(r, 0u));
        r = max(r, last);
        last = (uint32_t)__builtin_amdgcn_readlane((int)r, kWave - 1);
        const uint32_t sh = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((r - 1u) * 4u), (int)shift);
        return sh + min(t0 + lane, total - 1u);
    }
};

constexpr int kSteps = 6;  // groups of 64 entries in flight

template <int F, bool kHalf>
struct EntryGroup {
    EntryValue<F, kHalf> v[kSteps];
    uint32_t row[kSteps];

    __device__ __forceinline__ void load(RunSequence &seq, uint32_t t0, const EntryValue<F, kHalf> *__restrict__ values,
                                         const uint16_t *__restrict__ rows) {
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            if (t0 + q * kWave < seq.total) {  // the same for the whole wavefront
                const uint32_t e = seq.entry(t0 + q * kWave);
                v[q] = values[e];
                row[q] = rows[e];
            }
        }
    }
    template <uint32_t R>
    __device__ __forceinline__ void add(double *acc, uint32_t t0, uint32_t total) const {
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            const bool in = t0 + q * kWave + lane_id() < total;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const float x = v[q].get(f);
                if (in && x != 0.0f) atomicAdd(&acc[f * R + row[q]], (double)x);
            }
        }
    }
};

constexpr uint32_t kSplitBlocks = 512;  // two to a CU

// What becomes of a row's sum: stored in f32, an optimizer step, or stored in f16 (the
// gradient of an f16 table, rounded as a cast of the f32 sum would; a cast of the whole table
// afterwards took 10-14 us for 6.1 M rows).
enum { kFloatRows, kAdamRows, kHalfRows };

template <int F, bool kHalf, uint32_t R, int kOut>
__device__ __forceinline__ void
reduce_part(const HashGridDescriptor &d, const BwdPlan &p, uint32_t s, uint32_t part, uint32_t n_parts, uint32_t slot,
            uint32_t levels, const uint32_t *__restrict__ runs, const EntryValue<F, kHalf> *__restrict__ values,
            const uint16_t *__restrict__ entry_rows, double *__restrict__ partials, void *__restrict__ dtable, const AdamStep &adam, float *__restrict__ adam_p, float *__restrict__ adam_m,
            float *__restrict__ adam_v) {
    typedef EntryGroup<F, kHalf> Group;
    constexpr uint32_t kBucketEntries = bucket_entries(kHalf);
    constexpr uint32_t kWaves = kRunThreads / kWave;
    extern __shared__ double acc[];
    __shared__ uint32_t chosen[kRunThreads];
    __shared__ uint32_t marks[kWaves][kWave];
    const uint32_t rows = min(d.n_rows - s * R, R);
    for (uint32_t t = threadIdx.x; t < R * F / 2; t += kRunThreads) reinterpret_cast<double2 *>(acc)[t] = double2{0.0, 0.0};
    __syncthreads();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t lane = lane_id();
    RunSequence seq;
    seq.marks = marks[wave];
    seq.tag = 0;
    seq.marks[lane] = 0u;
    uint32_t carry = 0;  // entries of the items visited before
    for (uint32_t left = levels; left != 0; left &= left - 1u) {
        const uint32_t l = (uint32_t)__builtin_ctz(left);
        const uint32_t *level_runs = runs + run_index(p, l, s - p.s_lo[l], 0);
        for (uint32_t k0 = 0; k0 < p.n_bchunks; k0 += kRunThreads) {
            const uint32_t n_k = min(p.n_bchunks - k0, (uint32_t)kRunThreads);
            const uint32_t k = wave + lane * kWaves;  // this lane's run of the tile
            uint32_t my_run = 0;
            if (n_parts == 1) {
                if (k < n_k) my_run = level_runs[k0 + k];
            } else {
                const uint32_t r = threadIdx.x < n_k ? level_runs[k0 + threadIdx.x] : 0u;
                uint32_t tot;
                const uint32_t ex = block_exclusive_scan<kRunThreads>(run_length(r), &tot);
                chosen[threadIdx.x] = run_length(r) != 0u && (carry + ex) / p.run_part == part ? r : 0u;
                carry += tot;
                __syncthreads();
                my_run = chosen[k];
                __syncthreads();  // rewritten by the next tile
            }
            seq.init(run_length(my_run), (k0 + k) * kBucketEntries + run_start(my_run));
            const auto *v = values + (size_t)l * p.n_bchunks * kBucketEntries;
            const uint16_t *r = entry_rows + (size_t)l * p.n_bchunks * kBucketEntries;
            Group cur, next;
            cur.load(seq, 0, v, r);
            for (uint32_t t0 = 0; t0 < seq.total; t0 += kSteps * kWave) {
                next.load(seq, t0 + kSteps * kWave, v, r);
                cur.template add<R>(acc, t0, seq.total);
                cur = next;
            }
        }
    }
    __syncthreads();
    const size_t o = (size_t)s * R * F;
    if (kOut == kAdamRows && n_parts == 1) {
        // unrolled so that several rows' params, m and v loads are in flight at once
#pragma unroll 8
        for (uint32_t t = threadIdx.x; t < rows * F; t += kRunThreads) {
            float mk = adam_m[o + t], vk = adam_v[o + t];
            adam_p[o + t] = adam_step(adam, adam_p[o + t], (float)acc[(t % F) * R + t / F], mk, vk);
            adam_m[o + t] = mk;
            adam_v[o + t] = vk;
        }
        return;
    }
    if (n_parts > 1) {
        double2 *out = reinterpret_cast<double2 *>(partials + (size_t)slot * R * F);
        for (uint32_t t = threadIdx.x; t < R * F / 2; t += kRunThreads) out[t] = reinterpret_cast<const double2 *>(acc)[t];
        return;
    }
    for (uint32_t t = threadIdx.x; t < rows; t += kRunThreads) {
        float *out = static_cast<float *>(dtable) + o;
        if constexpr (kOut == kHalfRows) {
            static_assert(F == 2, "two features, one store");
            reinterpret_cast<__half2 *>(static_cast<__half *>(dtable) + o)[t] =
                __floats2half2_rn((float)acc[t], (float)acc[R + t]);
        } else if constexpr (F == 2) {
            reinterpret_cast<float2 *>(out)[t] = make_float2((float)acc[t], (float)acc[R + t]);
        } else {
            out[t] = (float)acc[t];
        }
    }
}

// The levels that have entries in slice s, in every lane, read from the runs of few items.
__device__ __forceinline__ uint32_t levels_of(const HashGridDescriptor &d, const BwdPlan &p, uint32_t s,
                                              const uint32_t *__restrict__ runs) {
    static_assert(2 * NGP_HASHGRID_MAX_LEVELS == kWave, "two lanes a level");
    const uint32_t l = lane_id() % NGP_HASHGRID_MAX_LEVELS;
    uint32_t any = 0;
    if (l < d.L && s >= p.s_lo[l] && s <= p.s_hi[l]) {
#pragma unroll 4
        for (uint32_t k = lane_id() / NGP_HASHGRID_MAX_LEVELS; k < p.n_bchunks; k += 2)
            any |= run_length(runs[run_index(p, l, s - p.s_lo[l], k)]);
    }
    const uint64_t m = __ballot(any != 0u);
    return (uint32_t)m | (uint32_t)(m >> 32);
}

template <int F, bool kHalf, uint32_t R, int kOut>
__global__ void __launch_bounds__(kRunThreads)
    bwd_reduce_runs_kernel(HashGridDescriptor d, BwdPlan p, const uint32_t *__restrict__ meta,
                           const uint32_t *__restrict__ slice_np, const uint32_t *__restrict__ first_part,
                           const uint32_t *__restrict__ part_slice, const uint32_t *__restrict__ slice_levels,
                           const uint32_t *__restrict__ runs,
                           const EntryValue<F, kHalf> *__restrict__ values, const uint16_t *__restrict__ entry_rows,
                           double *__restrict__ partials, void *__restrict__ dtable, AdamStep adam, float *__restrict__ adam_p,
                           float *__restrict__ adam_m, float *__restrict__ adam_v) {
    uint32_t s = blockIdx.x;
    if (!p.whole) {
        if (blockIdx.x < kSplitBlocks) {
            const uint32_t n = meta[0];
            for (uint32_t i = blockIdx.x; i < n; i += kSplitBlocks) {
                const uint32_t cut = part_slice[i];
                reduce_part<F, kHalf, R, kOut>(d, p, cut, i - first_part[cut], slice_np[cut], i, slice_levels[cut], runs,
                                                values, entry_rows, partials, dtable, adam, adam_p, adam_m, adam_v);
                __syncthreads();  // the sums are read out
            }
            return;
        }
        s -= kSplitBlocks;
        if (slice_np[s] != 1) return;
    }
    const uint32_t levels = __builtin_amdgcn_readfirstlane(p.whole ? levels_of(d, p, s, runs) : slice_levels[s]);
    reduce_part<F, kHalf, R, kOut>(d, p, s, 0, 1, 0, levels, runs, values, entry_rows, partials, dtable, adam, adam_p,
                                    adam_m, adam_v);
}

// One-pass table gradient, part 4: slices of several parts, in pieces of
// 1 / kCombineSplit of a slice's rows.  With kAdam the sums are not stored: the rows take
// the optimizer step in place.
constexpr uint32_t kCombineSplit = 16;
template <int F, uint32_t R, int kOut>
__global__ void __launch_bounds__(256)
    bwd_combine_runs_kernel(HashGridDescriptor d, const uint32_t *__restrict__ meta,
                            const uint32_t *__restrict__ slice_np, const uint32_t *__restrict__ first_part,
                            const uint32_t *__restrict__ split, const double *__restrict__ partials,
                            void *__restrict__ dtable, AdamStep adam, float *__restrict__ adam_p, float *__restrict__ adam_m, float *__restrict__ adam_v) {
    constexpr uint32_t kPer = R * F / kCombineSplit;
    constexpr uint32_t kBatch = 8;  // partial rows in flight per thread
    const uint32_t n_tasks = meta[1] * kCombineSplit;
    for (uint32_t task = blockIdx.x; task < n_tasks; task += gridDim.x) {
        const uint32_t s = split[task / kCombineSplit], piece = task % kCombineSplit;
        const uint32_t p0 = first_part[s], n_parts = slice_np[s];
        const uint32_t rows = min(d.n_rows - s * R, R);
        // feature f of row r is value f * R + r of a part
        for (uint32_t t = piece * kPer + threadIdx.x; t < (piece + 1) * kPer; t += 256) {
            const uint32_t f = t / R, r = t % R;
            if (r >= rows) continue;
            double all = 0.0;
            for (uint32_t q0 = 0; q0 < n_parts; q0 += kBatch) {
                double v[kBatch];
#pragma unroll
                for (uint32_t j = 0; j < kBatch; ++j)
                    v[j] = partials[(size_t)(p0 + min(q0 + j, n_parts - 1u)) * R * F + t];
#pragma unroll
                for (uint32_t j = 0; j < kBatch; ++j)
                    if (q0 + j < n_parts) all += v[j];
            }
            const float sum = (float)all;
            const size_t o = ((size_t)s * R + r) * F + f;
            if constexpr (kOut == kAdamRows) {
                float mk = adam_m[o], vk = adam_v[o];
                adam_p[o] = adam_step(adam, adam_p[o], sum, mk, vk);
                adam_m[o] = mk;
                adam_v[o] = vk;
            } else if constexpr (kOut == kHalfRows) {
                static_cast<__half *>(dtable)[o] = __float2half_rn(sum);
            } else {
                static_cast<float *>(dtable)[o] = sum;
            }
        }
    }
}

// 5. slices of several parts: rows = sum of the parts' partial rows, in part
// order.  Block (s, c) covers 1/kCombineSplit of slice s.
template <int F>
__global__ void __launch_bounds__(256)
    bwd_combine_kernel(HashGridDescriptor d, BwdPlan p, const uint32_t *__restrict__ parts,
                       const float *__restrict__ partials, float *__restrict__ dtable) {
    const uint32_t s = blockIdx.x;
    const uint32_t p0 = parts[s], n_parts = parts[s + 1] - p0;
    if (n_parts <= 1) return;
    const uint32_t n = min(d.n_rows - s * p.R, p.R) * F;  // floats of the slice
    const uint32_t per = (p.R * F) / kCombineSplit;      // a multiple of 4
    const uint32_t lo = blockIdx.y * per, hi = min(n, lo + per);
    const size_t pstride = (size_t)p.R * F;
    const float *src = partials + (size_t)p0 * pstride;
    const size_t o = (size_t)s * p.R * F;
    for (uint32_t t = lo + 4 * threadIdx.x; t < hi; t += 4 * 256) {
        if (t + 4 <= hi) {
            float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            for (uint32_t q = 0; q < n_parts; ++q) {
                const float4 v = *reinterpret_cast<const float4 *>(src + q * pstride + t);
                a.x += v.x;
                a.y += v.y;
                a.z += v.z;
                a.w += v.w;
            }
            *reinterpret_cast<float4 *>(dtable + o + t) = a;
        } else {
            for (uint32_t u = t; u < hi; ++u) {
                float a = 0.0f;
                for (uint32_t q = 0; q < n_parts; ++q) a += src[q * pstride + u];
                dtable[o + u] = a;
            }
        }
    }
}

// The optimizer step of rows no point reached (a zero gradient), for the fused
// update with no points.
__global__ void __launch_bounds__(256)
    adam_zero_grad_kernel(uint64_t n, AdamStep adam, float *__restrict__ adam_p, float *__restrict__ adam_m,
                          float *__restrict__ adam_v) {
    for (uint64_t k = (uint64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (uint64_t)gridDim.x * 256) {
        float mk = adam_m[k], vk = adam_v[k];
        adam_p[k] = adam_step(adam, adam_p[k], 0.0f, mk, vk);
        adam_m[k] = mk;
        adam_v[k] = vk;
    }
}

// `fused` (F <= 2, f32 table, one-pass plan only): the optimizer step in place of
// the gradient's store; dtable is then not written.
struct FusedAdam {
    AdamStep step;
    float *p, *m, *v;
};

template <typename K>
bool reserve_lds(K kernel, size_t lds, const char *target) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess)
        set_error(kLaunchFailed, "%s: cannot reserve %zu bytes of LDS: %s", target, lds, hipGetErrorString(e));
    return e == hipSuccess;
}

// The one-pass form on slices of R rows.
template <int F, bool kHalf, uint32_t R>
bool launch_backward_runs(const HashGridDescriptor &d, const BwdPlan &p, hipStream_t stream, const float *pos,
                          const float *g, void *dtable, uint8_t *ws, const char *target, const FusedAdam *fused,
                          bool half_rows) {
    auto word = [&](uint64_t off) { return reinterpret_cast<uint32_t *>(ws + off); };
    uint32_t *runs = word(p.runs_off), *meta = word(p.meta_off), *slice_np = word(p.slice_np_off);
    uint32_t *first_part = word(p.first_part_off), *split = word(p.split_off), *part_slice = word(p.part_slice_off);
    uint32_t *slice_levels = word(p.levels_off);
    double *partials = reinterpret_cast<double *>(ws + p.partials_off);
    auto *values = reinterpret_cast<EntryValue<F, kHalf> *>(ws + p.entries_off);
    uint16_t *entry_rows = reinterpret_cast<uint16_t *>(ws + p.rows_off);
    const size_t lds = (size_t)R * F * sizeof(double);
    constexpr uint32_t kCombineBlocks = 512;
    HashGridDescriptor db = d;
    if (p.transpose && (reinterpret_cast<uintptr_t>(g) & 7u) == 0) {
        float *lm = reinterpret_cast<float *>(ws + p.partials_off);
        hipLaunchKernelGGL(gradients_to_levels_kernel, dim3(div_up(d.n_points, kTransposePoints)), dim3(kBlock), 0, stream,
                           d.n_points, d.L, (const float2 *)g, (float2 *)lm);
        g = lm;
        db.enc_layout = NGP_ENC_LEVEL_MAJOR;
    }
    hipLaunchKernelGGL((p.wide ? bwd_bucket_kernel<F, kHalf, R, kMaxSlices> : bwd_bucket_kernel<F, kHalf, R, kStageSlices>),
                       dim3(p.n_bitems), dim3(kBucketThreads), 0, stream, db, p, pos, g, runs, values, entry_rows, meta);
    if (!p.whole)
        hipLaunchKernelGGL(bwd_slice_parts_kernel, dim3(p.n_slices), dim3(256), 0, stream, d, p, runs, meta, slice_np,
                           first_part, part_slice, split, slice_levels);
    const dim3 reduce_grid(p.n_slices + (p.whole ? 0 : kSplitBlocks));
    auto finish = [&](auto kind, const AdamStep &step, float *ap, float *am, float *av) {
        constexpr int kOut = decltype(kind)::value;
        const auto reduce = bwd_reduce_runs_kernel<F, kHalf, R, kOut>;
        if (!reserve_lds(reduce, lds, target)) return false;
        hipLaunchKernelGGL(reduce, reduce_grid, dim3(kRunThreads), lds, stream, d, p, meta, slice_np, first_part,
                           part_slice, slice_levels, runs, values, entry_rows, partials, dtable, step, ap, am, av);
        if (!p.whole)
            hipLaunchKernelGGL((bwd_combine_runs_kernel<F, R, kOut>), dim3(kCombineBlocks), dim3(256), 0, stream, d, meta,
                               slice_np, first_part, split, partials, dtable, step, ap, am, av);
        return true;
    };
    if constexpr (!kHalf) {
        if (fused != nullptr)
            return finish(std::integral_constant<int, kAdamRows>{}, fused->step, fused->p, fused->m, fused->v);
    } else if constexpr (F == 2) {
        if (half_rows) return finish(std::integral_constant<int, kHalfRows>{}, AdamStep{}, nullptr, nullptr, nullptr);
    }
    return finish(std::integral_constant<int, kFloatRows>{}, AdamStep{}, nullptr, nullptr, nullptr);
}

template <int F, bool kHalf>
bool launch_backward(const HashGridDescriptor &d, hipStream_t stream, const float *pos, const float *g, void *dtable_,
                     uint8_t *ws, const char *target, const FusedAdam *fused = nullptr, bool half_rows = false) {
    float *dtable = static_cast<float *>(dtable_);
    const BwdPlan p = make_plan(d);
    uint32_t *meta = reinterpret_cast<uint32_t *>(ws + p.meta_off);
    uint32_t *parts = reinterpret_cast<uint32_t *>(ws + p.parts_off);
    uint32_t *part_slice = reinterpret_cast<uint32_t *>(ws + p.part_slice_off);
    float *partials = reinterpret_cast<float *>(ws + p.partials_off);
    uint32_t *entries = reinterpret_cast<uint32_t *>(ws + p.entries_off);
    const size_t lds = (size_t)p.R * F * sizeof(double);
    if constexpr (F <= 2) {
        if (p.bucket) {
            constexpr uint32_t kSmall = kRunSliceBytes / (8 * F), kLarge = kSliceBytes / (8 * F);
            return p.R == kSmall ? launch_backward_runs<F, kHalf, kSmall>(d, p, stream, pos, g, dtable_, ws, target, fused,
                                                                          half_rows)
                                 : launch_backward_runs<F, kHalf, kLarge>(d, p, stream, pos, g, dtable_, ws, target, fused,
                                                                          half_rows);
        }
    }
    if (fused != nullptr) {
        set_error(kBadDescriptor, "%s: the fused update needs the one-pass table gradient", target);
        return false;
    }
    uint32_t *counts = reinterpret_cast<uint32_t *>(ws + p.counts_off);
    uint32_t *sums = reinterpret_cast<uint32_t *>(ws + p.sums_off);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&bwd_reduce_kernel<F, kHalf>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
        set_error(kLaunchFailed, "%s: cannot reserve %zu bytes of LDS: %s", target, lds, hipGetErrorString(e));
        return false;
    }
    hipLaunchKernelGGL(bwd_count_kernel<F>, dim3(p.n_items), dim3(kItemThreads), 0, stream, d, p, pos, counts);
    hipLaunchKernelGGL(scan_sums_kernel, dim3((uint32_t)p.scan_blocks), dim3(kScanThreads), 0, stream, p.M, counts,
                       sums);
    hipLaunchKernelGGL(scan_apply_kernel, dim3((uint32_t)p.scan_blocks), dim3(kScanThreads), 0, stream, p.M, counts,
                       sums, meta);
    hipLaunchKernelGGL(plan_parts_kernel, dim3(1), dim3(kScanThreads), 0, stream, p, counts, meta, parts,
                       part_slice);
    hipLaunchKernelGGL((bwd_scatter_kernel<F, kHalf>), dim3(p.n_items), dim3(kItemThreads), 0, stream, d, p, pos, g,
                       counts, entries);
    hipLaunchKernelGGL((bwd_reduce_kernel<F, kHalf>), dim3(p.max_parts), dim3(kReduceThreads), lds, stream, d, p, counts,
                       meta, parts, part_slice, entries, partials, dtable);
    hipLaunchKernelGGL(bwd_combine_kernel<F>, dim3(p.n_slices, kCombineSplit), dim3(256), 0, stream, d, p, parts,
                       partials, dtable);
    return true;
}

__global__ void zero_table_kernel(float4 *__restrict__ a, size_t n4, float *__restrict__ tail, size_t n_tail) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (size_t j = g; j < n4; j += stride) a[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (g < n_tail) tail[g] = 0.0f;
}

bool validate(const HashGridDescriptor &d, const char *target) {
    if (d.L == 0 || d.L > NGP_HASHGRID_MAX_LEVELS) {
        set_error(kBadDescriptor, "%s: L=%u must be in [1, %d]", target, d.L, NGP_HASHGRID_MAX_LEVELS);
        return false;
    }
    if (!(d.F == 1 || d.F == 2 || d.F == 4 || d.F == 8)) {
        set_error(kBadDescriptor, "%s: F=%u must be 1, 2, 4 or 8", target, d.F);
        return false;
    }
    if (d.T == 0 || d.first_hash_level > d.L || d.n_rows == 0 || d.offsets[0] != 0 || d.offsets[d.L] != d.n_rows ||
        !(d.bound > 0.0f)) {
        set_error(kBadDescriptor, "%s: inconsistent level table (T=%u first_hash_level=%u n_rows=%u bound=%g)", target,
                  d.T, d.first_hash_level, d.n_rows, (double)d.bound);
        return false;
    }
    for (uint32_t l = 0; l < d.L; ++l) {
        if (d.offsets[l + 1] < d.offsets[l]) {
            set_error(kBadDescriptor, "%s: offsets must be non-decreasing", target);
            return false;
        }
    }
    if (d.enc_layout != NGP_ENC_POINT_MAJOR && d.enc_layout != NGP_ENC_LEVEL_MAJOR) {
        set_error(kBadDescriptor, "%s: enc_layout=%u must be 0 (point-major) or 1 (level-major)", target, d.enc_layout);
        return false;
    }
    if (d.table_dtype != NGP_DTYPE_F32 && d.table_dtype != NGP_DTYPE_F16) {
        set_error(kBadDescriptor, "%s: table_dtype=%u must be 0 (f32) or 1 (f16)", target, d.table_dtype);
        return false;
    }
    return true;
}

template <typename TT>
void launch_fwd(const HashGridDescriptor &d, hipStream_t s, const float *pos, const void *table, float *enc) {
    const TT *t = static_cast<const TT *>(table);
    const dim3 b(kBlock);
    // (few points fill the chip with neither, and the other kernel's blocks are shorter)
    const uint64_t level_bytes = (uint64_t)d.T * d.F * sizeof(TT);
    const uint64_t threads = (uint64_t)d.n_points * d.L;
    if (d.enc_layout == NGP_ENC_POINT_MAJOR && level_bytes > 2 * kL2Bytes && (uint64_t)d.n_points * d.F >= 1u << 17 &&
        threads <= 0xffffff00ull) {
        const dim3 g(div_up(threads, kBlock));
        switch (d.F) {
            case 1: hipLaunchKernelGGL((hashgrid_fwd_points_kernel<1, TT>), g, b, 0, s, d, pos, t, enc); break;
            case 2: hipLaunchKernelGGL((hashgrid_fwd_points_kernel<2, TT>), g, b, 0, s, d, pos, t, enc); break;
            case 4: hipLaunchKernelGGL((hashgrid_fwd_points_kernel<4, TT>), g, b, 0, s, d, pos, t, enc); break;
            default: hipLaunchKernelGGL((hashgrid_fwd_points_kernel<8, TT>), g, b, 0, s, d, pos, t, enc); break;
        }
        return;
    }
    // the grouped gather writes a row's two features as one 8-byte vector
    const bool groups = grouped_rows_ok(d, table) && (reinterpret_cast<uintptr_t>(enc) & 7u) == 0;
    const dim3 g(level_grid(d.n_points, d.L));
    switch (d.F) {
        case 1: hipLaunchKernelGGL((hashgrid_fwd_kernel<1, TT, false>), g, b, 0, s, d, pos, t, enc); break;
        case 2:
            if (groups) hipLaunchKernelGGL((hashgrid_fwd_kernel<2, TT, true>), g, b, 0, s, d, pos, t, enc);
            else hipLaunchKernelGGL((hashgrid_fwd_kernel<2, TT, false>), g, b, 0, s, d, pos, t, enc);
            break;
        case 4: hipLaunchKernelGGL((hashgrid_fwd_kernel<4, TT, false>), g, b, 0, s, d, pos, t, enc); break;
        default: hipLaunchKernelGGL((hashgrid_fwd_kernel<8, TT, false>), g, b, 0, s, d, pos, t, enc); break;
    }
}

}  // namespace
}  // namespace ngp

using namespace ngp;

extern "C" void hashgrid_encode(ngp_stream_t stream_, void **buffers, const char *opaque, size_t opaque_len) {
    const char *target = "hashgrid_encode";
    HashGridDescriptor d;
    if (!read_descriptor(opaque, opaque_len, &d, target)) return;
    if (!validate(d, target)) return;
    if (d.n_points == 0) return;
    if (!check_buffers(buffers, 3, target)) return;
    hipStream_t stream = (hipStream_t)stream_;
    const float *pos = (const float *)buffers[0];
    float *enc = (float *)buffers[2];
    if (d.table_dtype == NGP_DTYPE_F32) launch_fwd<float>(d, stream, pos, buffers[1], enc);
    else launch_fwd<__half>(d, stream, pos, buffers[1], enc);
    check_launch(target);
}

extern "C" void hashgrid_encode_staged(ngp_stream_t stream_, void **buffers, const char *opaque, size_t opaque_len) {
    const char *target = "hashgrid_encode_staged";
    HashGridDescriptor d;
    if (!read_descriptor(opaque, opaque_len, &d, target)) return;
    if (!validate(d, target)) return;
    if (!(d.F == 2 || d.F == 4) || d.enc_layout != NGP_ENC_POINT_MAJOR) {
        set_error(kBadDescriptor, "%s: F must be 2 or 4 and enc_layout 0 (point-major)", target);
        return;
    }
    if (d.n_points == 0) return;
    if (!check_buffers(buffers, 4, target)) return;
    if (((reinterpret_cast<uintptr_t>(buffers[2]) | reinterpret_cast<uintptr_t>(buffers[3])) & (4 * d.F - 1u)) != 0) {
        set_error(kBadArgument, "%s: encodings and the workspace must be %u-byte aligned", target, 4 * d.F);
        return;
    }
    hipStream_t stream = (hipStream_t)stream_;
    const float *pos = (const float *)buffers[0];
    float *lm = (float *)buffers[3];
    HashGridDescriptor dl = d;
    dl.enc_layout = NGP_ENC_LEVEL_MAJOR;
    // pieces, so that the workspace does not grow with the points past 256 MiB (L = 16, F = 2)
    for (uint32_t n0 = 0; n0 < d.n_points;) {
        dl.n_points = std::min(d.n_points - n0, NGP_ENCODE_STAGE_POINTS);
        const float *p = pos + 3 * (size_t)n0;
        float *out = (float *)buffers[2] + (size_t)n0 * d.L * d.F;
        if (d.table_dtype == NGP_DTYPE_F32) launch_fwd<float>(dl, stream, p, buffers[1], lm);
        else launch_fwd<__half>(dl, stream, p, buffers[1], lm);
        if (!check_launch(target)) return;
        const dim3 g(div_up(dl.n_points, kTransposePoints)), b(kBlock);
        if (d.F == 2)
            hipLaunchKernelGGL(encodings_to_points_kernel<float2>, g, b, 0, stream, dl.n_points, d.L, (const float2 *)lm,
                               (float2 *)out);
        else
            hipLaunchKernelGGL(encodings_to_points_kernel<float4>, g, b, 0, stream, dl.n_points, d.L, (const float4 *)lm,
                               (float4 *)out);
        if (!check_launch(target)) return;
        n0 += dl.n_points;
    }
}

extern "C" int hashgrid_encode_backward_adam_supported(const char *opaque, size_t opaque_len) {
    const char *target = "hashgrid_encode_backward_adam_supported";
    HashGridDescriptor d;
    if (!read_descriptor(opaque, opaque_len, &d, target)) return 0;
    if (!validate(d, target)) return 0;
    return d.F <= 2 && d.table_dtype == NGP_DTYPE_F32 && make_plan(d).bucket ? 1 : 0;
}

extern "C" void hashgrid_encode_backward_adam(ngp_stream_t stream_, void **buffers, const char *opaque,
                                              size_t opaque_len) {
    const char *target = "hashgrid_encode_backward_adam";
    static_assert(offsetof(HashGridAdamDescriptor, adam) == sizeof(HashGridDescriptor), "no padding");
    HashGridAdamDescriptor q;
    if (!read_descriptor(opaque, opaque_len, &q, target)) return;
    const HashGridDescriptor &d = q.grid;
    if (!validate(d, target)) return;
    if (d.F > 2 || d.table_dtype != NGP_DTYPE_F32 || q.adam.flags != 0u || q.adam.mirror_dtype != NGP_DTYPE_F32 ||
        q.adam.n != (uint64_t)d.n_rows * d.F) {
        set_error(kBadDescriptor,
                  "%s: needs F <= 2, an f32 table, no loss scaling or f16 mirror, and adam.n = n_rows * F", target);
        return;
    }
    const BwdPlan plan = make_plan(d);
    if (!plan.bucket || plan.n_slices > kMaxSlices) {
        set_error(kBadDescriptor, "%s: the table's levels must fit the one-pass table gradient", target);
        return;
    }
    if ((uint64_t)d.n_points * d.L * 8 >= 0xffffffffull) {
        set_error(kBadDescriptor, "%s: n_points * L * 8 must stay below 2^32", target);
        return;
    }
    if (!check_buffer_list(buffers, {2, 3, 4}, target)) return;
    hipStream_t stream = (hipStream_t)stream_;
    FusedAdam f{make_adam_step(q.adam), (float *)buffers[2], (float *)buffers[3], (float *)buffers[4]};
    if (d.n_points == 0) {
        const uint64_t n = q.adam.n;
        const uint32_t grid = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((n + 255) / 256, 16384));
        hipLaunchKernelGGL(adam_zero_grad_kernel, dim3(grid), dim3(256), 0, stream, n, f.step, f.p, f.m, f.v);
        check_launch(target);
        return;
    }
    if (!check_buffers(buffers, 6, target)) return;
    uint8_t *ws = (uint8_t *)buffers[5];
    if ((reinterpret_cast<uintptr_t>(ws) & 255u) != 0 ||
        ((reinterpret_cast<uintptr_t>(f.p) | reinterpret_cast<uintptr_t>(f.m) | reinterpret_cast<uintptr_t>(f.v)) &
         15u) != 0) {
        set_error(kBadArgument, "%s: params, m and v must be 16-byte and the workspace 256-byte aligned", target);
        return;
    }
    const float *pos = (const float *)buffers[0];
    const float *g = (const float *)buffers[1];
    const bool ok = d.F == 1 ? launch_backward<1, false>(d, stream, pos, g, nullptr, ws, target, &f)
                             : launch_backward<2, false>(d, stream, pos, g, nullptr, ws, target, &f);
    if (!ok) return;
    check_launch(target);
}

extern "C" size_t hashgrid_encode_backward_workspace_size(const char *opaque, size_t opaque_len) {
    HashGridDescriptor d;
    if (!read_descriptor(opaque, opaque_len, &d, "hashgrid_encode_backward_workspace_size")) return 0;
    if (!validate(d, "hashgrid_encode_backward_workspace_size")) return 0;
    return (size_t)make_plan(d).bytes;
}

static bool half_rows_ok(const HashGridDescriptor &d, const BwdPlan &p) {
    return d.F == 2 && d.table_dtype == NGP_DTYPE_F16 && p.bucket;
}

extern "C" int hashgrid_encode_backward_f16_supported(const char *opaque, size_t opaque_len) {
    HashGridDescriptor d;
    if (!read_descriptor(opaque, opaque_len, &d, "hashgrid_encode_backward_f16_supported")) return 0;
    if (!validate(d, "hashgrid_encode_backward_f16_supported")) return 0;
    return half_rows_ok(d, make_plan(d)) ? 1 : 0;
}

// Both table gradients: rows in f32, or (half_rows) in f16.
static void encode_backward(ngp_stream_t stream_, void **buffers, const char *opaque, size_t opaque_len,
                            const char *target, bool half_rows) {
    HashGridDescriptor d;
    if (!read_descriptor(opaque, opaque_len, &d, target)) return;
    if (!validate(d, target)) return;
    const BwdPlan plan = make_plan(d);
    if (half_rows && !half_rows_ok(d, plan)) {
        set_error(kBadDescriptor, "%s: needs F = 2, an f16 table and the one-pass table gradient", target);
        return;
    }
    if (plan.n_slices > kMaxSlices) {
        set_error(kBadDescriptor, "%s: table of %u rows exceeds %u row slices", target, d.n_rows, kMaxSlices);
        return;
    }
    if ((uint64_t)d.n_points * d.L * 8 >= 0xffffffffull) {
        set_error(kBadDescriptor, "%s: n_points * L * 8 must stay below 2^32", target);
        return;
    }
    if (!check_buffer_list(buffers, {2}, target)) return;
    if (d.n_points > 0 && !check_buffers(buffers, 4, target)) return;
    hipStream_t stream = (hipStream_t)stream_;
    const float *pos = (const float *)buffers[0];
    const float *g = (const float *)buffers[1];
    float *dtable = (float *)buffers[2];
    if (d.n_points == 0) {
        // no contributions: the gradient is zero
        const size_t n = (size_t)d.n_rows * d.F / (half_rows ? 2 : 1);  // in floats
        const bool vec = (reinterpret_cast<uintptr_t>(dtable) & 15u) == 0;
        const size_t n4 = vec ? n / 4 : 0;
        const size_t n_tail = n - 4 * n4;
        const uint32_t zgrid =
            (uint32_t)std::max<size_t>(1, std::min<size_t>((std::max(n4, n_tail) + 255) / 256, 16384));
        hipLaunchKernelGGL(zero_table_kernel, dim3(zgrid), dim3(256), 0, stream, reinterpret_cast<float4 *>(dtable),
                           n4, dtable + 4 * n4, n_tail);
        check_launch(target);
        return;
    }
    uint8_t *ws = (uint8_t *)buffers[3];
    if ((reinterpret_cast<uintptr_t>(ws) & 255u) != 0 || (reinterpret_cast<uintptr_t>(dtable) & 15u) != 0) {
        set_error(kBadArgument, "%s: dL_dtable must be 16-byte and the workspace 256-byte aligned", target);
        return;
    }
    bool ok = false;
    const bool half = d.table_dtype == NGP_DTYPE_F16;
    switch (d.F) {
        case 1: ok = launch_backward<1, false>(d, stream, pos, g, dtable, ws, target); break;
        case 2:
            ok = half ? launch_backward<2, true>(d, stream, pos, g, dtable, ws, target, nullptr, half_rows)
                      : launch_backward<2, false>(d, stream, pos, g, dtable, ws, target);
            break;
        case 4:
            ok = half ? launch_backward<4, true>(d, stream, pos, g, dtable, ws, target)
                      : launch_backward<4, false>(d, stream, pos, g, dtable, ws, target);
            break;
        default: ok = launch_backward<8, false>(d, stream, pos, g, dtable, ws, target); break;
    }
    if (!ok) return;
    check_launch(target);
}

extern "C" void hashgrid_encode_backward(ngp_stream_t stream, void **buffers, const char *opaque, size_t opaque_len) {
    encode_backward(stream, buffers, opaque, opaque_len, "hashgrid_encode_backward", false);
}

extern "C" void hashgrid_encode_backward_f16(ngp_stream_t stream, void **buffers, const char *opaque,
                                             size_t opaque_len) {
    encode_backward(stream, buffers, opaque, opaque_len, "hashgrid_encode_backward_f16", true);
}
