// hashgrid_device.h — per-level vertex rows and weights of the hash encoding
// (models/encoders.py:116-213), shared by the encoder kernels and the fused
// inference field kernel.
#pragma once

#include <hip/hip_fp16.h>

#include <type_traits>

#include "ngp_common.h"

namespace ngp {

struct LevelTables {
    float scale[NGP_HASHGRID_MAX_LEVELS];
    uint32_t res[NGP_HASHGRID_MAX_LEVELS];
    uint32_t offset[NGP_HASHGRID_MAX_LEVELS];
};

template <typename TT>
__device__ __forceinline__ float to_f32(TT v);
template <>
__device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ float to_f32<__half>(__half v) { return __half2float(v); }
template <>
__device__ __forceinline__ float to_f32<_Float16>(_Float16 v) { return (float)v; }

// A level's index rule, as a compile-time choice where it is the same for the whole
// wavefront: one branch around the eight corners instead of several in each.
enum LevelRule { kDenseRule, kHashRule, kLaneRule };

// (px, py, pz) normalised to [0, 1]: the divisor's kind is tested once for all three.
__device__ __forceinline__ void normalise(const Divisor &two_b, float bound, const float pos[3], float p[3]) {
    const float x = pos[0] + bound, y = pos[1] + bound, z = pos[2] + bound;
    if (two_b.pow2) {
        p[0] = x * two_b.inv;
        p[1] = y * two_b.inv;
        p[2] = z * two_b.inv;
    } else {
        p[0] = x / two_b.d;
        p[1] = y / two_b.d;
        p[2] = z / two_b.d;
    }
}

// Vertex rows and weights of point (px,py,pz) (already normalised to [0,1]) at one
// level.  kLaneRule: `dense` differs between lanes.  Row order: x is the slowest corner
// bit, so corners c and 4 + c are the two ends of an edge along x.
template <LevelRule kRule, bool kPow2>
__device__ __forceinline__ void level_vertices_t(float px, float py, float pz, float scale, uint32_t res, bool dense,
                                                 uint32_t T, uint32_t offset, uint32_t last_row, uint32_t idx[8],
                                                 float w[8]) {
    const float sx = px * scale + 0.5f, sy = py * scale + 0.5f, sz = pz * scale + 0.5f;
    const float fx = floorf(sx), fy = floorf(sy), fz = floorf(sz);
    const float rx = sx - fx, ry = sy - fy, rz = sz - fz;
    const bool d = kRule == kDenseRule || (kRule == kLaneRule && dense);
    const uint32_t my = d ? res : 2654435761u, mz = d ? res * res : 805459861u;
    const uint32_t x[2] = {(uint32_t)fx, (uint32_t)(fx + 1.0f)};
    const uint32_t y[2] = {(uint32_t)fy * my, (uint32_t)(fy + 1.0f) * my};
    const uint32_t z[2] = {(uint32_t)fz * mz, (uint32_t)(fz + 1.0f) * mz};
    const float wx[2] = {1.0f - rx, rx}, wy[2] = {1.0f - ry, ry}, wz[2] = {1.0f - rz, rz};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int ox = (c >> 2) & 1, oy = (c >> 1) & 1, oz = c & 1;
        const uint32_t hd = x[ox] + y[oy] + z[oz], hh = x[ox] ^ y[oy] ^ z[oz];
        const uint32_t h = kRule == kDenseRule ? hd : (kRule == kHashRule ? hh : (dense ? hd : hh));
        const uint32_t r = (kPow2 ? (h & (T - 1u)) : (h % T)) + offset;
        idx[c] = r > last_row ? last_row : r;
        w[c] = (wx[ox] * wy[oy]) * wz[oz];
    }
}

// The same where nothing is known at compile time.
__device__ __forceinline__ void level_vertices(float px, float py, float pz, float scale, uint32_t res, bool dense,
                                               uint32_t T, bool pow2, uint32_t offset, uint32_t last_row,
                                               uint32_t idx[8], float w[8]) {
    if (pow2) level_vertices_t<kLaneRule, true>(px, py, pz, scale, res, dense, T, offset, last_row, idx, w);
    else level_vertices_t<kLaneRule, false>(px, py, pz, scale, res, dense, T, offset, last_row, idx, w);
}

// Calls f(rule, pow2) with both as std::integral_constants, for a level that is the
// same for the whole wavefront.
template <typename Fn>
__device__ __forceinline__ void with_rule(bool dense, bool pow2, Fn f) {
    if (!pow2) f(std::integral_constant<LevelRule, kLaneRule>{}, std::false_type{});
    else if (dense) f(std::integral_constant<LevelRule, kDenseRule>{}, std::true_type{});
    else f(std::integral_constant<LevelRule, kHashRule>{}, std::true_type{});
}

// Rows of two features gathered by aligned groups.  The two corners of a cell edge
// along x are rows h and h + 1 (dense) or x0 ^ h and x1 ^ h (hashed): where x0 is not
// the last of its aligned group of kRows rows, both lie in one 16-byte group, so one
// load brings both.  The gathers are bound by the number of lane addresses the vector
// memory unit takes (one lookup per lane and load), not by bytes: an f32 table then
// needs 4 + 4/2 lookups a point and level instead of 8, an f16 table 4 + 4/4.  Needs
// a 16-byte aligned table of a whole number of groups under 4 GiB (see
// grouped_rows_ok), so that a group never reaches past the table and row addresses
// are 32-bit offsets from its base.
template <typename TT>
struct RowGroup;

template <>
struct RowGroup<float> {
    typedef float4 Vec;
    typedef float2 Row;
    static constexpr uint32_t kRows = 2;
    static __device__ __forceinline__ Row pick(const Vec &v, uint32_t i) {
        Row r;  // value by value: a select of whole structs would go through memory
        r.x = (i & 1u) ? v.z : v.x;
        r.y = (i & 1u) ? v.w : v.y;
        return r;
    }
    static __device__ __forceinline__ Row select(bool first, Row a, Row b) {
        Row r;
        r.x = first ? a.x : b.x;
        r.y = first ? a.y : b.y;
        return r;
    }
    static __device__ __forceinline__ float2 f32(Row r) { return r; }
    static __device__ __forceinline__ Vec load_group(__amdgpu_buffer_rsrc_t t, uint32_t off) {
        return __builtin_bit_cast(Vec, __builtin_amdgcn_raw_buffer_load_b128(t, off, 0, 0));
    }
    static __device__ __forceinline__ Row load_row(__amdgpu_buffer_rsrc_t t, uint32_t off) {
        return __builtin_bit_cast(Row, __builtin_amdgcn_raw_buffer_load_b64(t, off, 0, 0));
    }
};

template <>
struct RowGroup<__half> {
    typedef uint4 Vec;
    typedef uint32_t Row;
    static constexpr uint32_t kRows = 4;
    static __device__ __forceinline__ Row pick(const Vec &v, uint32_t i) {
        const uint32_t a = (i & 1u) ? v.y : v.x, b = (i & 1u) ? v.w : v.z;
        return (i & 2u) ? b : a;
    }
    static __device__ __forceinline__ Row select(bool first, Row a, Row b) { return first ? a : b; }
    static __device__ __forceinline__ float2 f32(Row r) {
        return __half22float2(__builtin_bit_cast(__half2, r));
    }
    static __device__ __forceinline__ Vec load_group(__amdgpu_buffer_rsrc_t t, uint32_t off) {
        return __builtin_bit_cast(Vec, __builtin_amdgcn_raw_buffer_load_b128(t, off, 0, 0));
    }
    static __device__ __forceinline__ Row load_row(__amdgpu_buffer_rsrc_t t, uint32_t off) {
        return __builtin_amdgcn_raw_buffer_load_b32(t, off, 0, 0);
    }
};

template <>
struct RowGroup<_Float16> : RowGroup<__half> {};

// A byte offset past every table the grouped gather takes.
constexpr uint32_t kPastTable = 0xfffffff0u;

// The table as a bounds-checked buffer of its own size.
template <typename TT>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t table_buffer(const HashGridDescriptor &d, const TT *table) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<TT *>(table), 0,
                                             (int)(d.n_rows * (uint32_t)sizeof(typename RowGroup<TT>::Row)), 0x00020000);
}

inline bool grouped_rows_ok(const HashGridDescriptor &d, const void *table) {
    const bool half = d.table_dtype == NGP_DTYPE_F16;
    const uint64_t row_bytes = half ? 4 : 8;
    const uint32_t rows = half ? RowGroup<__half>::kRows : RowGroup<float>::kRows;
    return d.F == 2 && (reinterpret_cast<uintptr_t>(table) & 15u) == 0 && d.n_rows % rows == 0 &&
           d.n_rows * row_bytes <= kPastTable;
}

// The loads of one point at one level, issued before any is used (several points'
// loads can be in flight together), and the weighted sum in corner order, the same
// operations as a gather row by row.  The second load of an edge is a buffer load
// whose offset lies past the table in the lanes that do not need it: those lanes read
// zero without a memory access, and there is no branch between the two loads of an
// edge, which mostly share a cache line (issued later, the line was fetched twice:
// 193 us instead of 70 for 2^18 points of an f32 table).
template <typename TT>
struct GroupedGather {
    typedef RowGroup<TT> RG;
    typename RG::Vec near[4];
    typename RG::Row far[4];

    static __device__ __forceinline__ bool apart(const uint32_t idx[8], int q) {
        return idx[q] / RG::kRows != idx[4 + q] / RG::kRows;
    }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t table, const uint32_t idx[8]) {
        constexpr uint32_t kRow = sizeof(typename RG::Row);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            near[q] = RG::load_group(table, (idx[q] / RG::kRows) * (kRow * RG::kRows));
            far[q] = RG::load_row(table, apart(idx, q) ? idx[4 + q] * kRow : kPastTable);
        }
    }
    __device__ __forceinline__ float2 sum(const uint32_t idx[8], const float w[8]) const {
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int q = c & 3;
            typename RG::Row r = RG::pick(near[q], idx[c]);
            if (c >= 4) r = RG::select(apart(idx, q), far[q], r);
            const float2 v = RG::f32(r);
            a0 = a0 + v.x * w[c];
            a1 = a1 + v.y * w[c];
        }
        return make_float2(a0, a1);
    }
};

}  // namespace ngp
