// march.hip — occupancy-grid ray marching for training and inference.
//
// march_rays:            deps/volume-rendering-jax/lib/impl/marching.cu:101-268 (kernel), 435-522 (launcher)
// march_rays_inference:  marching.cu:271-397 (kernel), 524-604 (launcher)
//
// Training marcher.  The reference reserves each ray's output range with an
// atomicAdd in scheduling order and marches every ray twice.  Here the ranges are
// an exclusive prefix sum of the per-ray counts in ray order, which makes the
// output deterministic and equal to processing rays one after another:
//   1. march_begin:  marks every ray's count and start as "past the filled buffer";
//   2. march_count:  workgroups take blocks of rays in rounds, count their samples and add
//                    them to the round's counter.  A workgroup that finds the earlier
//                    rounds' counters at total_samples stops: all of them are of earlier
//                    rays, so the rays left are invalid whatever their counts and keep their
//                    marks.  Each ray leaves a record of its samples (see RayRecord) in
//                    the xyzs output, which nothing has written yet;
//   3. march_scan:   one workgroup scans the counts, finds the ray where the sample buffer
//                    fills up and writes the two helper counters;
//   4. march_emit:   one wavefront per valid ray writes its samples' t to z_vals at its
//                    offset: from its record, or marched again where it has none;
//   5. march_fill:   one wavefront per valid ray writes the outputs that follow from
//                    t (index, position, direction, step size);
//   6. march_finish: validity, final counts and offsets, zeros in the unused tail.
// A ray is valid iff the samples of the rays before it leave room (prefix <
// total_samples), t_end > t_start, and its own samples fit; rays after the buffer
// fills are invalid, as the reference's early exit at marching.cu:135 makes them.
//
// Wavefront marching.  Every t the reference's loop visits (marching.cu:162-192)
// lies on the sequence c_0 = t_start, c_{k+1} = c_k + step_size(c_k): an occupied
// step moves to the next element, an empty-cell skip to the first later element
// at or past the cell's exit.  So a wavefront generates 64 consecutive elements
// (one per lane), looks up all 64 cells and exit distances at once, and walks the
// visited elements with ballots: runs of occupied lanes are emitted together, a skip is
// a search for the first lane past the exit.
// Samples go to their slots by lane prefix counts.  The walk visits exactly the
// reference's t values in its order; where the chain stops growing (t + ds == t)
// the ray finishes on one lane with the serial loop, which handles that case.
#include "ngp_common.h"
#include "ngp_device.h"

namespace ngp {
namespace {

constexpr int kBlock = 256;
constexpr int kRaysPerBlock = kBlock / kWave;  // one wavefront per ray
constexpr int kScanThreads = 1024;
// count of a ray that was not marched: the sample buffer was already full
constexpr uint32_t kPastFill = 0xffffffffu;

struct Ray {
    float ox, oy, oz, dx, dy, dz, idx, idy, idz, t1;
};

__device__ __forceinline__ Ray load_ray(const float *__restrict__ rays_o, const float *__restrict__ rays_d, uint32_t i,
                                        float t1) {
    Ray r;
    r.ox = rays_o[3 * (size_t)i];
    r.oy = rays_o[3 * (size_t)i + 1];
    r.oz = rays_o[3 * (size_t)i + 2];
    r.dx = rays_d[3 * (size_t)i];
    r.dy = rays_d[3 * (size_t)i + 1];
    r.dz = rays_d[3 * (size_t)i + 2];
    r.idx = 1.0f / r.dx;
    r.idy = 1.0f / r.dy;
    r.idz = 1.0f / r.dz;
    r.t1 = t1;
    return r;
}

// Where a marching wavefront writes its samples: the t of sample k goes to ts[k]
// (the other outputs follow from t, see march_fill_kernel).
struct RaySamples {
    float *ts;
};

// A ray's record: for every window of 64 chain elements (see Window) that holds samples,
// the window's first element and the mask of the elements that are samples, three words;
// word 0 holds the number of windows, or kNoRecord for a ray with more than the record
// takes or one that left the windows.  52 words a ray at bound 1 instead of its up to
// 1,024 t values, at a place that does not depend on its count, and no LDS: the marcher
// runs beside the MLP backward, whose two workgroups take a CU's whole LDS.
struct RayRecord {
    uint32_t *words;  // null: none is kept
    uint32_t max_windows;
};
constexpr uint32_t kNoRecord = 0xffffffffu;

// The reference's loop (marching.cu:162-192) from position t with n samples taken,
// on one lane.
template <bool kWrite>
__device__ uint32_t march_serial(const MarchParams &p, const uint8_t *__restrict__ bits, BitCache &cache, const Ray &r,
                                 float t, uint32_t n, uint32_t cap, const RaySamples &o) {
    while (n < cap && t < r.t1) {
        const float px = r.ox + t * r.dx, py = r.oy + t * r.dy, pz = r.oz + t * r.dz;
        const float ds = step_size(p, t);
        float gx, gy, gz, mb;
        if (lookup_cell(p, bits, cache, px, py, pz, ds, gx, gy, gz, mb)) {
            if (kWrite) o.ts[n] = t;
            ++n;
            t = t + ds;
        } else {
            const float next_t = cell_exit_t(p, t, px, py, pz, gx, gy, gz, mb, r.dx, r.dy, r.dz, r.idx, r.idy, r.idz);
            t = skip_to(p, t, ds, next_t);
        }
    }
    return n;
}

// 64 consecutive elements of the chain c_0 = base, c_{j+1} = c_j + step_size(c_j), one
// per lane, with what the walk needs of each.
struct Window {
    float w;        // c_lane
    float exit;     // exit distance of its cell
    uint64_t word;  // the occupancy word (or byte) of its cell
    uint32_t bit;   // its bit there
    uint32_t cell;  // its index
    bool live;      // w < t_end
    bool clear;     // kOne: no plane of the grid within the rounding error (see march_ray_wave)
    // the same in all lanes
    float base, next;  // c_0, c_64
    bool stall;        // the chain stops growing
};

// Lane j's element of the chain c_0 = base, c_{j+1} = c_j + k (k > 0 constant).
// While the chain stays in base's binade, where every float is a multiple of the
// ulp u, each step adds the same m = k rounded to a multiple of u, so
// c_j = base + (j*m)*u with exact arithmetic.  Every lane then checks the
// recurrence c_{j+1} == c_j + k against its neighbour; the values are used only
// if all checks pass (by induction they are the chain), which fails where the
// chain leaves the binade, at rounding ties and for non-positive or non-normal
// base.  On success also returns c_64 in `next`; a chain that stops growing
// (next == c_63) is left to the serial generation, which detects it.
__device__ __forceinline__ bool chain_in_binade(float base, float k, int lane, float &w, float &next) {
    const uint32_t e8 = __float_as_uint(base) >> 23;  // sign bit included: negative base fails
    if (e8 < 24u || e8 >= 255u) return false;
    const float u = __uint_as_float((e8 - 23u) << 23);
    // k / u is a scaling by a power of two: exact, also as a product with 1 / u (normal
    // for the exponents that pass the test above and leave m in range)
    const float m = e8 <= 253u ? rintf(k * __uint_as_float((277u - e8) << 23)) : 0.0f;
    if (!(m >= 1.0f && m <= 65536.0f)) return false;
    const float x = base + ((float)lane * m) * u;
    const float nx = x + k;
    const float up = __shfl_down(x, 1, kWave);
    const bool ok = lane == kWave - 1 || (up == nx && up != x);
    if (__ballot(!ok) != 0ull) return false;
    const float n63 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(nx), kWave - 1));
    const float x63 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), kWave - 1));
    if (n63 == x63) return false;
    w = x;
    next = n63;
    return true;
}

// The 64 elements from `base` on: lane j's in w, c_64 in next; `stall` where the chain
// stops growing.
__device__ __forceinline__ void chain_window(const MarchParams &p, bool const_step, float k_step, float base, float &w,
                                             float &next, bool &stall) {
    const int lane = lane_id();
    stall = false;
    if (const_step && chain_in_binade(base, k_step, lane, w, next)) return;
    float c = base;
    w = base;
    bool stops = false;
#pragma unroll 4
    for (int q = 0; q < kWave; ++q) {
        if (lane == q) w = c;
        const float nx = c + (const_step ? k_step : step_size(p, c));
        stops |= nx == c;
        c = nx;
    }
    next = c;
    stall = __ballot(stops) != 0ull;
}

// The window starting at `base`, its occupancy load issued.  Call with all lanes active.
template <bool kOne>
__device__ __forceinline__ Window make_window(const MarchParams &p, const uint8_t *__restrict__ bits, bool word_ok,
                                              const Ray &r, bool const_step, float k_step, float margin, float base) {
    Window v;
    v.base = base;
    chain_window(p, const_step, k_step, base, v.w, v.next, v.stall);
    v.live = v.w < r.t1;
    const float px = r.ox + v.w * r.dx, py = r.oy + v.w * r.dy, pz = r.oz + v.w * r.dz;
    float gx, gy, gz, mb;
    const uint32_t idx = cell_index<kOne>(p, px, py, pz, step_size(p, v.w), gx, gy, gz, mb);
    v.cell = idx;
    v.clear = kOne && fmaxf(fabsf(gx - floorf(gx) - 0.5f), fmaxf(fabsf(gy - floorf(gy) - 0.5f),
                                                                 fabsf(gz - floorf(gz) - 0.5f))) <= 0.5f - margin;
    v.word = 0ull;
    if (word_ok) {
        v.bit = idx & 63u;
        if (v.live) v.word = reinterpret_cast<const uint64_t *>(bits)[idx >> 6];
    } else {
        v.bit = idx & 7u;
        if (v.live) v.word = bits[idx >> 3];
    }
    v.exit = cell_exit_t(p, v.w, px, py, pz, gx, gy, gz, mb, r.dx, r.dy, r.dz, r.idx, r.idy, r.idz);
    return v;
}

__device__ __forceinline__ float lane_float(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Counts the samples of one ray with the whole wavefront, starting at t_start,
// taking at most cap samples (kWrite: also writes their t; with a record: also keeps
// it).  Call with all 64 lanes active.  The next window is made, its occupancy load in flight, before this
// one is walked.
// kOne (a grid of one cascade): the walk crosses a stretch of empty cells at once instead of
// cell by cell.  Every visited element of a cell has the same exit but for rounding, and the
// next visited one is the first past it: the first element of the next cell, unless an
// element lies within the rounding error of a plane between cells, on either side or as a
// cell's index and exit see it.  So if no element of the window does (`clear`; nine windows
// in ten), the walk takes the first element of the last empty cell before the next
// occupied one, and its exit.
template <bool kWrite, bool kOne>
__device__ uint32_t march_ray_wave(const MarchParams &p, const uint8_t *__restrict__ bits, bool word_ok, const Ray &r,
                                   float t_start, uint32_t cap, const RaySamples &o, const RayRecord &rec) {
    const int lane = lane_id();
    uint32_t windows = 0;  // in the record
    const uint64_t below = (1ull << lane) - 1ull;
    // with stepsize_portion 0 every step is the same constant, for every t
    const bool const_step = p.portion == 0.0f;
    const float k_step = step_size(p, 0.0f);
    uint32_t n = 0;
    bool pending = false;  // a skip is searching for the first element >= thr
    float thr = 0.0f;
    if (cap == 0) {
        if (rec.words != nullptr && lane == 0) rec.words[0] = 0u;
        return 0;
    }
    // A position carries up to 2^-24 (|o| + t|d| + 1) on an axis, an exit distance that, its
    // own roundings of as much and the position's again, over |d|: less than 2^-21 of the sum
    // in all, here in cells.
    const float reach = fmaxf(fabsf(r.ox) + fabsf(r.t1 * r.dx),
                              fmaxf(fabsf(r.oy) + fabsf(r.t1 * r.dy), fabsf(r.oz) + fabsf(r.t1 * r.dz)));
    const float margin = 4.7683716e-7f * (reach + 2.0f) * (0.5f * (float)p.G) / fminf(1.0f, p.bound);
    Window v = make_window<kOne>(p, bits, word_ok, r, const_step, k_step, margin, t_start);
    for (;;) {
        if (v.stall) {
            // the chain stops growing at or after `base`: the serial loop on one lane
            uint32_t nn = n;
            if (lane == 0) {
                BitCache cache = make_bit_cache(bits, word_ok);
                float t = v.base;
                if (pending) {
                    // rest of skip_to: t is the first step past the skipped element
                    while (t < thr) {
                        const float s2 = t + step_size(p, t);
                        if (s2 == t) {
                            t = __builtin_huge_valf();
                            break;
                        }
                        t = s2;
                    }
                }
                nn = march_serial<kWrite>(p, bits, cache, r, t, n, cap, o);
                if (rec.words != nullptr) rec.words[0] = kNoRecord;
            }
            return (uint32_t)__builtin_amdgcn_readlane((int)nn, 0);
        }
        const uint64_t live_m = __ballot(v.live);
        const bool last = (live_m >> (kWave - 1)) == 0ull;  // the chain reaches t_end here
        Window next;
        if (!last) next = make_window<kOne>(p, bits, word_ok, r, const_step, k_step, margin, v.next);
        const uint64_t occ_m = __ballot(v.live && ((v.word >> v.bit) & 1ull));
        const uint32_t n0 = n;
        uint64_t emit = 0ull, starts = 0ull;  // first elements of cells
        bool clear = false;
        if constexpr (kOne) {
            constexpr int kWaveShr1 = 0x138;
            const uint32_t before =
                (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v.cell, kWaveShr1, 0xf, 0xf, false);
            starts = __ballot(v.cell != before);
            clear = __ballot(v.live && !v.clear) == 0ull;
        }
        int cur = 0;
        while (cur < kWave) {
            if (pending) {
                // skip_to stops at the first element with !(t < thr)
                const uint64_t m = __ballot(!(v.w < thr)) & (~0ull << cur);
                if (m == 0ull) break;  // the target lies past this window
                cur = __builtin_ctzll(m);
                pending = false;
            }
            if (((live_m >> cur) & 1ull) == 0ull) break;  // at or past t_end: `last` holds
            if ((occ_m >> cur) & 1ull) {
                const uint64_t from = occ_m >> cur;
                const int run = ~from == 0ull ? kWave - cur : __builtin_ctzll(~from);
                const uint32_t take = min((uint32_t)run, cap - n);
                emit |= (take >= 64u ? ~0ull : ((1ull << take) - 1ull)) << cur;
                n += take;
                if (n >= cap) break;
                cur += run;
            } else {
                if (kOne && clear) {
                    const uint64_t ahead = occ_m >> cur;
                    const uint64_t upto = ahead == 0ull ? ~0ull : (1ull << (cur + __builtin_ctzll(ahead))) - 1ull;
                    cur = max(cur, kWave - 1 - __builtin_clzll((starts & upto) | 1ull));
                }
                thr = lane_float(v.exit, cur);
                pending = true;
                cur += 1;
            }
        }
        if (kWrite && ((emit >> lane) & 1ull)) o.ts[n0 + (uint32_t)__popcll(emit & below)] = v.w;
        if (rec.words != nullptr && emit != 0ull) {
            if (windows < rec.max_windows && lane < 3)
                rec.words[1 + 3 * windows + lane] =
                    lane == 0 ? __float_as_uint(v.base) : (uint32_t)(emit >> (lane == 1 ? 0 : 32));
            ++windows;
        }
        if (last || n >= cap) {
            if (rec.words != nullptr && lane == 0) rec.words[0] = windows <= rec.max_windows ? windows : kNoRecord;
            return n;
        }
        v = next;
    }
}

__device__ __forceinline__ float start_t(const MarchParams &p, float t0, float noise) {
    return t0 + step_size(p, t0) * noise;  // marching.cu:159-160
}

// Marks every ray as not marched.  Of a block's start slots the first takes its sample
// prefix (march_scan_kernel); the second of block c is counter c of the count rounds.
__global__ void __launch_bounds__(kBlock)
    march_begin_kernel(uint32_t n_rays, uint32_t *__restrict__ rays_n_samples, uint32_t *__restrict__ startidx) {
    const size_t stride = (size_t)gridDim.x * kBlock;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n_rays; i += stride) {
        rays_n_samples[i] = kPastFill;
        startidx[i] = i % kRaysPerBlock == 0 ? kPastFill : 0u;
    }
}

// The records of rays [0, n): `words` words each, in the xyzs output.
struct RecordStore {
    uint32_t *base;
    uint32_t n, words;
};

__device__ __forceinline__ RayRecord record_of(const RecordStore &st, uint32_t i) {
    return i < st.n ? RayRecord{st.base + (size_t)i * st.words, (st.words - 1u) / 3u} : RayRecord{nullptr, 0u};
}

// Counts the rays of blocks [block_begin, block_end), one block a workgroup and round,
// one ray a wavefront.  Round r of the launch has counter first_counter + r, and a
// workgroup goes into it only while the counters before it, all of rays before its own,
// are short of total_samples; what it reads too early costs a block marched in vain, no
// more.  (Drawing rays from one shared counter instead cost a device atomic on one
// address per ray, about 10 ns each one after another: 4096 rays took 114 us.)
// The march is bound by one ray's latency, a chain of windows of about 250
// instructions: few wavefronts in flight lose little and march few rays past the fill.
// march_rays of 2^18 camera rays, about 38 samples each, into 2^18 slots, a call: 571 us with
// launches of growing size, now 161 (0.4 of it in rounds, 0.28 with empty stretches crossed
// at once).  Rounds of 4,096 rays take 10 us more, and beside a training step's MLP backward
// 21 us of the step.  Two cascades and growing steps (bound 2, from inside): 713 -> 371, 4,096
// rays into more slots than they fill 335 -> 182; bounds 4 and 16 5,590 -> 1,145 and 7,490 ->
// 4,738.  The exception is a grid without an empty cell, where the first round fills the
// buffer and the workgroups that end early march a block in vain: 2^16 rays, two cascades, 92
// -> 109 (2^18 rays 93 -> 75).  A watch on the last round's counter between windows mends that
// at the price of 50 us in the first case, the first round in a launch of its own at 12.
template <bool kOne>
__global__ void __launch_bounds__(kBlock)
    march_count_kernel(MarchParams p, bool word_ok, uint32_t n_rays, uint32_t total_samples, uint32_t block_begin,
                       uint32_t block_end, uint32_t first_counter, const float *__restrict__ rays_o,
                       const float *__restrict__ rays_d, const float *__restrict__ t_starts,
                       const float *__restrict__ t_ends, const float *__restrict__ noises,
                       const uint8_t *__restrict__ bits, RecordStore records, uint32_t *__restrict__ rays_n_samples,
                       uint32_t *__restrict__ counters /* = rays_sample_startidx */) {
    __shared__ uint32_t wave_n[kRaysPerBlock];
    __shared__ uint64_t before;
    const int lane = lane_id(), wave = (int)threadIdx.x / kWave;
    uint32_t c = first_counter;
    for (uint32_t blk = block_begin + blockIdx.x; blk < block_end; blk += gridDim.x, ++c) {
        if (c > 0) {
            if (wave == 0) {
                uint64_t sum = 0;
                for (uint32_t j = lane; j < c; j += kWave)
                    sum += __hip_atomic_load(counters + (size_t)j * kRaysPerBlock + 1, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
                sum = wave_sum64(sum);
                if (lane == 0) before = sum;
            }
            __syncthreads();
            if (before >= total_samples) return;
        }
        const uint32_t i = __builtin_amdgcn_readfirstlane(blk * kRaysPerBlock + wave);
        uint32_t n = 0;
        if (i < n_rays) {
            const float t0 = t_starts[i], t1 = t_ends[i];
            if (t1 > t0) {
                const Ray r = load_ray(rays_o, rays_d, i, t1);
                n = march_ray_wave<false, kOne>(p, bits, word_ok, r, start_t(p, t0, noises[i]), p.n_cap, RaySamples{},
                                          record_of(records, i));
            }
            if (lane == 0) rays_n_samples[i] = min(n, kPastFill - 1u);
        }
        if (lane == 0) wave_n[wave] = n;
        __syncthreads();
        // (clamped so that a counter cannot wrap: counting less only stops later)
        if (threadIdx.x == 0 && (uint64_t)c * kRaysPerBlock + 1 < n_rays) {
            uint32_t s = 0;
#pragma unroll
            for (int w = 0; w < kRaysPerBlock; ++w) s += min(wave_n[w], 1u << 17);
            if (s > 0) atomicAdd(counters + (size_t)c * kRaysPerBlock + 1, s);
        }
    }
}

__device__ __forceinline__ uint32_t sat_add(uint32_t a, uint32_t b) {
    const uint32_t c = a + b;
    return c < a ? 0xffffffffu : c;
}

// Single workgroup.  Writes each block's exclusive sample prefix (a block is
// kRaysPerBlock consecutive rays; saturated: only its comparison with total_samples
// matters) to the first of its rays_sample_startidx slots, and
// next_sample_write_location / number_of_exceeded_samples.  Blocks are read in
// tiles of 4096 with all loads of a tile in flight; the scan stops after the first
// block with a ray that was not marched (the rays before it already fill the buffer,
// and the marks of later blocks are prefixes past it).
constexpr int kScanPerThread = 4;
__global__ void __launch_bounds__(kScanThreads)
    march_scan_kernel(uint32_t n_rays, uint32_t n_blocks, uint32_t total_samples,
                      const uint32_t *__restrict__ rays_n_samples, uint32_t *__restrict__ block_slots,
                      uint32_t *__restrict__ next_loc, uint32_t *__restrict__ exceeded) {
    constexpr uint32_t kTile = kScanThreads * kScanPerThread;
    __shared__ uint32_t first_past;
    __shared__ uint32_t fill_block;
    __shared__ uint32_t wave_tot[kScanThreads / kWave];
    const uint32_t tid = threadIdx.x;
    const int lane = lane_id(), wave = (int)tid / kWave;
    if (tid == 0) fill_block = 0xffffffffu;
    uint32_t carry = 0;  // saturated prefix of the tiles before
    uint32_t scanned = 0;
    for (uint32_t t0 = 0; t0 < n_blocks; t0 += kTile) {
        if (tid == 0) first_past = 0xffffffffu;
        uint32_t v[kScanPerThread], my_first = 0xffffffffu;
        {
            uint32_t cnt[kScanPerThread][kRaysPerBlock];
#pragma unroll
            for (int k = 0; k < kScanPerThread; ++k)
#pragma unroll
                for (int j = 0; j < kRaysPerBlock; ++j) {
                    const uint64_t r = (uint64_t)(t0 + tid * kScanPerThread + k) * kRaysPerBlock + j;
                    cnt[k][j] = r < n_rays ? rays_n_samples[r] : 0u;
                }
            // the samples of the block's rays before its first unmarched one
#pragma unroll
            for (int k = kScanPerThread - 1; k >= 0; --k) {
                bool past = false;
                v[k] = 0u;
#pragma unroll
                for (int j = 0; j < kRaysPerBlock; ++j) {
                    past = past || cnt[k][j] == kPastFill;
                    if (!past) v[k] = sat_add(v[k], cnt[k][j]);
                }
                if (past) my_first = t0 + tid * kScanPerThread + k;
            }
        }
        __syncthreads();
        // first such block of the tile: block indices grow with the thread and slot,
        // so the lowest lane holding one has the wave's first; one LDS atomic per wave
        // (not one per block, which serialised on the one address)
        const uint64_t has = __ballot(my_first != 0xffffffffu);
        if (has != 0ull && lane == __ffsll((unsigned long long)has) - 1) atomicMin(&first_past, my_first);
        __syncthreads();
        const uint32_t stop = first_past == 0xffffffffu ? first_past : first_past + 1u;
        uint32_t mine = 0;
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k) {
            if (t0 + tid * kScanPerThread + k >= stop) v[k] = 0;
            mine = sat_add(mine, v[k]);
        }
        // inclusive saturated scan over the wave, then over the waves
        uint32_t incl = mine;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d, kWave);
            if (lane >= d) incl = sat_add(incl, o);
        }
        if (lane == kWave - 1) wave_tot[wave] = incl;
        __syncthreads();
        uint32_t before = carry, tile_total = carry;
        for (int w = 0; w < kScanThreads / kWave; ++w) {
            if (w < wave) before = sat_add(before, wave_tot[w]);
            tile_total = sat_add(tile_total, wave_tot[w]);
        }
        uint32_t run = sat_add(before, incl - mine);  // exclusive prefix of this thread's first block
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k) {
            const uint32_t b = t0 + tid * kScanPerThread + k;
            if (b < stop && b < n_blocks) {
                // the first block whose inclusive prefix passes total_samples holds the fill point
                const uint32_t incl_b = sat_add(run, v[k]);
                if (incl_b > total_samples && run <= total_samples) atomicMin(&fill_block, b);
                block_slots[(size_t)b * kRaysPerBlock] = run;
                run = incl_b;
            }
        }
        carry = tile_total;
        __syncthreads();  // wave_tot and first_past are rewritten by the next tile
        if (stop != 0xffffffffu) {
            scanned = min(stop, n_blocks);
            break;
        }
        scanned = min(n_blocks, t0 + kTile);
    }
    __syncthreads();
    if (tid == 0) {
        const uint32_t grand = carry;
        if (grand <= total_samples) {
            *next_loc = grand;
            *exceeded = 0;
        } else {
            // walk the fill block's rays: first ray whose inclusive prefix passes total_samples
            const uint32_t b = fill_block < scanned ? fill_block : scanned - 1;  // set whenever grand > S
            uint64_t pre = block_slots[(size_t)b * kRaysPerBlock];
            const uint32_t first = b * kRaysPerBlock, last = min(n_rays - first, (uint32_t)kRaysPerBlock);
            uint32_t cnt[kRaysPerBlock];
#pragma unroll
            for (uint32_t j = 0; j < kRaysPerBlock; ++j) cnt[j] = j < last ? rays_n_samples[first + j] : 0u;
            uint32_t measured = (uint32_t)pre, over = 0;
#pragma unroll
            for (uint32_t j = 0; j < kRaysPerBlock; ++j) {
                const uint32_t n = cnt[j];
                if (pre + n > total_samples) {
                    measured = (uint32_t)pre;
                    over = pre < total_samples ? n : 0;
                    break;
                }
                pre += n;
            }
            *next_loc = measured + over;
            *exceeded = over;
        }
    }
}

// Sample range of ray i from the scanned block prefixes (slot of i's block) and
// the counts of the rays before i in its block.
__device__ __forceinline__ uint64_t ray_start(const uint32_t *__restrict__ rays_n_samples,
                                              const uint32_t *__restrict__ block_slots, uint32_t i) {
    const uint32_t first = i / kRaysPerBlock * kRaysPerBlock;
    uint64_t start = block_slots[first];
    for (uint32_t j = first; j < i; ++j) start += rays_n_samples[j];
    return start;
}

// Wavefront per ray, grid-stride over rays: writes the t of every valid ray's
// samples to z_vals at the ray's range, made from its record, or marched again
// where it has none.  Stops at the first ray whose block prefix reaches
// total_samples (every later ray is past the filled buffer).  Runs before
// march_finish_kernel overwrites the block slots.
template <bool kOne>
__global__ void __launch_bounds__(kBlock)
    march_emit_kernel(MarchParams p, bool word_ok, uint32_t n_rays, uint32_t total_samples,
                      const float *__restrict__ rays_o, const float *__restrict__ rays_d,
                      const float *__restrict__ t_starts, const float *__restrict__ t_ends,
                      const float *__restrict__ noises, const uint8_t *__restrict__ bits, RecordStore records,
                      const uint32_t *__restrict__ rays_n_samples,
                      const uint32_t *__restrict__ block_slots, float *__restrict__ zs) {
    const uint32_t n_waves = gridDim.x * kRaysPerBlock;
    for (uint32_t i = blockIdx.x * kRaysPerBlock + threadIdx.x / kWave; i < n_rays; i += n_waves) {
        if (block_slots[i / kRaysPerBlock * kRaysPerBlock] >= total_samples) break;
        const uint64_t start = ray_start(rays_n_samples, block_slots, i);
        const uint32_t n = rays_n_samples[i];
        const float t0 = t_starts[i], t1 = t_ends[i];
        if (start < total_samples && t1 > t0 && start + n <= total_samples && n > 0) {
            const uint32_t s = (uint32_t)start;
            const RayRecord rec = record_of(records, i);
            const uint32_t windows = rec.words != nullptr ? rec.words[0] : kNoRecord;
            if (windows != kNoRecord) {
                uint32_t k = s;
                for (uint32_t j = 0; j < windows; ++j) {
                    const uint32_t *e = rec.words + 1 + 3 * j;
                    const uint64_t mask = (uint64_t)e[2] << 32 | e[1];
                    float w, next;
                    bool stall;
                    chain_window(p, p.portion == 0.0f, step_size(p, 0.0f), __uint_as_float(e[0]), w, next, stall);
                    const int lane = lane_id();
                    if ((mask >> lane) & 1ull) zs[k + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = w;
                    k += (uint32_t)__popcll(mask);
                }
            } else {
                const Ray r = load_ray(rays_o, rays_d, i, t1);
                march_ray_wave<true, kOne>(p, bits, word_ok, r, start_t(p, t0, noises[i]), min(p.n_cap, n),
                                     RaySamples{zs + s}, RayRecord{nullptr, 0u});
            }
        }
    }
}

// Wavefront per valid ray, lanes over its samples: the outputs that follow from t
// (marching.cu:178-187): ray index, position o + t d, direction, step size.
__global__ void __launch_bounds__(kBlock)
    march_fill_kernel(MarchParams p, uint32_t n_rays, uint32_t total_samples, const float *__restrict__ rays_o,
                      const float *__restrict__ rays_d, const float *__restrict__ t_starts,
                      const float *__restrict__ t_ends, const uint32_t *__restrict__ rays_n_samples,
                      const uint32_t *__restrict__ block_slots, const float *__restrict__ zs,
                      uint32_t *__restrict__ idcs, float *__restrict__ xyzs, float *__restrict__ dirs,
                      float *__restrict__ dss) {
    const uint32_t n_waves = gridDim.x * kRaysPerBlock;
    for (uint32_t i = blockIdx.x * kRaysPerBlock + threadIdx.x / kWave; i < n_rays; i += n_waves) {
        if (block_slots[i / kRaysPerBlock * kRaysPerBlock] >= total_samples) break;
        const uint64_t start = ray_start(rays_n_samples, block_slots, i);
        const uint32_t n = rays_n_samples[i];
        const float t0 = t_starts[i], t1 = t_ends[i];
        if (start < total_samples && t1 > t0 && start + n <= total_samples && n > 0) {
            const Ray r = load_ray(rays_o, rays_d, i, t1);
            for (uint32_t k = lane_id(); k < n; k += kWave) {
                const size_t j = start + k;
                const float t = zs[j];
                idcs[j] = i;
                xyzs[3 * j + 0] = r.ox + t * r.dx;
                xyzs[3 * j + 1] = r.oy + t * r.dy;
                xyzs[3 * j + 2] = r.oz + t * r.dz;
                dirs[3 * j + 0] = r.dx;
                dirs[3 * j + 1] = r.dy;
                dirs[3 * j + 2] = r.dz;
                dss[j] = step_size(p, t);
            }
        }
    }
}

// Thread per ray: validity, final counts and start indices (replacing the block
// slots), and zeros in the sample slots no valid ray owns, [measured, total_samples).
__global__ void __launch_bounds__(kBlock)
    march_finish_kernel(uint32_t n_rays, uint32_t total_samples, const float *__restrict__ t_starts,
                        const float *__restrict__ t_ends, const uint32_t *__restrict__ next_loc,
                        const uint32_t *__restrict__ exceeded, bool *__restrict__ ray_is_valid,
                        uint32_t *__restrict__ rays_n_samples, uint32_t *__restrict__ rays_sample_startidx,
                        uint32_t *__restrict__ idcs, float *__restrict__ xyzs, float *__restrict__ dirs,
                        float *__restrict__ dss, float *__restrict__ zs) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    const int lane = lane_id();
    // a block's rays are kRaysPerBlock consecutive lanes of one wavefront
    const uint32_t n = i < n_rays ? rays_n_samples[i] : 0u;
    const uint32_t slot = i < n_rays ? rays_sample_startidx[i / kRaysPerBlock * kRaysPerBlock] : 0u;
    const int k = lane % kRaysPerBlock;
    uint64_t start = slot;
#pragma unroll
    for (int d = 1; d < kRaysPerBlock; ++d) {
        const uint32_t o = __shfl_up(n, d, kWave);
        if (k >= d) start += o;
    }
    if (i < n_rays) {
        const float t0 = t_starts[i], t1 = t_ends[i];
        const bool valid = start < total_samples && t1 > t0 && start + n <= total_samples;
        ray_is_valid[i] = valid;
        rays_n_samples[i] = valid ? n : 0u;
        rays_sample_startidx[i] = (valid && n > 0) ? (uint32_t)start : 0u;
    }
    const uint32_t measured = *next_loc - *exceeded;
    const size_t stride = (size_t)gridDim.x * kBlock;
    for (size_t j = (size_t)measured + blockIdx.x * kBlock + threadIdx.x; j < total_samples; j += stride) {
        idcs[j] = 0u;
        xyzs[3 * j + 0] = 0.0f;
        xyzs[3 * j + 1] = 0.0f;
        xyzs[3 * j + 2] = 0.0f;
        dirs[3 * j + 0] = 0.0f;
        dirs[3 * j + 1] = 0.0f;
        dirs[3 * j + 2] = 0.0f;
        dss[j] = 0.0f;
        zs[j] = 0.0f;
    }
}

// n_rays == 0: no rays, every sample slot zero, both counters zero.
__global__ void march_empty_kernel(uint32_t total_samples, uint32_t *next_loc, uint32_t *exceeded,
                                   uint32_t *__restrict__ idcs, float *__restrict__ xyzs, float *__restrict__ dirs,
                                   float *__restrict__ dss, float *__restrict__ zs) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g == 0) {
        *next_loc = 0;
        *exceeded = 0;
    }
    for (size_t j = g; j < total_samples; j += stride) {
        idcs[j] = 0u;
        xyzs[3 * j + 0] = xyzs[3 * j + 1] = xyzs[3 * j + 2] = 0.0f;
        dirs[3 * j + 0] = dirs[3 * j + 1] = dirs[3 * j + 2] = 0.0f;
        dss[j] = 0.0f;
        zs[j] = 0.0f;
    }
}

// ---------------------------------------------------------------------------
// inference
// ---------------------------------------------------------------------------

// Terminated slots take new ray indices in slot order (the reference hands them
// out with atomicAdd, marching.cu:300).  Up to kMaxAssignOnce slots every block counts the
// terminated ones before its own range by itself, in one launch (2^18 slots: 8 us
// instead of 11 us); past that, where this would read too much, and with next_in and next_out
// in one place, in three launches without scratch memory:
// per-block counts of terminated slots are parked in the first slot of each
// block's range of indices_out, one workgroup turns them into exclusive prefixes
// (and writes next_out), and every block then assigns its range.
constexpr int kAssignBlock = 1024;

constexpr uint32_t kMaxAssignOnce = 1u << 19;

__global__ void __launch_bounds__(kAssignBlock)
    assign_kernel(uint32_t n_rays, const bool *__restrict__ terminated, const uint32_t *__restrict__ indices_in,
                  const uint32_t *__restrict__ next_in, uint32_t *__restrict__ next_out,
                  uint32_t *__restrict__ indices_out) {
    const uint32_t first = blockIdx.x * kAssignBlock, j = first + threadIdx.x;
    uint32_t c = 0, before = 0, own = 0;
    // (bools are 0 or 1; the flags are 16-byte aligned; kLoads of them in flight)
    constexpr uint32_t kLoads = 8;
    for (uint32_t q0 = threadIdx.x; q0 < first / 16u; q0 += kLoads * kAssignBlock) {
        uint4 v[kLoads];
#pragma unroll
        for (uint32_t u = 0; u < kLoads; ++u) {
            const uint32_t q = q0 + u * kAssignBlock;
            v[u] = q < first / 16u ? reinterpret_cast<const uint4 *>(terminated)[q] : make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (uint32_t u = 0; u < kLoads; ++u)
            c += (uint32_t)(__popc(v[u].x) + __popc(v[u].y) + __popc(v[u].z) + __popc(v[u].w));
    }
    block_exclusive_scan<kAssignBlock>(c, &before);
    before += *next_in;
    const bool t = j < n_rays && terminated[j];
    const uint32_t at = before + block_exclusive_scan<kAssignBlock>(t ? 1u : 0u, &own);
    if (j < n_rays) indices_out[j] = t ? at : indices_in[j];
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *next_out = before + own;
}

__global__ void __launch_bounds__(kAssignBlock)
    assign_count_kernel(uint32_t n_rays, const bool *__restrict__ terminated, uint32_t *__restrict__ indices_out) {
    __shared__ uint32_t wave_cnt[kAssignBlock / kWave];
    const uint32_t j = blockIdx.x * kAssignBlock + threadIdx.x;
    const bool t = j < n_rays && terminated[j];
    const uint32_t c = (uint32_t)__popcll(__ballot(t));
    if (lane_id() == 0) wave_cnt[threadIdx.x / kWave] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t s = 0;
        for (int w = 0; w < kAssignBlock / kWave; ++w) s += wave_cnt[w];
        indices_out[(size_t)blockIdx.x * kAssignBlock] = s;
    }
}

__global__ void __launch_bounds__(kScanThreads)
    assign_scan_kernel(uint32_t n_blocks, const uint32_t *__restrict__ next_in, uint32_t *__restrict__ next_out,
                       uint32_t *__restrict__ indices_out) {
    const uint32_t first = *next_in;  // read before anything is written (next_out may alias it)
    uint32_t carry = first;
    for (uint32_t c0 = 0; c0 < n_blocks; c0 += kScanThreads) {
        const uint32_t b = c0 + threadIdx.x;
        const uint32_t v = b < n_blocks ? indices_out[(size_t)b * kAssignBlock] : 0u;
        uint32_t tot;
        const uint32_t ex = block_exclusive_scan<kScanThreads>(v, &tot);
        if (b < n_blocks) indices_out[(size_t)b * kAssignBlock] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) *next_out = carry;
}

__global__ void __launch_bounds__(kAssignBlock)
    assign_write_kernel(uint32_t n_rays, const bool *__restrict__ terminated, const uint32_t *__restrict__ indices_in,
                        uint32_t *__restrict__ indices_out) {
    __shared__ uint32_t base;
    __shared__ uint32_t wave_cnt[kAssignBlock / kWave];
    const uint32_t j = blockIdx.x * kAssignBlock + threadIdx.x;
    if (threadIdx.x == 0) base = indices_out[(size_t)blockIdx.x * kAssignBlock];
    const bool t = j < n_rays && terminated[j];
    const uint64_t m = __ballot(t);
    if (lane_id() == 0) wave_cnt[threadIdx.x / kWave] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t before = base;
    const int wave = (int)threadIdx.x / kWave;
    for (int w = 0; w < wave; ++w) before += wave_cnt[w];
    const uint64_t below = (1ull << lane_id()) - 1ull;
    if (j < n_rays) indices_out[j] = t ? before + (uint32_t)__popcll(m & below) : indices_in[j];
}

// One ray's march in a cascade of one grid over [-1, 1]^3 with a constant step k (K = 1,
// bound >= 1, stepsize_portion = 0), on one lane.  The lanes of a wavefront are rays, each
// as long as its slowest (a slot's new ray crosses empty space, the others take their next
// samples), and issuing instructions bounds it: the general loop spends 150 on a cell and
// 30 on steps that a skip adds one by one.  A round of 2^18 slots, 800 x 800 rays through
// G = 128: 182 -> 78 us (58 with the outputs staged, below).  Here:
//   * a skip is one multiplication.  Inside a binade of t every addition of k adds the same
//     `inc`, k rounded to the ulp (ties, where that depends on t, take the loop), so the
//     n-th step is t + n inc, exactly.
//   * an occupancy word holds a 4x4x4 block.  If it is zero the skip goes to the first step
//     past the block.  The loop gets there too: every step it visits inside the block is
//     empty, and each visit's exit distance lies before the block's up to rounding, so only
//     a step within the rounding error of the block's exit could be judged differently; if
//     there is one between the bounds lo and hi below, the cell's own exit is taken.
struct PlainMarch {
    float half_G, inv_G, gmax, k;
    float sx, sy, sz, hx, hy, hz;  // towards the exit: half a cell, a block or none
    float ex, ey, ez, slack;       // bounds of the rounding error of exit distances
    float limit, inc, per_inc;     // of the binade t is in (limit: its end)

    __device__ __forceinline__ PlainMarch(const MarchParams &p, const Ray &r) {
        half_G = 0.5f * (float)p.G;
        inv_G = p.inv_G;
        gmax = (float)(p.G - 1);
        k = step_size(p, 0.0f);
        sx = copysignf(0.5f, r.dx);
        sy = copysignf(0.5f, r.dy);
        sz = copysignf(0.5f, r.dz);
        hx = sx > 0.0f ? 4.0f : 0.0f;
        hy = sy > 0.0f ? 4.0f : 0.0f;
        hz = sz > 0.0f ? 4.0f : 0.0f;
        ex = error_bound(r.ox, r.dx, r.idx, r.t1);
        ey = error_bound(r.oy, r.dy, r.idy, r.t1);
        ez = error_bound(r.oz, r.dz, r.idz, r.t1);
        const float inf = __builtin_huge_valf();
        // 1 / d overflows for a tiny d: exit distances say nothing then
        const bool tiny = (r.dx != 0.0f && fabsf(r.idx) == inf) || (r.dy != 0.0f && fabsf(r.idy) == inf) ||
                          (r.dz != 0.0f && fabsf(r.idz) == inf);
        slack = tiny ? inf : 2.3841858e-7f * fabsf(r.t1);  // 2^-22: t + exit
        limit = 0.0f;
        inc = per_inc = 0.0f;
    }

    // A position carries up to 2^-24 (|o| + 2 t|d| + 3), a plane 2^-24, and the exit distance
    // has two positions' errors over d: 2^-21 (|o| + t|d| + 1.5) is more than twice that.
    static __device__ __forceinline__ float error_bound(float o, float d, float id, float t1) {
        return d == 0.0f ? 0.0f : 4.7683716e-7f * (fabsf(o) + fabsf(t1 * d) + 1.5f) * fabsf(id);
    }

    __device__ __forceinline__ void enter_binade(float t) {
        const uint32_t e8 = __float_as_uint(t) >> 23;  // sign bit included: a negative t has no inc
        inc = per_inc = 0.0f;
        limit = 0.0f;
        if (e8 < 24u || e8 > 253u) return;
        limit = __uint_as_float((e8 + 1u) << 23);
        const float q = k * __uint_as_float((277u - e8) << 23);  // k in ulps of t, exact
        const float m = rintf(q);
        if (m >= 1.0f && m <= 65536.0f && fabsf(q - m) != 0.5f) {
            inc = m * __uint_as_float((e8 - 23u) << 23);
            per_inc = 1.0f / inc;
        }
    }

    // First step after t at or past thr; false where it is not inside t's binade.
    __device__ __forceinline__ bool step_to(float t, float thr, float &nt) const {
        const float n = fmaxf(1.0f, ceilf((thr - t) * per_inc));
        nt = fmaf(n, inc, t);
        if (!(nt < limit)) return false;  // a sum past the binade is rounded
        if (n > 1.0f && nt - inc >= thr) nt -= inc;
        if (nt < thr) nt += inc;
        return inc > 0.0f && nt < limit;
    }

    // t of the next visited step after the empty cell at t, position (px, py, pz) and grid
    // coordinates (gx, gy, gz).
    __device__ __forceinline__ float skip(const MarchParams &p, const Ray &r, bool empty_block, float t, float px, float py,
                                          float pz, float gx, float gy, float gz) {
        if (!(t < limit)) enter_binade(t);
        float nt;
        if (empty_block) {
            const float bx = exit_plane(fmaf(4.0f, floorf(gx * 0.25f), hx), px) * r.idx;
            const float by = exit_plane(fmaf(4.0f, floorf(gy * 0.25f), hy), py) * r.idy;
            const float bz = exit_plane(fmaf(4.0f, floorf(gz * 0.25f), hz), pz) * r.idz;
            const float lo = t + (fminf(bx - ex, fminf(by - ey, bz - ez)) - slack);
            const float hi = t + (fminf(bx + ex, fminf(by + ey, bz + ez)) + slack);
            if (step_to(t, hi, nt) && nt - inc < lo && nt < r.t1) return nt;
        }
        const float cx = exit_plane(floorf((gx + 0.5f) + sx), px) * r.idx;
        const float cy = exit_plane(floorf((gy + 0.5f) + sy), py) * r.idy;
        const float cz = exit_plane(floorf((gz + 0.5f) + sz), pz) * r.idz;
        const float thr = t + fmaxf(0.0f, fminf(cx, fminf(cy, cz)));
        return step_to(t, thr, nt) ? nt : skip_to(p, t, k, thr);
    }

    // distance from x to the plane at grid coordinate n: the products are exact, so this
    // rounds as ((n * inv_G) - 0.5) * 2 - x does
    __device__ __forceinline__ float exit_plane(float n, float x) const {
        return fmaf(2.0f, fmaf(n, inv_G, -0.5f), -x);
    }
};

// PlainMarch's case of lookup_cell.
__device__ __forceinline__ bool lookup_plain(const PlainMarch &m, BitCache &cache, float px, float py, float pz, float &gx,
                                             float &gy, float &gz) {
    gx = (px + 1.0f) * m.half_G;  // the factor is a power of two: exact
    gy = (py + 1.0f) * m.half_G;
    gz = (pz + 1.0f) * m.half_G;
    const uint32_t ix = (uint32_t)fminf(fmaxf(gx, 0.0f), m.gmax);
    const uint32_t iy = (uint32_t)fminf(fmaxf(gy, 0.0f), m.gmax);
    const uint32_t iz = (uint32_t)fminf(fmaxf(gz, 0.0f), m.gmax);
    return occupied(cache, nullptr, morton_spread10(ix) | (morton_spread10(iy) << 1) | (morton_spread10(iz) << 2));
}

// Where a lane's samples go until its wavefront writes them.  Stored sample by sample, or
// zero by zero, a lane's outputs are stores to 64 lines each; a round of 2^18 slots that
// had next to no rays left took 61 us (now 36, one ray's march).  So a lane keeps the t of
// its samples in LDS and its wavefront computes and writes all entries of its 64 slots in
// order: 78 -> 58 us a round on average.  A cap past kMaxStagedCap stores directly.
constexpr uint32_t kStagePitch = kBlock + 8;
constexpr uint32_t kMaxStagedCap = 65536 / (4 * kStagePitch);

template <bool kPlain, bool kStaged>
__global__ void __launch_bounds__(kBlock)
    march_inference_kernel(MarchParams p, bool word_ok, uint32_t n_total_rays, uint32_t n_rays, uint32_t cap,
                           const float *__restrict__ rays_o, const float *__restrict__ rays_d,
                           const float *__restrict__ t_starts, const float *__restrict__ t_ends,
                           const uint8_t *__restrict__ bits, const uint32_t *__restrict__ indices,
                           uint32_t *__restrict__ n_samples, float *__restrict__ t_out, float *__restrict__ xyzs,
                           float *__restrict__ dss, float *__restrict__ zs) {
    extern __shared__ float staged[];
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    const bool in_range = i < n_rays;
    if (!kStaged && !in_range) return;
    float *rx = xyzs + (size_t)i * cap * 3;
    float *rds = dss + (size_t)i * cap;
    float *rz = zs + (size_t)i * cap;
    const uint32_t r = in_range ? indices[i] : n_total_rays;
    uint32_t steps = 0;
    float t = 0.0f;
    // the sample that ends at the far plane, and its step
    uint32_t cut = 0xffffffffu;
    float cut_ds = 0.0f;
    Ray ray = {};
    const auto take = [&](float px, float py, float pz, float ds, float at) {
        if constexpr (kStaged) {
            staged[steps * kStagePitch + threadIdx.x] = at;
        } else {
            rx[3 * steps + 0] = px;
            rx[3 * steps + 1] = py;
            rx[3 * steps + 2] = pz;
            rds[steps] = ds;
            rz[steps] = at;
        }
        ++steps;
    };
    if (r < n_total_rays) {
        const float t0 = t_starts[r], t1 = t_ends[r];
        if (!(t1 < t0)) {
            ray = load_ray(rays_o, rays_d, r, t1);
            BitCache cache = make_bit_cache(bits, kPlain || word_ok);
            t = t0;
            float last_t = 0.0f;  // of the last sample
            if constexpr (kPlain) {
                PlainMarch m(p, ray);
                while (steps < cap && t < t1) {
                    const float px = ray.ox + t * ray.dx, py = ray.oy + t * ray.dy, pz = ray.oz + t * ray.dz;
                    float gx, gy, gz;
                    if (lookup_plain(m, cache, px, py, pz, gx, gy, gz)) {
                        take(px, py, pz, m.k, t);
                        last_t = t;
                        t = t + m.k;
                    } else {
                        t = m.skip(p, ray, cache.word == 0ull, t, px, py, pz, gx, gy, gz);
                    }
                }
            } else {
                while (steps < cap && t < t1) {
                    const float px = ray.ox + t * ray.dx, py = ray.oy + t * ray.dy, pz = ray.oz + t * ray.dz;
                    const float ds = step_size(p, t);
                    float gx, gy, gz, mb;
                    if (lookup_cell(p, bits, cache, px, py, pz, ds, gx, gy, gz, mb)) {
                        take(px, py, pz, ds, t);
                        last_t = t;
                        t = t + ds;
                    } else {
                        t = skip_to(p, t, ds, cell_exit_t(p, t, px, py, pz, gx, gy, gz, mb, ray.dx, ray.dy, ray.dz,
                                                          ray.idx, ray.idy, ray.idz));
                    }
                }
            }
            // far-plane sample (marching.cu:367-394)
            if (t >= t1) {
                const float px = ray.ox + t1 * ray.dx, py = ray.oy + t1 * ray.dy, pz = ray.oz + t1 * ray.dz;
                const float ds = step_size(p, t1);
                float gx, gy, gz, mb;
                if (lookup_cell(p, bits, cache, px, py, pz, ds, gx, gy, gz, mb)) {
                    if (steps > 0 && step_size(p, last_t) + last_t >= t1) {
                        cut = steps - 1;
                        cut_ds = t1 - last_t;
                        if (!kStaged) rds[cut] = cut_ds;
                    }
                    if (steps < cap) take(px, py, pz, ds, t1);
                    else t = t1;
                }
            }
        }
    }
    if (in_range) {
        n_samples[i] = steps;
        t_out[i] = t;
    }
    // unused sample slots are zero (the reference memsets them, marching.cu:565-570)
    if constexpr (!kStaged) {
        for (uint32_t k = steps; k < cap; ++k) {
            rx[3 * k + 0] = 0.0f;
            rx[3 * k + 1] = 0.0f;
            rx[3 * k + 2] = 0.0f;
            rds[k] = 0.0f;
            rz[k] = 0.0f;
        }
    } else {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const uint32_t lane = (uint32_t)lane_id();
        const uint32_t first = i - lane;  // the wavefront's slots
        if (first >= n_rays) return;
        const uint32_t n_entries = min(n_rays - first, (uint32_t)kWave) * cap;
        const size_t base = (size_t)first * cap;
        const uint32_t slot_step = kWave / cap, k_step = kWave % cap;
        uint32_t slot = lane / cap, k = lane % cap;
        for (uint32_t e0 = 0; e0 < n_entries; e0 += kWave) {
            const uint32_t e = e0 + lane;
            const int from = (int)min(slot, (uint32_t)kWave - 1u);
            const float ox = __shfl(ray.ox, from), oy = __shfl(ray.oy, from), oz = __shfl(ray.oz, from);
            const float dx = __shfl(ray.dx, from), dy = __shfl(ray.dy, from), dz = __shfl(ray.dz, from);
            const uint32_t n = __shfl(steps, from), cut_k = __shfl(cut, from);
            const float ds_k = __shfl(cut_ds, from);
            if (e < n_entries) {
                float px = 0.0f, py = 0.0f, pz = 0.0f, ds = 0.0f, at = 0.0f;
                if (k < n) {
                    at = staged[k * kStagePitch + (threadIdx.x - lane) + slot];
                    px = ox + at * dx;
                    py = oy + at * dy;
                    pz = oz + at * dz;
                    ds = k == cut_k ? ds_k : step_size(p, at);
                }
                float *x = xyzs + 3 * (base + e);
                x[0] = px;
                x[1] = py;
                x[2] = pz;
                dss[base + e] = ds;
                zs[base + e] = at;
            }
            slot += slot_step;
            k += k_step;
            if (k >= cap) {
                k -= cap;
                ++slot;
            }
        }
    }
}

// 64-bit words need an 8-byte aligned bitfield of a whole number of words.
bool bitfield_words_ok(const uint8_t *bits, uint32_t K, uint32_t G) {
    const uint64_t n_bytes = (uint64_t)K * G * G * G / 8;
    return (reinterpret_cast<uintptr_t>(bits) & 7u) == 0 && n_bytes % 8 == 0 && n_bytes > 0;
}

bool valid_march_statics(uint32_t diag, uint32_t K, uint32_t G, float bound, float portion, const char *target) {
    // Morton codes of cells in [0, G)^3 stay below G^3 only for power-of-two G
    const bool g_ok = G != 0 && G <= 1024 && (G & (G - 1)) == 0 && (uint64_t)K * G * G * G <= 0xffffffffull;
    if (diag == 0 || K == 0 || !g_ok || !(bound > 0.0f) || !(bound < 3.0e38f) || !(portion >= 0.0f) ||
        !(portion < 3.0e38f)) {
        set_error(kBadDescriptor,
                  "%s: invalid statics (diagonal_n_steps=%u K=%u G=%u bound=%g stepsize_portion=%g); need positive "
                  "diagonal_n_steps and K, G a power of two <= 1024 with K*G^3 < 2^32, finite bound > 0, finite "
                  "portion >= 0",
                  target, diag, K, G, (double)bound, (double)portion);
        return false;
    }
    return true;
}

}  // namespace
}  // namespace ngp

using namespace ngp;

extern "C" void march_rays(ngp_stream_t stream_, void **buffers, const char *opaque, size_t opaque_len) {
    const char *target = "march_rays";
    MarchingDescriptor d;
    if (!read_descriptor(opaque, opaque_len, &d, target)) return;
    if (!valid_march_statics(d.diagonal_n_steps, d.K, d.G, d.bound, d.stepsize_portion, target)) return;
    if (d.total_samples == 0) {
        set_error(kBadDescriptor, "%s: total_samples must be positive", target);
        return;
    }
    if (!check_buffer_list(buffers, {6, 7, 11, 12, 13, 14, 15}, target)) return;
    if (d.n_rays > 0 && !check_buffers(buffers, 16, target)) return;
    hipStream_t stream = (hipStream_t)stream_;
    const float *rays_o = (const float *)buffers[0];
    const float *rays_d = (const float *)buffers[1];
    const float *t_starts = (const float *)buffers[2];
    const float *t_ends = (const float *)buffers[3];
    const float *noises = (const float *)buffers[4];
    const uint8_t *bits = (const uint8_t *)buffers[5];
    uint32_t *next_loc = (uint32_t *)buffers[6];
    uint32_t *exceeded = (uint32_t *)buffers[7];
    bool *valid = (bool *)buffers[8];
    uint32_t *n_samples = (uint32_t *)buffers[9];
    uint32_t *startidx = (uint32_t *)buffers[10];
    uint32_t *idcs = (uint32_t *)buffers[11];
    float *xyzs = (float *)buffers[12];
    float *dirs = (float *)buffers[13];
    float *dss = (float *)buffers[14];
    float *zs = (float *)buffers[15];
    const MarchParams p = make_march_params(d.diagonal_n_steps, d.K, d.G, d.bound, d.stepsize_portion);
    const bool word_ok = bitfield_words_ok(bits, d.K, d.G);
    if (d.n_rays == 0) {
        hipLaunchKernelGGL(march_empty_kernel, dim3(min(div_up(d.total_samples, 256), 4096u)), dim3(256), 0, stream,
                           d.total_samples, next_loc, exceeded, idcs, xyzs, dirs, dss, zs);
        check_launch(target);
        return;
    }
    const bool one = d.K == 1;
    const uint32_t n_blocks = div_up(d.n_rays, kRaysPerBlock);
    constexpr uint32_t kMaxCountBlocks = 2048;
    hipLaunchKernelGGL(march_begin_kernel, dim3(std::min(div_up(d.n_rays, kBlock), 2048u)), dim3(kBlock), 0, stream,
                       d.n_rays, n_samples, startidx);
    if (!check_launch(target)) return;
    // records of the first rays in xyzs: a ray across the bound's diagonal, one that starts
    // and ends inside a window, has at most n_cap / 64 + 2 windows
    RecordStore rec;
    rec.base = (uint32_t *)xyzs;
    rec.words = 1u + 3u * (std::min(p.n_cap, 1u << 16) / kWave + 2u);
    rec.n = (uint32_t)std::min<uint64_t>(d.n_rays, 3ull * d.total_samples / rec.words);
    // the first rays, which fill a training batch, in rounds of 2048, the rest in rounds of
    // 8192 (every ray of a sparse field is marched: more wavefronts, more throughput)
    constexpr uint32_t kFirstBlocks = 512, kFirstRounds = 8;
    const uint32_t first_end = std::min(n_blocks, kFirstBlocks * kFirstRounds);
    for (int c = 0; c < 2; ++c) {
        const uint32_t begin = c == 0 ? 0 : first_end, end = c == 0 ? first_end : n_blocks;
        if (end <= begin) continue;
        hipLaunchKernelGGL(one ? march_count_kernel<true> : march_count_kernel<false>, dim3(std::min(end - begin, c == 0 ? kFirstBlocks : kMaxCountBlocks)),
                           dim3(kBlock), 0, stream, p, word_ok, d.n_rays, d.total_samples, begin, end,
                           c == 0 ? 0 : kFirstRounds, rays_o, rays_d, t_starts, t_ends, noises, bits, rec, n_samples,
                           startidx);
        if (!check_launch(target)) return;
    }
    hipLaunchKernelGGL(march_scan_kernel, dim3(1), dim3(kScanThreads), 0, stream, d.n_rays, n_blocks, d.total_samples,
                       n_samples, startidx, next_loc, exceeded);
    if (!check_launch(target)) return;
    hipLaunchKernelGGL(one ? march_emit_kernel<true> : march_emit_kernel<false>, dim3(std::min(n_blocks, kMaxCountBlocks)), dim3(kBlock), 0, stream, p, word_ok,
                       d.n_rays, d.total_samples, rays_o, rays_d, t_starts, t_ends, noises, bits, rec,
                       n_samples, startidx, zs);
    if (!check_launch(target)) return;
    hipLaunchKernelGGL(march_fill_kernel, dim3(std::min(n_blocks, kMaxCountBlocks)), dim3(kBlock), 0, stream, p,
                       d.n_rays, d.total_samples, rays_o, rays_d, t_starts, t_ends, n_samples, startidx, zs, idcs, xyzs,
                       dirs, dss);
    if (!check_launch(target)) return;
    // a thread per ray, and enough workgroups for the tail's zeros when rays are few
    const uint32_t finish_grid = std::max(div_up(d.n_rays, kBlock), std::min(div_up(d.total_samples, kBlock), 2048u));
    hipLaunchKernelGGL(march_finish_kernel, dim3(finish_grid), dim3(kBlock), 0, stream, d.n_rays,
                       d.total_samples, t_starts, t_ends, next_loc, exceeded, valid, n_samples, startidx, idcs, xyzs,
                       dirs, dss, zs);
    check_launch(target);
}

extern "C" void march_rays_inference(ngp_stream_t stream_, void **buffers, const char *opaque, size_t opaque_len) {
    const char *target = "march_rays_inference";
    MarchingInferenceDescriptor d;
    if (!read_descriptor(opaque, opaque_len, &d, target)) return;
    if (!valid_march_statics(d.diagonal_n_steps, d.K, d.G, d.bound, d.stepsize_portion, target)) return;
    if (d.march_steps_cap == 0) {
        set_error(kBadDescriptor, "%s: march_steps_cap must be positive", target);
        return;
    }
    if (d.n_rays == 0) return;
    if (!check_buffers(buffers, 15, target)) return;
    hipStream_t stream = (hipStream_t)stream_;
    const float *rays_o = (const float *)buffers[0];
    const float *rays_d = (const float *)buffers[1];
    const float *t_starts = (const float *)buffers[2];
    const float *t_ends = (const float *)buffers[3];
    const uint8_t *bits = (const uint8_t *)buffers[4];
    const uint32_t *next_in = (const uint32_t *)buffers[5];
    const bool *terminated = (const bool *)buffers[6];
    const uint32_t *indices_in = (const uint32_t *)buffers[7];
    uint32_t *next_out = (uint32_t *)buffers[8];
    uint32_t *indices_out = (uint32_t *)buffers[9];
    uint32_t *n_samples = (uint32_t *)buffers[10];
    float *t_out = (float *)buffers[11];
    float *xyzs = (float *)buffers[12];
    float *dss = (float *)buffers[13];
    float *zs = (float *)buffers[14];
    const MarchParams p = make_march_params(d.diagonal_n_steps, d.K, d.G, d.bound, d.stepsize_portion);
    const uint32_t n_assign = div_up(d.n_rays, kAssignBlock);
    if (d.n_rays <= kMaxAssignOnce && next_in != next_out && (reinterpret_cast<uintptr_t>(terminated) & 15u) == 0) {
        hipLaunchKernelGGL(assign_kernel, dim3(n_assign), dim3(kAssignBlock), 0, stream, d.n_rays, terminated, indices_in,
                           next_in, next_out, indices_out);
    } else {
        hipLaunchKernelGGL(assign_count_kernel, dim3(n_assign), dim3(kAssignBlock), 0, stream, d.n_rays, terminated,
                           indices_out);
        hipLaunchKernelGGL(assign_scan_kernel, dim3(1), dim3(kScanThreads), 0, stream, n_assign, next_in, next_out,
                           indices_out);
        hipLaunchKernelGGL(assign_write_kernel, dim3(n_assign), dim3(kAssignBlock), 0, stream, d.n_rays, terminated,
                           indices_in, indices_out);
    }
    if (!check_launch(target)) return;
    const bool word_ok = bitfield_words_ok(bits, d.K, d.G);
    const bool plain = word_ok && d.K == 1 && d.bound >= 1.0f && d.stepsize_portion == 0.0f;
    const bool staged = d.march_steps_cap <= kMaxStagedCap;
    const auto kernel = plain ? (staged ? march_inference_kernel<true, true> : march_inference_kernel<true, false>)
                              : (staged ? march_inference_kernel<false, true> : march_inference_kernel<false, false>);
    hipLaunchKernelGGL(kernel, dim3(div_up(d.n_rays, kBlock)), dim3(kBlock),
                       staged ? d.march_steps_cap * kStagePitch * sizeof(float) : 0, stream, p, word_ok, d.n_total_rays,
                       d.n_rays, d.march_steps_cap, rays_o, rays_d, t_starts, t_ends, bits, indices_out, n_samples, t_out,
                       xyzs, dss, zs);
    check_launch(target);
}
