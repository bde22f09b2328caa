// wc_kernels.hip -- gfx950 kernels of the SPH step: grid build (hash + histogram, decoupled
// look-back scan, place, stable within-cell rank + gather), density/pressure, force + integrate.
// Every pass is one launch over all scenes of a context.
//
// Floating-point contract (shared with the CPU transcription): binary32, correctly rounded '/'
// and sqrtf (-fhip-fp32-correctly-rounded-divide-sqrt), subnormals kept, no FMA contraction
// (-ffp-contract=off), every expression associated left to right as the GLSL source writes it.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "wc_arith.hpp"
#include "wc_internal.hpp"

namespace wc {
namespace {

__device__ __forceinline__ int cell_axis(float x, float bin, int R) {
    // ivec3(p / binSize) truncates toward zero, then clamp(.., 0, R-1) (count.comp:32).
    const float q = x / bin;
    if (!(q >= 0.0f)) return 0;
    if (q >= (float)R) return R - 1;
    const int c = (int)q;
    return c > R - 1 ? R - 1 : c;
}

__device__ __forceinline__ uint32_t cell_key(const StepConsts& c, float x, float y, float z) {
    const int cx = cell_axis(x, c.bin, c.R);
    const int cy = cell_axis(y, c.bin, c.R);
    const int cz = cell_axis(z, c.bin, c.R);
    return (uint32_t)((cz * c.R + cy) * c.R + cx);
}

__device__ __forceinline__ float poly6(const StepConsts& c, float r) {
    const float a = c.hh - r * r;
    return ((a * a) * a) * c.poly6;
}

__device__ __forceinline__ unsigned lane_id() { return __lane_id(); }

// The dispatcher hands workgroup b to XCD b % 8.  Renumber workgroups so that every XCD works
// through one contiguous run of logical blocks: neighbouring particles (which read the same
// neighbour cells) then share one XCD's L2 instead of being fetched by all eight.
constexpr uint32_t kNumXcd = 8;
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nblocks) {
    const uint32_t q = nblocks / kNumXcd, r = nblocks % kNumXcd;
    const uint32_t x = b % kNumXcd, k = b / kNumXcd;
    return x * q + min(x, r) + k;
}

// Scene owning logical block (or tile) b: a table load when the context holds several scenes.
__device__ __forceinline__ uint32_t scene_of(const uint32_t* __restrict__ table, uint32_t num_scenes, uint32_t b) {
    return num_scenes == 1 ? 0u : table[b];
}
template <int BLOCK>
__device__ __forceinline__ const uint32_t* scene_table(const Scenes& S) {
    return BLOCK == 64 ? S.scene64 : (BLOCK == 128 ? S.scene128 : S.scene256);
}

template <int BLOCK>
__device__ __forceinline__ const uint32_t* first_blocks(const Scenes& S) {
    return BLOCK == 64 ? S.blk64 : (BLOCK == 128 ? S.blk128 : S.blk256);
}
template <int BLOCK>
__device__ __forceinline__ uint32_t total_blocks(const Scenes& S) {
    return BLOCK == 64 ? S.blocks64 : (BLOCK == 128 ? S.blocks128 : S.blocks256);
}

// Bits of rho_max[1], the force pass's division mode: 0 lets it share reciprocals (quot).
constexpr uint32_t kDivUnsafe = 1u;   // an operand of this step is outside div_operand's range
constexpr uint32_t kDivPending = 2u;  // sorted since the last density pass

// Walks the in-grid neighbour cells of scene-local cell `key` in NEIGHBORHOOD order
// (density.comp:40-50: dx outermost, dz innermost); visit(start, end, own) receives each cell's
// slot range (clipped to `limit`) and whether it is the particle's own cell (the 14th of the 27,
// the same iteration in every lane: std::true_type there, std::false_type elsewhere), and
// end_plane() runs after every dx plane.  The trip counts of both cell loops are wave-uniform.
template <typename Visit, typename EndPlane>
__device__ __forceinline__ void for_each_neighbour_cell(uint32_t key, const uint2* __restrict__ range,
                                                        const StepConsts& c, uint32_t limit, Visit& visit,
                                                        EndPlane& end_plane) {
    const int R = c.R;
    const int cx = (int)(key % (uint32_t)R);
    const int cy = (int)((key / (uint32_t)R) % (uint32_t)R);
    const int cz = (int)(key / ((uint32_t)R * (uint32_t)R));
#pragma unroll 1
    for (int dx = -1; dx <= 1; ++dx) {
        const int nx = cx + dx;
#pragma unroll 1
        for (int dyz = 0; dyz < 9; ++dyz) {
            const int ny = cy + (dyz / 3 - 1);
            const int nz = cz + (dyz % 3 - 1);
            if (nx < 0 || ny < 0 || nz < 0 || nx >= R || ny >= R || nz >= R) continue;
            const uint2 rg = range[(nz * R + ny) * R + nx];
            if (dx == 0 && dyz == 4)
                visit(rg.x, min(rg.x + rg.y, limit), std::true_type{});
            else
                visit(rg.x, min(rg.x + rg.y, limit), std::false_type{});
        }
        end_plane();
    }
}

// ------------------------------------------------------------------------------------------
// 1. cell hash + histogram (count.comp:25-36).  Consecutive lanes that fall in the same cell
//    form one run; the run's first lane does a single atomicAdd for the whole run, every lane
//    keeps its arrival rank.  Also resets the scan's look-back state and the per-scene clocks
//    for this step.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kHashBlock) void k_hash(Scenes S, const float4* __restrict__ posrho,
                                                     uint32_t* __restrict__ key, uint32_t* __restrict__ rank,
                                                     uint32_t* __restrict__ counts,
                                                     unsigned long long* __restrict__ scan_status,
                                                     unsigned long long* __restrict__ scene_done,
                                                     unsigned long long* __restrict__ step_start,
                                                     uint32_t* __restrict__ rho_max,
                                                     uint32_t* __restrict__ crowd_count,
                                                     uint32_t* __restrict__ tile_count) {
    const uint32_t g = blockIdx.x * kHashBlock + threadIdx.x;
    if (g < S.total_tiles) scan_status[g] = 0ull;
    if (g < S.num_scenes) scene_done[g] = 0ull;
    if (tile_count && S.num_scenes > 1 && g < S.num_scenes) tile_count[kSceneSparse + g] = 0u;
    if (g == 0) {
        *crowd_count = 0u;
        if (tile_count) tile_count[0] = tile_count[1] = tile_count[kListCount] = tile_count[kSceneSparse - 1] = 0u;
        *step_start = wall_clock64();
        rho_max[0] = 0u;
        rho_max[1] = kDivPending;  // the force pass's operands are unchecked until a density pass runs
    }
    const uint32_t b = blockIdx.x;
    bool valid = false;
    uint32_t k = kNoKey, i = 0, c_off = 0;
    if (b < S.blocks256) {
        const uint32_t s = scene_of(S.scene256, S.num_scenes, b);
        const SceneDesc& d = S.desc[s];
        const uint32_t lt = (b - S.blk256[s]) * kHashBlock + threadIdx.x;
        valid = lt < d.c.n;
        if (valid) {
            i = d.p_off + lt;
            c_off = d.c_off;
            const float4 p = posrho[i];
            k = cell_key(d.c, p.x, p.y, p.z);
        }
    }
    const unsigned lane = lane_id();
    const uint32_t prev = __shfl_up(k, 1);
    const bool leader = (lane == 0) || (prev != k);
    const unsigned long long leaders = __ballot(leader);
    const unsigned long long upto = (2ull << lane) - 1ull;  // lanes 0..lane
    const int first = 63 - __clzll((long long)(leaders & upto));
    const unsigned long long above = leaders & ~upto;
    const int next = above ? (__ffsll((long long)above) - 1) : 64;
    uint32_t base = 0;
    if (leader && valid) base = atomicAdd(&counts[c_off + k], (uint32_t)(next - first));
    base = __shfl(base, first);
    if (valid) {
        key[i] = k;
        rank[i] = base + (uint32_t)((int)lane - first);
    }
}

// ------------------------------------------------------------------------------------------
// 2. exclusive scan of the per-cell counts (linearScan.comp:15-28), single pass with decoupled
//    look-back, each scene on its own chain of tiles.  Writes range[cell] = (first slot, count)
//    and zeroes the counts for the next step.
//    Look-back word: (flag << 32) | value; flag 1 = tile aggregate, 2 = inclusive prefix.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long ld_status(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_status(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

__global__ __launch_bounds__(kScanThreads) void k_scan(Scenes S, uint32_t* __restrict__ counts,
                                                       uint2* __restrict__ range,
                                                       unsigned long long* __restrict__ status,
                                                       uint32_t* __restrict__ error_flag) {
    __shared__ uint32_t s_wave[kScanThreads / 64];
    __shared__ uint32_t s_prefix;
    const unsigned tid = threadIdx.x;
    const unsigned lane = lane_id();
    const unsigned wave = tid >> 6;
    // Tile = workgroup index.  Each XCD dispatches its workgroups in index order, so the lowest
    // unfinished tile has been dispatched, and it waits on nothing (its predecessors are done):
    // the look-back always makes progress.  (A ticket counter gives the same guarantee, but
    // every workgroup then queues on one atomic: about 25-30 ns per tile.)
    const uint32_t tile = blockIdx.x;
    const uint32_t s = scene_of(S.scene_tile, S.num_scenes, tile);
    const uint32_t first_tile = S.tiles[s];
    const SceneDesc& d = S.desc[s];
    const uint32_t ncells = d.c.ncells;
    const size_t local = (size_t)(tile - first_tile) * kScanTile + (size_t)tid * kScanItems;
    uint32_t* cnt = counts + d.c_off;
    uint2* rng = range + d.c_off;

    uint32_t v[kScanItems];
    if (local + kScanItems <= ncells) {
        const uint4* src = reinterpret_cast<const uint4*>(cnt + local);
#pragma unroll
        for (int q = 0; q < kScanItems / 4; ++q) {
            const uint4 w = src[q];
            v[4 * q + 0] = w.x;
            v[4 * q + 1] = w.y;
            v[4 * q + 2] = w.z;
            v[4 * q + 3] = w.w;
        }
        uint4* dst = reinterpret_cast<uint4*>(cnt + local);
#pragma unroll
        for (int q = 0; q < kScanItems / 4; ++q) dst[q] = make_uint4(0u, 0u, 0u, 0u);
    } else {
#pragma unroll
        for (int j = 0; j < kScanItems; ++j) {
            v[j] = (local + j < ncells) ? cnt[local + j] : 0u;
            if (local + j < ncells) cnt[local + j] = 0u;
        }
    }
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) sum += v[j];

    uint32_t incl = sum;
#pragma unroll
    for (int dd = 1; dd < 64; dd <<= 1) {
        const uint32_t t = __shfl_up(incl, dd);
        if ((int)lane >= dd) incl += t;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    uint32_t wave_prefix = 0, tile_total = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w) {
        const uint32_t t = s_wave[w];
        if ((unsigned)w < wave) wave_prefix += t;
        tile_total += t;
    }
    const uint32_t thread_excl = wave_prefix + incl - sum;

    if (wave == 0) {
        uint32_t tile_prefix = 0;
        if (tile == first_tile) {
            if (lane == 0) st_status(&status[tile], (2ull << 32) | tile_total);
        } else {
            if (lane == 0) st_status(&status[tile], (1ull << 32) | tile_total);
            long long look = (long long)tile - 1;
            uint32_t acc = 0, spins = 0;
            for (;;) {
                const long long idx = look - (long long)lane;
                // tiles before the scene's first tile count as a zero prefix
                unsigned long long w = (idx >= (long long)first_tile) ? ld_status(&status[idx]) : (2ull << 32);
                const uint32_t flag = (uint32_t)(w >> 32);
                const unsigned long long not_ready = __ballot(flag == 0u);
                const unsigned long long is_prefix = __ballot(flag == 2u);
                const int first_prefix = is_prefix ? (__ffsll((long long)is_prefix) - 1) : 64;
                const unsigned long long window =
                    (first_prefix >= 63) ? ~0ull : ((2ull << first_prefix) - 1ull);
                if (not_ready & window) {
                    if (++spins > kLookbackSpinLimit) {
                        if (lane == 0) atomicOr(error_flag, 1u);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                const uint32_t contrib = ((int)lane <= first_prefix) ? (uint32_t)w : 0u;
                acc += wave_sum(contrib);
                if (first_prefix < 64) break;
                look -= 64;
            }
            tile_prefix = acc;
            if (lane == 0) st_status(&status[tile], (2ull << 32) | (uint32_t)(acc + tile_total));
        }
        if (lane == 0) s_prefix = tile_prefix;
    }
    __syncthreads();
    uint32_t run = d.p_off + s_prefix + thread_excl;
    if (local + kScanItems <= ncells) {
        uint4* dst = reinterpret_cast<uint4*>(rng + local);
#pragma unroll
        for (int q = 0; q < kScanItems / 2; ++q) {
            const uint32_t a = run;
            run += v[2 * q];
            const uint32_t b2 = run;
            run += v[2 * q + 1];
            dst[q] = make_uint4(a, v[2 * q], b2, v[2 * q + 1]);
        }
    } else {
#pragma unroll
        for (int j = 0; j < kScanItems; ++j) {
            if (local + j < ncells) rng[local + j] = make_uint2(run, v[j]);
            run += v[j];
        }
    }
}

// ------------------------------------------------------------------------------------------
// The tile passes' work list and cell tables (the passes themselves follow the force pass).  They need
// only the scan's ranges, so further workgroups of k_place form the list and further ones of k_gather
// the tables: a launch of their own each cost 4-5 us a step.
//
// Listed are the base boxes that hold particles.  One whose records with its halo exceed LDS is listed
// as boxes of 2x2x2 cells, then as single cells, then as chunks of particles that search in HBM.
// ------------------------------------------------------------------------------------------
constexpr uint32_t kEntryDirect = 1u << 12;                 // particles searched for directly: e.w + i
constexpr uint32_t kEntrySparse = 1u;                       // ... their slots at sparse[e.w + i]
constexpr int kMaxBox = 4;                                  // cells per side of a box
constexpr int kMaxHalo = kMaxBox + 2;
constexpr int kMaxCells = kMaxHalo * kMaxHalo * kMaxHalo;   // of a box and its halo

// (first slot, count) of a cell, inside the scene whatever a failed scan left in the ranges.
__device__ __forceinline__ uint2 cell_range_in(const uint2* __restrict__ range, uint32_t cell, uint32_t p_off,
                                               uint32_t n) {
    uint2 rg = range[cell];
    if (rg.x - p_off > n) return make_uint2(p_off, 0u);
    rg.y = min(rg.y, p_off + n - rg.x);
    return rg;
}

// Slots of the cells [x0, x1] x {y} x {z} (consecutive cells of a row hold consecutive slots).
__device__ __forceinline__ uint2 row_slots(const SceneDesc& d, const uint2* __restrict__ range, int x0, int x1, int y,
                                           int z) {
    const int R = d.c.R;
    const uint2* row = range + d.c_off + ((size_t)z * R + y) * R;
    const uint2 a = cell_range_in(row, (uint32_t)x0, d.p_off, d.c.n);
    const uint2 b = cell_range_in(row, (uint32_t)x1, d.p_off, d.c.n);
    const uint32_t end = b.x + b.y;
    return make_uint2(a.x, end > a.x ? end - a.x : 0u);
}

__device__ __forceinline__ void list_tile(const TileWork& T, uint32_t* __restrict__ error_flag, const uint4& e) {
    const uint32_t at = atomicAdd(T.count, 1u);
    if (at < T.cap)
        T.tiles[at] = e;
    else
        atomicOr(error_flag, 2u);  // cannot happen when the scan succeeded
}

// A box's lanes, 64 at a time, have a chunk of list memory each: the box's are e.w, e.w + 1, ...
__device__ __forceinline__ uint32_t box_chunks(uint32_t particles, int nx, int ny) {
    return (particles + 3u * (uint32_t)(nx * ny) + 63u) / 64u;  // columns of whole groups of four lanes
}

__device__ __forceinline__ uint4 box_entry(int x, int y, int z, int nx, int ny, int nz, uint32_t s, uint32_t chunk) {
    return make_uint4((uint32_t)x | (uint32_t)y << 10 | (uint32_t)z << 20,
                      (uint32_t)nx | (uint32_t)ny << 4 | (uint32_t)nz << 8,
                      s, chunk);
}

// A box of at most 2x2x2 cells that does not fit LDS: its cells one by one, or a cell's particles in
// chunks (one thread's work; dense clusters only).
__device__ __forceinline__ void list_cells(const SceneDesc& d, const uint2* __restrict__ range, int x, int y, int z,
                                           int nx, int ny, int nz, uint32_t s, const TileWork& T,
                                           uint32_t* __restrict__ error_flag) {
    const int R = d.c.R;
#pragma unroll 1
    for (int k = z; k < min(z + nz, R); ++k)
#pragma unroll 1
        for (int j = y; j < min(y + ny, R); ++j)
#pragma unroll 1
            for (int i = x; i < min(x + nx, R); ++i) {
                const uint2 slots = row_slots(d, range, i, i, j, k);
                if (slots.y == 0) continue;
                uint32_t all = 0;
                for (int r = 0; r < 9; ++r) {
                    const int cy = j + r % 3 - 1, cz = k + r / 3 - 1;
                    if (cy >= 0 && cz >= 0 && cy < R && cz < R)
                        all += row_slots(d, range, max(i - 1, 0), min(i + 2, R) - 1, cy, cz).y;
                }
                if (all <= T.rec_cap) {
                    const uint32_t chunk = atomicAdd(T.count + kListCount, box_chunks(slots.y, 1, 1));
                    list_tile(T, error_flag, box_entry(i, j, k, 1, 1, 1, s, chunk));
                } else {
                    for (uint32_t a = 0; a < slots.y; a += T.chunk)
                        list_tile(T, error_flag,
                                  make_uint4(0u, kEntryDirect | min(T.chunk, slots.y - a) << 13, s, slots.x + a));
                }
            }
}

// Records of a box and of the box with its halo, by LANES lanes: lane `row` of the group takes one halo
// row (two dependent loads for the whole box).
template <int LANES>
__device__ __forceinline__ uint2 box_records_by(const SceneDesc& d, const uint2* __restrict__ range, int row, bool any,
                                                int x, int y, int z, int nx, int ny, int nz) {
    const int R = d.c.R, ry = row % (ny + 2), rz = row / (ny + 2), cy = y - 1 + ry, cz = z - 1 + rz;
    uint32_t own = 0, all = 0;
    const bool in = any && rz < nz + 2 && cy >= 0 && cz >= 0 && cy < R && cz < R;
    if (in && ry > 0 && rz > 0 && ry <= ny && rz <= nz) own = row_slots(d, range, x, min(x + nx, R) - 1, cy, cz).y;
#pragma unroll
    for (int m = LANES / 2; m >= 1; m >>= 1) own += __shfl_xor(own, m);
    if (own == 0) return make_uint2(0u, 0u);  // most boxes of a large grid: their halo is not read
    if (in) all = row_slots(d, range, max(x - 1, 0), min(x + nx + 1, R) - 1, cy, cz).y;
#pragma unroll
    for (int m = LANES / 2; m >= 1; m >>= 1) all += __shfl_xor(all, m);
    return make_uint2(own, all);
}

// Classifies S.tper base boxes per workgroup.  Boxes that hold particles are appended in order within a
// workgroup (one atomic per workgroup: atomics on the one counter serialise at about 11 ns each); one
// whose halo does not fit LDS is split by a wave.
template <int LANES>
__device__ __forceinline__ void classify_boxes(const Scenes& S, const uint2* __restrict__ range, const TileWork& T,
                                               uint32_t* __restrict__ error_flag, uint32_t b) {
    __shared__ uint2 s_rec[kTileBlock];  // records of the box, of the box and its halo
    __shared__ uint3 s_wave[kTileBlock / 64], s_base;  // boxes, slots of sparse ones, list chunks
    const uint32_t s = scene_of(S.scene_tblk, S.num_scenes, b);
    const SceneDesc& d = S.desc[s];
    const int R = d.c.R, bx = (int)S.bx, by = (int)S.by, bz = (int)S.bz;
    const uint32_t first = (b - S.tblk[s]) * S.tper;
    auto origin = [&](uint32_t t, int& x, int& y, int& z) {
        x = (int)(t % d.tnx) * bx;
        y = (int)(t / d.tnx % d.tny) * by;
        z = (int)(t / (d.tnx * d.tny)) * bz;
    };
    int x, y, z;
    // four boxes' loads in flight
    for (uint32_t k0 = threadIdx.x / LANES; k0 < S.tper; k0 += 4 * (kTileBlock / LANES)) {
        uint2 rec[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t k = k0 + u * (kTileBlock / LANES);
            origin(first + k, x, y, z);
            rec[u] = box_records_by<LANES>(d, range, (int)(threadIdx.x % LANES), k < S.tper && first + k < d.ntiles,
                                           x, y, z, bx, by, bz);
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t k = k0 + u * (kTileBlock / LANES);
            if (k < S.tper && threadIdx.x % LANES == 0) s_rec[k] = rec[u];
        }
    }
    __syncthreads();
    const uint2 rec = threadIdx.x < S.tper ? s_rec[threadIdx.x] : make_uint2(0u, 0u);
    const bool few = rec.x != 0 && rec.y <= T.sparse_max;
    const bool fits = rec.x != 0 && !few && rec.y <= T.rec_cap;
    const unsigned long long m = __ballot(fits);
    const unsigned lane = lane_id(), wave = threadIdx.x >> 6;
    const uint32_t take = few ? rec.x : 0u, lists = fits ? box_chunks(rec.x, bx, by) : 0u;
    uint32_t incl = take, lists_incl = lists;
#pragma unroll
    for (int dd = 1; dd < 64; dd <<= 1) {
        const uint32_t t = __shfl_up(incl, dd), u = __shfl_up(lists_incl, dd);
        if ((int)lane >= dd) {
            incl += t;
            lists_incl += u;
        }
    }
    if (lane == 63) s_wave[wave] = make_uint3((uint32_t)__popcll(m), incl, lists_incl);
    __syncthreads();
    uint32_t before = 0, listed = 0, sparse = 0, list_chunks = 0;
    uint32_t sparse_before = incl - take, chunk = lists_incl - lists;
    for (unsigned w = 0; w < kTileBlock / 64; ++w) {
        before += w < wave ? s_wave[w].x : 0u;
        sparse_before += w < wave ? s_wave[w].y : 0u;
        chunk += w < wave ? s_wave[w].z : 0u;
        listed += s_wave[w].x;
        sparse += s_wave[w].y;
        list_chunks += s_wave[w].z;
    }
    if (threadIdx.x == 0) {
        // the scene's sparse slots start at its first particle's place
        const bool one = S.num_scenes == 1;
        const unsigned long long add = (unsigned long long)(one ? sparse : 0u) << 32 | listed;
        const unsigned long long old = add ? atomicAdd(reinterpret_cast<unsigned long long*>(T.count), add) : 0ull;
        s_base.x = (uint32_t)old;
        s_base.y = one ? (uint32_t)(old >> 32)
                       : (sparse ? d.p_off + atomicAdd(T.count + kSceneSparse + s, sparse) : 0u);
    }
    if (threadIdx.x == 64) s_base.z = list_chunks ? atomicAdd(T.count + kListCount, list_chunks) : 0u;
    if (threadIdx.x < S.tper) s_rec[threadIdx.x] = make_uint2(few ? 0x80000000u | sparse_before : rec.x, rec.y);
    __syncthreads();
    if (fits) {
        const uint32_t at = s_base.x + before + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        origin(first + threadIdx.x, x, y, z);
        if (at < T.cap)
            T.tiles[at] = box_entry(x, y, z, min(bx, R - x), min(by, R - y), min(bz, R - z), s, s_base.z + chunk);
        else
            atomicOr(error_flag, 2u);
    }
    if (sparse != 0u) {
        // a few lanes a box: lane `row` lists the particles of one row
        for (uint32_t k = threadIdx.x / LANES; k < S.tper; k += kTileBlock / LANES) {
            const uint32_t at = s_rec[k].x;
            if (!(at & 0x80000000u)) continue;  // the same for the box's lanes
            origin(first + k, x, y, z);
            const int row = (int)(threadIdx.x % LANES), cy = y + row % by, cz = z + row / by;
            uint2 slots = make_uint2(0u, 0u);
            if (row < by * bz && cy < R && cz < R) slots = row_slots(d, range, x, min(x + bx, R) - 1, cy, cz);
            uint32_t end = slots.y;
#pragma unroll
            for (int dd = 1; dd < LANES; dd <<= 1) {
                const uint32_t t = __shfl_up(end, dd, LANES);
                if (row >= dd) end += t;
            }
            const uint32_t to = s_base.y + (at & 0x7fffffffu) + end - slots.y;
            for (uint32_t i = 0; i < slots.y; ++i)
                if (to + i < S.total_particles) T.sparse[to + i] = slots.x + i;
        }
    }
    const bool split = bx > 2 || by > 2 || bz > 2;
    for (uint32_t k = split ? wave : threadIdx.x; k < S.tper; k += split ? kTileBlock / 64 : kTileBlock) {
        const uint2 r = s_rec[k];
        if (r.x == 0 || (r.x & 0x80000000u) || r.y <= T.rec_cap) continue;
        origin(first + k, x, y, z);
        if (!split) {
            list_cells(d, range, x, y, z, bx, by, bz, s, T, error_flag);
            continue;
        }
        // parts of 2x2x2, 16 lanes each (wave-uniform loop)
        const int px = (bx + 1) / 2, py = (by + 1) / 2, parts = px * py * ((bz + 1) / 2);
        for (int q0 = 0; q0 < parts; q0 += 4) {
            const int q = q0 + (int)(lane / 16u);
            const int i = x + q % px * 2, j = y + q / px % py * 2, l = z + q / (px * py) * 2;
            // a part ends with its box
            const int ex = min(min(2, x + bx - i), R - i), ey = min(min(2, y + by - j), R - j);
            const int ez = min(min(2, z + bz - l), R - l);
            const bool any = q < parts && ex > 0 && ey > 0 && ez > 0;
            const uint2 part = box_records_by<16>(d, range, (int)(lane % 16u), any, i, j, l, ex, ey, ez);
            if (lane % 16u == 0 && part.x != 0) {
                if (part.y <= T.rec_cap) {
                    const uint32_t chunk = atomicAdd(T.count + kListCount, box_chunks(part.x, ex, ey));
                    list_tile(T, error_flag, box_entry(i, j, l, ex, ey, ez, s, chunk));
                } else {
                    list_cells(d, range, i, j, l, ex, ey, ez, s, T, error_flag);
                }
            }
        }
    }
}

// A staged box: its halo's cells with z fastest, each cell's records consecutive in LDS.  The three cells
// (dx, dy, -1..1) about a cell are then one window, in the reference's order (dz innermost).
struct BoxTable {
    uint32_t cell[kMaxCells];             // first record | end << 16
    uint32_t slot[kMaxCells];             // slot of a cell's record r: r + slot
    uint32_t own[kMaxBox * kMaxBox + 4];  // lanes before each of the box's columns (whole groups of four), then all
    uint32_t records;
    uint32_t pad[3];
};
static_assert(sizeof(BoxTable) == kTileTableBytes && sizeof(BoxTable) % 16 == 0, "copied in 16-byte pieces");

struct BoxShared : BoxTable {
    uint32_t wave_sum[4];
    uint32_t rho;                    // largest density of the box
};

struct Box {
    int x, y, z, nx, ny, nz;  // first cell and cells per side
    int hx, hy, hz;           // with the halo
};

__device__ __forceinline__ Box box_of(const uint4& e) {
    Box b;
    b.x = (int)(e.x & 1023u);
    b.y = (int)(e.x >> 10 & 1023u);
    b.z = (int)(e.x >> 20 & 1023u);
    b.nx = (int)(e.y & 15u);
    b.ny = (int)(e.y >> 4 & 15u);
    b.nz = (int)(e.y >> 8 & 15u);
    b.hx = b.nx + 2;
    b.hy = b.ny + 2;
    b.hz = b.nz + 2;
    return b;
}

// i / d for i < 256, d <= 36
__device__ __forceinline__ int small_div(int i, int d) {
    return (int)((uint32_t)i * (uint32_t)((65536 + d - 1) / d) >> 16);
}

// Halo cell (x fastest) i of a box, as its index in the table (z fastest).
__device__ __forceinline__ int table_cell(const Box& b, int i) {
    const int r = small_div(i, b.hx), z = small_div(r, b.hy);
    return ((i - r * b.hx) * b.hy + (r - z * b.hy)) * b.hz + z;
}
__device__ __forceinline__ int own_column(const Box& b, int q) {  // table index of column q's first halo cell
    const int x = small_div(q, b.ny);
    return ((x + 1) * b.hy + (q - x * b.ny + 1)) * b.hz;
}

// Lanes before each of the box's columns, columns rounded up to whole groups of four lanes (by wave 0).
__device__ __forceinline__ void box_lanes(BoxShared& sh, const Box& b) {
    const int lane = (int)threadIdx.x, ncol = b.nx * b.ny;
    if (lane < 64) {
        uint32_t n = 0;
        if (lane < ncol) {
            const int c = own_column(b, lane);
            n = ((sh.cell[c + b.nz] >> 16) - (sh.cell[c + 1] & 0xffffu) + 3u) & ~3u;
        }
        uint32_t incl = n;
#pragma unroll
        for (int dd = 1; dd < 16; dd <<= 1) {
            const uint32_t t = __shfl_up(incl, dd);
            if (lane >= dd) incl += t;
        }
        const uint32_t all = (uint32_t)__shfl((int)incl, ncol - 1);
        if (lane < kMaxBox * kMaxBox + 4) sh.own[lane] = lane < ncol ? incl - n : all;
    }
}

// Cell table of a box: every thread takes a halo cell (out-of-grid cells are empty), a prefix sum over the
// counts gives each its records in LDS.  BLOCK threads take ceil(216 / BLOCK) cells each, in order.
template <int BLOCK>
__device__ __forceinline__ void box_cells(BoxShared& sh, const Box& b, const SceneDesc& d,
                                          const uint2* __restrict__ range) {
    constexpr int kPer = (kMaxCells + BLOCK - 1) / BLOCK;
    const int tid = threadIdx.x, ncell = b.hx * b.hy * b.hz, R = d.c.R;
    const unsigned lane = lane_id(), wave = threadIdx.x >> 6;
    for (int i = tid; i < ncell; i += BLOCK) {  // read along x
        const int r = small_div(i, b.hx), cx = b.x - 1 + (i - r * b.hx);
        const int rz = small_div(r, b.hy), cy = b.y - 1 + (r - rz * b.hy), cz = b.z - 1 + rz;
        uint2 rg = make_uint2(0u, 0u);
        if (cx >= 0 && cy >= 0 && cz >= 0 && cx < R && cy < R && cz < R)
            rg = cell_range_in(range + d.c_off, (uint32_t)((cz * R + cy) * R + cx), d.p_off, d.c.n);
        const int at = table_cell(b, i);
        sh.cell[at] = rg.y;
        sh.slot[at] = rg.x;
    }
    __syncthreads();
    uint32_t cnt[kPer], sum = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const int i = tid * kPer + k;
        cnt[k] = i < ncell ? sh.cell[i] : 0u;
        sum += cnt[k];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int dd = 1; dd < 64; dd <<= 1) {
        const uint32_t t = __shfl_up(incl, dd);
        if ((int)lane >= dd) incl += t;
    }
    if (lane == 63 && wave < 4) sh.wave_sum[wave] = incl;
    __syncthreads();
    uint32_t base = incl - sum, total = 0;
#pragma unroll
    for (unsigned w = 0; w < 4 && w < BLOCK / 64; ++w) {
        base += w < wave ? sh.wave_sum[w] : 0u;
        total += sh.wave_sum[w];
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const int i = tid * kPer + k;
        if (i < ncell) {
            sh.cell[i] = base | (base + cnt[k]) << 16;
            sh.slot[i] -= base;
        }
        base += cnt[k];
    }
    if (tid == 0) sh.records = total;
    __syncthreads();
    box_lanes(sh, b);
    __syncthreads();
}

// Tables of the listed boxes, one workgroup each.
__device__ __forceinline__ void form_tables(const Scenes& S, const uint2* __restrict__ range, const TileWork& T,
                                            uint32_t block, uint32_t nblocks) {
    __shared__ BoxShared sh;
    const uint32_t listed = min(min(*T.count, T.cap), T.table_cap);
    if (block == 0 && S.num_scenes > 1) {
        // several scenes' sparse particles: entries of a scene each, from the work list's end down
        for (uint32_t s = threadIdx.x; s < S.num_scenes; s += kHashBlock) {
            const SceneDesc& d = S.desc[s];
            const uint32_t n = min(T.count[kSceneSparse + s], d.c.n), chunks = (n + T.chunk - 1) / T.chunk;
            const uint32_t at = chunks ? atomicAdd(T.count + kSceneSparse - 1, chunks) : 0u;
            for (uint32_t k = 0; k < chunks && at + k < T.cap; ++k)
                T.tiles[T.cap - 1u - at - k] =
                    make_uint4(0u, kEntryDirect | kEntrySparse | min(T.chunk, n - k * T.chunk) << 13, s,
                               d.p_off + k * T.chunk);
        }
    }
    for (uint32_t item = block; item < listed; item += nblocks) {
        const uint4 e = T.tiles[item];
        if (e.y & kEntryDirect) continue;
        const Box b = box_of(e);
        box_cells<kHashBlock>(sh, b, S.desc[e.z], range);
        for (uint32_t k = threadIdx.x; k < sizeof(BoxTable) / 16; k += kHashBlock)
            reinterpret_cast<uint4*>(&reinterpret_cast<BoxTable*>(T.tables)[item])[k] =
                reinterpret_cast<const uint4*>(static_cast<const BoxTable*>(&sh))[k];
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------------
// 3. place: slot = first slot of the cell + arrival rank (reorder.comp:38-43 without the copy).
// ------------------------------------------------------------------------------------------
// The first particle to arrive in a cell of more than kGatherDirectMax also lists the cell for the
// leading workgroups of k_gather, which sort its input indices instead of ranking them one by one.
// TILES: further workgroups form the tile passes' work list (their code costs the others 1.6 us of 7.5 on a
// million particles, so contexts without those passes run none of it).
template <bool TILES>
__global__ __launch_bounds__(kHashBlock) void k_place(Scenes S, const uint32_t* __restrict__ key,
                                                      const uint32_t* __restrict__ rank,
                                                      const uint2* __restrict__ range,
                                                      uint32_t* __restrict__ slot_tmp, uint2* __restrict__ crowd,
                                                      uint32_t* __restrict__ crowd_count, uint32_t crowd_cap,
                                                      uint32_t* __restrict__ error_flag, TileWork tiles) {
    const uint32_t b = blockIdx.x;
    if (TILES && b >= S.blocks256) {
        if ((S.by + 2) * (S.bz + 2) <= 16)
            classify_boxes<16>(S, range, tiles, error_flag, b - S.blocks256);
        else
            classify_boxes<32>(S, range, tiles, error_flag, b - S.blocks256);
        return;
    }
    const uint32_t s = scene_of(S.scene256, S.num_scenes, b);
    const SceneDesc& d = S.desc[s];
    const uint32_t lt = (b - S.blk256[s]) * kHashBlock + threadIdx.x;
    if (lt >= d.c.n) return;
    const uint32_t i = d.p_off + lt;
    const uint32_t k = key[i];
    const uint2 rg = range[d.c_off + k];
    const uint32_t r = rank[i];
    const uint32_t slot = rg.x + r;
    if (slot - d.p_off < d.c.n) slot_tmp[slot] = i;  // always true when the scan succeeded
    if (rg.y > kGatherDirectMax && r == 0u) {       // one entry per crowded cell
        const uint32_t at = atomicAdd(crowd_count, 1u);
        if (at < crowd_cap)
            crowd[at] = make_uint2(d.c_off + k, s);
        else
            atomicOr(error_flag, 2u);  // cannot happen when the scan succeeded
    }
}

// ------------------------------------------------------------------------------------------
// 4. stable rank + gather: the particle that arrived at slot t moves to the cell's first slot +
//    (number of particles of its cell with a smaller input index), so every cell keeps input
//    order; the record is copied there (reorder.comp:44) and the cell index kept beside it.
//    Counting costs one pass over the cell per particle, so only cells of at most
//    kGatherDirectMax particles are ranked this way.  k_place lists each more crowded cell, and
//    the first kCrowdBlocks workgroups of k_gather sort its input indices instead.
// ------------------------------------------------------------------------------------------
// Moves the particle with input index i to slot dst of the sorted buffer (reorder.comp:44).
__device__ __forceinline__ void move_record(uint32_t i, uint32_t dst, uint32_t k, const float4* __restrict__ posrho_in,
                                            const float4* __restrict__ velp_in, float4* __restrict__ posrho_out,
                                            float4* __restrict__ velp_out, uint32_t* __restrict__ sorted,
                                            uint32_t* __restrict__ skey, const uint32_t* __restrict__ id_in,
                                            uint32_t* __restrict__ id_out, uint32_t* __restrict__ div_flags) {
    sorted[dst] = i;
    skey[dst] = k;
    const float4 v = velp_in[i];
    posrho_out[dst] = posrho_in[i];
    velp_out[dst] = v;
    if (id_out) id_out[dst] = id_in[i];
    // velocities are operands of the force pass's quotients (the density pass checks the rest)
    if (!(div_operand(v.x) && div_operand(v.y) && div_operand(v.z))) atomicOr(div_flags, kDivUnsafe);
}

// Crowded cells: one workgroup per listed cell (a loop over the list with stride nblocks, whose
// length k_place left in crowd_count) sorts the cell's input indices, slot_tmp[first .. first + c),
// in ascending order: chunks of kCrowdChunk by a bitonic sort in LDS, then merge passes between
// slot_tmp and sorted over the same slots (each element's place in the merged run is its index in
// its own run plus the number of smaller elements of the other run, by binary search; indices are
// unique).  The particle with the r-th smallest index moves to slot first + r, exactly the rank
// k_gather would give it.  Every loop is bounded by the cell's size: O(c log^2 c) work per cell.
constexpr uint32_t kCrowdChunk = 4096;
constexpr unsigned kCrowdBlocks = 32;

__device__ __forceinline__ uint32_t count_below(const uint32_t* __restrict__ run, uint32_t n, uint32_t x) {
    uint32_t a = 0, b = n;
    while (a < b) {
        const uint32_t m = (a + b) >> 1;
        if (run[m] < x)
            a = m + 1;
        else
            b = m;
    }
    return a;
}

__device__ __forceinline__ void gather_crowded_cells(
    const Scenes& S, const uint2* __restrict__ crowd, const uint32_t* __restrict__ crowd_count, uint32_t crowd_cap,
    uint32_t* __restrict__ slot_tmp, const uint2* __restrict__ range, const float4* __restrict__ posrho_in,
    const float4* __restrict__ velp_in, float4* __restrict__ posrho_out, float4* __restrict__ velp_out,
    uint32_t* __restrict__ sorted, uint32_t* __restrict__ skey, const uint32_t* __restrict__ id_in,
    uint32_t* __restrict__ id_out, uint32_t* __restrict__ div_flags, uint32_t* s_v, uint32_t block,
    uint32_t nblocks) {
    const uint32_t listed = min(*crowd_count, crowd_cap);
    for (uint32_t item = block; item < listed; item += nblocks) {
        const uint2 e = crowd[item];  // (context cell, scene)
        const SceneDesc& d = S.desc[e.y];
        const uint2 rg = range[e.x];
        const uint32_t first = rg.x, lim = d.p_off + d.c.n;
        if (first < d.p_off || first >= lim) continue;  // only after a failed scan
        const uint32_t c = min(rg.y, lim - first);
        uint32_t* src = slot_tmp + first;
        uint32_t* dst = sorted + first;
        for (uint32_t lo = 0; lo < c; lo += kCrowdChunk) {
            const uint32_t m = min(c - lo, kCrowdChunk);
            uint32_t P = 1;
            while (P < m) P <<= 1;
            for (uint32_t j = threadIdx.x; j < P; j += kHashBlock) s_v[j] = j < m ? src[lo + j] : 0xFFFFFFFFu;
            __syncthreads();
            for (uint32_t k = 2; k <= P; k <<= 1) {
                for (uint32_t j = k >> 1; j > 0; j >>= 1) {
                    for (uint32_t a = threadIdx.x; a < P; a += kHashBlock) {
                        const uint32_t b = a ^ j;
                        if (b > a) {
                            const uint32_t x = s_v[a], y = s_v[b];
                            if ((x > y) == ((a & k) == 0)) {
                                s_v[a] = y;
                                s_v[b] = x;
                            }
                        }
                    }
                    __syncthreads();
                }
            }
            for (uint32_t j = threadIdx.x; j < m; j += kHashBlock) src[lo + j] = s_v[j];
            __syncthreads();
        }
        for (uint32_t w = kCrowdChunk; w < c; w <<= 1) {
            for (uint32_t j = threadIdx.x; j < c; j += kHashBlock) {
                const uint32_t run = j / w;
                const uint32_t lo = (run & ~1u) * w;
                const uint32_t mid = min(lo + w, c), hi = min(lo + 2 * w, c);
                const uint32_t x = src[j];
                const uint32_t at = (run & 1u) == 0u ? (j - lo) + count_below(src + mid, hi - mid, x)
                                                     : (j - mid) + count_below(src + lo, mid - lo, x);
                dst[lo + at] = x;
            }
            __syncthreads();
            uint32_t* tmp = src;
            src = dst;
            dst = tmp;
        }
        const uint32_t k = e.x - d.c_off;
        for (uint32_t r = threadIdx.x; r < c; r += kHashBlock)
            move_record(src[r], first + r, k, posrho_in, velp_in, posrho_out, velp_out, sorted, skey, id_in, id_out,
                        div_flags);
        __syncthreads();  // the next cell reuses the LDS chunk
    }
}

template <bool TILES>  // as for k_place: further workgroups form the cell tables
__global__ __launch_bounds__(kHashBlock) void k_gather(Scenes S, uint32_t* __restrict__ slot_tmp,
                                                       const uint32_t* __restrict__ key,
                                                       const uint2* __restrict__ range,
                                                       const float4* __restrict__ posrho_in,
                                                       const float4* __restrict__ velp_in,
                                                       float4* __restrict__ posrho_out, float4* __restrict__ velp_out,
                                                       uint32_t* __restrict__ sorted, uint32_t* __restrict__ skey,
                                                       const uint32_t* __restrict__ id_in,
                                                       uint32_t* __restrict__ id_out,
                                                       uint32_t* __restrict__ div_flags,
                                                       const uint2* __restrict__ crowd,
                                                       const uint32_t* __restrict__ crowd_count, uint32_t crowd_cap,
                                                       TileWork tiles) {
    __shared__ uint32_t s_v[kCrowdChunk];
    if (blockIdx.x < kCrowdBlocks) {  // the leading workgroups take the crowded cells k_place listed
        gather_crowded_cells(S, crowd, crowd_count, crowd_cap, slot_tmp, range, posrho_in,
                             velp_in, posrho_out, velp_out, sorted, skey, id_in, id_out, div_flags, s_v, blockIdx.x,
                             kCrowdBlocks);
        return;
    }
    // kCrowdBlocks is a multiple of the XCD count, so block b still runs on XCD b mod 8
    if (TILES && blockIdx.x >= kCrowdBlocks + S.blocks256) {
        form_tables(S, range, tiles, blockIdx.x - kCrowdBlocks - S.blocks256, gridDim.x - kCrowdBlocks - S.blocks256);
        return;
    }
    const uint32_t b = xcd_block(blockIdx.x - kCrowdBlocks, S.blocks256);
    const uint32_t s = scene_of(S.scene256, S.num_scenes, b);
    const SceneDesc& d = S.desc[s];
    const uint32_t lt = (b - S.blk256[s]) * kHashBlock + threadIdx.x;
    if (lt >= d.c.n) return;
    const uint32_t t = d.p_off + lt;
    const uint32_t lim = d.p_off + d.c.n;
    const uint32_t i = slot_tmp[t];
    if (i - d.p_off >= d.c.n) return;  // only after a failed scan (error flag set)
    const uint32_t k = key[i];
    const uint2 rg = range[d.c_off + k];
    if (rg.y > kGatherDirectMax) return;  // a crowded cell: sorted by the leading workgroups
    const uint32_t end = min(rg.x + rg.y, lim);
    uint32_t r = 0;
    for (uint32_t u = rg.x; u < end; ++u) r += (slot_tmp[u] < i) ? 1u : 0u;
    const uint32_t dst = rg.x + r;
    if (dst >= lim) return;
    move_record(i, dst, k, posrho_in, velp_in, posrho_out, velp_out, sorted, skey, id_in, id_out, div_flags);
}

// ------------------------------------------------------------------------------------------
// Neighbour search shared by the density and the force pass.
//
// Each lane owns one particle.  The 27 neighbour cells are visited in NEIGHBORHOOD order with a
// wave-uniform cell loop; inside a cell each lane walks its own slot range CHUNK slots at a time
// (CHUNK loads in flight).  Candidate tests are branch-free: every candidate is written to the
// lane's next entry of an LDS list and the entry count advances by the test's outcome.  The lists
// are drained at the end, (PLANE_DRAIN) after every dx plane, and whenever one lane's list could
// overflow on its next chunk; every lane drains then, not only the full ones.  The per-neighbour
// arithmetic thus runs over compacted entries with all lanes busy instead of under a mask where
// ~15% of the lanes accept a given candidate.  Entries are drained in enumeration order, so
// every sum is formed exactly as the reference forms it, and the result does not depend on
// BLOCK, CAP, CHUNK or PLANE_DRAIN (the tuning knobs of the passes) or on when the lists drain.
// ------------------------------------------------------------------------------------------
// Pointers into LDS (32-bit addresses, so list arithmetic stays 32-bit).
template <typename T>
using lds_ptr = __attribute__((address_space(3))) T*;

template <int BLOCK, int CAP, int CHUNK, bool PLANE_DRAIN, typename Entry, typename Drain>
__device__ __forceinline__ void search_neighbours(uint32_t key, uint32_t t, uint32_t limit, float px, float py,
                                                  float pz, const float4* __restrict__ pos,
                                                  const uint2* __restrict__ range, const StepConsts& c,
                                                  lds_ptr<Entry> list, Drain& drain_fn) {
    static_assert(CAP >= CHUNK, "list must hold a chunk");
    static_assert(CHUNK <= (int)kRecordPad + 1, "chunked loads may run CHUNK - 1 records past a cell");
    // `next` is the lane's next free list entry; the list holds (next - list) / BLOCK entries
    lds_ptr<Entry> next = list;
    const lds_ptr<Entry> full = list + (CAP - CHUNK) * BLOCK;  // past this a chunk might not fit
    auto drain = [&]() {
        drain_fn((int)((next - list) / BLOCK));
        next = list;
    };
    auto visit = [&](uint32_t start, uint32_t end, auto own) {
        // the chunks of a cell run in step across the wave: every lane visiting the cell takes part
        // in each iteration (with its own slots, or none once its range is done), so when one list
        // fills, every lane drains with it instead of waiting on a drain of a few lanes
        for (uint32_t u = start; __any(u < end); u += CHUNK) {
            if (__any(next > full)) drain();
            if (u >= end) continue;
            const uint32_t left = end - u;  // slots of the cell from u on (>= 1 here): u + j is one iff j < left
            // slots past the cell are loaded (the buffers are padded) and rejected below
            const float4* q = pos + u;
            float4 r[CHUNK];
#pragma unroll
            for (int j = 0; j < CHUNK; ++j) r[j] = q[j];
#pragma unroll
            for (int j = 0; j < CHUNK; ++j) {
                const float rx = px - r[j].x, ry = py - r[j].y, rz = pz - r[j].z;
                const float d2 = (rx * rx + ry * ry) + rz * rz;
                // dist < h  <=>  !(d2 >= cut2), NaN included (sqrtf(NaN) >= h is false)
                bool ok = ((uint32_t)j < left) & !(d2 >= c.cut2);
                if constexpr (decltype(own)::value) ok &= (u + (uint32_t)j != t);
                if constexpr (std::is_same<Entry, float>::value)
                    *next = d2;  // density: squared distance
                else
                    *next = u + (uint32_t)j;  // force pass: the neighbour's slot
                next += ok ? BLOCK : 0;
                // keep `next` an address in one register (not base + offset: one add fewer per candidate)
                asm("" : "+v"(next));
            }
        }
    };
    auto end_plane = [&]() {
        if (PLANE_DRAIN) drain();
    };
    for_each_neighbour_cell(key, range, c, limit, visit, end_plane);
    drain();
}

// ------------------------------------------------------------------------------------------
// 5. density + pressure (density.comp:81-137), in place on the sorted buffer.  The LDS list
//    holds each accepted neighbour's squared distance.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ float wall_density(const StepConsts& c, float x, float y, float z) {
    // density.comp:57-79; the z branch's else-test reads p.y (line 74)
    float d = 0.0f;
    if (x < c.h) d += c.m * poly6(c, x);
    else if (x > c.size_minus_h) d += c.m * poly6(c, c.size - x);
    if (y < c.h) d += c.m * poly6(c, y);
    else if (y > c.size_minus_h) d += c.m * poly6(c, c.size - y);
    if (z < c.h) d += c.m * poly6(c, z);
    else if (y > c.size_minus_h) d += c.m * poly6(c, c.size - z);
    return d * 4.0f;
}

__device__ __forceinline__ float eos(const StepConsts& c, float rho) {
    if (c.eos == WC_EOS_LINEAR) return c.p0 + c.k * (rho - c.rho0);
    const float x = rho / c.rho0;
    return c.p0 + c.k * (((x * x) * x) - 1.0f);
}

// LIST: the LDS list holds slots instead; the drain recomputes each squared distance (the same
// expression, so the same bits) and also appends the slot to the particle's neighbour list in
// HBM, loading neighbour k + 1's position while neighbour k is summed.
template <int BLOCK, int CAP, int CHUNK, bool PLANE_DRAIN, bool LIST>
__global__ __launch_bounds__(BLOCK) void k_density(Scenes S, float4* __restrict__ posrho, float4* __restrict__ velp,
                                                   const uint32_t* __restrict__ skey,
                                                   const uint2* __restrict__ range, uint32_t* __restrict__ rho_max,
                                                   uint32_t* __restrict__ nlist, uint32_t* __restrict__ ncount) {
    using Entry = typename std::conditional<LIST, uint32_t, float>::type;
    __shared__ Entry s_list[CAP * BLOCK];
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAnd(&rho_max[1], ~kDivPending);
    const uint32_t b = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t s = scene_of(scene_table<BLOCK>(S), S.num_scenes, b);
    const SceneDesc& d = S.desc[s];
    // the constants by value: read through a reference, every LDS store of the neighbour loop
    // could alias them (generic pointers may point into LDS), and they were reloaded per chunk
    const StepConsts c = d.c;
    const uint32_t lt = (b - first_blocks<BLOCK>(S)[s]) * BLOCK + threadIdx.x;
    if (lt - __lane_id() >= c.n) return;  // the whole wave is past the scene's last particle
    const bool active = lt < c.n;
    float density = 0.0f;
    if (active) {
        const uint32_t t = d.p_off + lt;
        const float4 p = posrho[t];
        const lds_ptr<Entry> list = (lds_ptr<Entry>)s_list + threadIdx.x;
        float rho = c.m * poly6(c, 0.0f);
        uint32_t written = 0;  // LIST: neighbours found so far
        auto drain = [&](int cnt) {
            if constexpr (LIST) {
                if (cnt <= 0) return;
                uint32_t u = list[0];
                float4 q = posrho[u];
                for (int k = 0; k < cnt; ++k) {
                    const uint32_t un = list[(k + 1 < cnt ? k + 1 : k) * BLOCK];
                    const float4 qn = posrho[un];
                    const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
                    const float d2 = (rx * rx + ry * ry) + rz * rz;
                    rho += c.m * poly6(c, sqrtf(d2));
                    if (written < kNeighbourListMax) nlist[(size_t)written * S.total_particles + t] = u;
                    ++written;
                    u = un;
                    q = qn;
                }
            } else {
                for (int k = 0; k < cnt; ++k) rho += c.m * poly6(c, sqrtf(list[k * BLOCK]));
            }
        };
        search_neighbours<BLOCK, CAP, CHUNK, PLANE_DRAIN>(skey[t], t, d.p_off + c.n, p.x, p.y, p.z, posrho,
                                                          range + d.c_off, c, list, drain);
        if constexpr (LIST) ncount[t] = written <= kNeighbourListMax ? written : kListOverflow;
        const float wall = c.wall_density ? wall_density(c, p.x, p.y, p.z) : 0.0f;
        density = rho + wall;
        const float pressure = eos(c, rho);
        reinterpret_cast<float*>(posrho)[4 * (size_t)t + 3] = density;
        reinterpret_cast<float*>(velp)[4 * (size_t)t + 3] = pressure;
        // the other operands of the force pass's quotients (the sort checks the velocities)
        const bool ok = div_operand(p.x) && div_operand(p.y) && div_operand(p.z) && div_operand(pressure) &&
                        div_operand(density) && density != 0.0f;
        if (!ok) atomicOr(&rho_max[1], kDivUnsafe);
    }
    // largest density of the pass (positive floats order as their bit patterns; NaN ranks highest);
    // lanes past the scene's last particle take part as 0
    uint32_t bits = active ? __float_as_uint(density) & 0x7fffffffu : 0u;
    for (int k = 32; k >= 1; k >>= 1) bits = max(bits, (uint32_t)__shfl_xor((int)bits, k));
    if ((threadIdx.x & 63) == 0) atomicMax(rho_max, bits);
}

// ------------------------------------------------------------------------------------------
// 6. forces + symplectic Euler + cube boundary (update.comp:134-232): sorted buffer -> buffer 1.
// ------------------------------------------------------------------------------------------
struct V3 {
    float x, y, z;
};

template <bool FAST = false>
__device__ __forceinline__ V3 spiky(const StepConsts& c, float rx, float ry, float rz, float d) {
    const float a = c.h - d;
    const float s = a * a;
    if constexpr (FAST) {
        const float y = 1.0f / d;
        return V3{(s * quot(rx, d, y)) * c.spiky, (s * quot(ry, d, y)) * c.spiky, (s * quot(rz, d, y)) * c.spiky};
    }
    return V3{(s * (rx / d)) * c.spiky, (s * (ry / d)) * c.spiky, (s * (rz / d)) * c.spiky};
}

__device__ __forceinline__ V3 wall_forces(const StepConsts& c, float x, float y, float z) {
    // update.comp:71-100; vec3.length() is 3
    V3 f{0.0f, 0.0f, 0.0f};
    if (x < c.h) {
        const V3 w = spiky(c, 0.0f - x, y - y, z - z, 3.0f);
        f.x += w.x; f.y += w.y; f.z += w.z;
    } else if (x > c.size_minus_h) {
        const V3 w = spiky(c, c.size - x, y - y, z - z, 3.0f);
        f.x += w.x; f.y += w.y; f.z += w.z;
    }
    if (y < c.h) {
        const V3 w = spiky(c, x - x, 0.0f - y, z - z, 3.0f);
        f.x += w.x; f.y += w.y; f.z += w.z;
    } else if (y > c.size_minus_h) {
        const V3 w = spiky(c, x - x, c.size - y, z - z, 3.0f);
        f.x += w.x; f.y += w.y; f.z += w.z;
    }
    if (z < c.h) {
        const V3 w = spiky(c, x - x, y - y, 0.0f - z, 3.0f);
        f.x += w.x; f.y += w.y; f.z += w.z;
    } else if (z > c.size_minus_h) {
        const V3 w = spiky(c, x - x, y - y, c.size - z, 3.0f);
        f.x += w.x; f.y += w.y; f.z += w.z;
    }
    return V3{f.x * 0.01f, f.y * 0.01f, f.z * 0.01f};
}

__device__ __forceinline__ V3 mouse_force(const StepConsts& c, float px, float py, float pz, float pressure) {
    // update.comp:105-132
    const float o[3] = {c.cam[0], c.cam[1], c.cam[2]};
    float t1[3], t2[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float tmin = (0.0f - o[a]) / c.dir[a];
        const float tmax = (c.size - o[a]) / c.dir[a];
        t1[a] = fminf(tmin, tmax);
        t2[a] = fmaxf(tmin, tmax);
    }
    const float tnear = fmaxf(fmaxf(t1[0], t1[1]), t1[2]);
    const float tfar = fminf(fminf(t2[0], t2[1]), t2[2]);
    if (tnear > tfar) return V3{0.0f, 0.0f, 0.0f};
    const float tx = px - o[0], ty = py - o[1], tz = pz - o[2];
    const float cx = c.dir[1] * tz - ty * c.dir[2];
    const float cy = c.dir[2] * tx - tz * c.dir[0];
    const float cz = c.dir[0] * ty - tx * c.dir[1];
    const float dist = sqrtf((cx * cx + cy * cy) + cz * cz);
    if (dist > c.h) return V3{0.0f, 0.0f, 0.0f};
    const V3 w = spiky(c, tx, ty, tz, dist + 1e-16f);
    const float s = (-c.m) * pressure;
    return V3{(s * w.x) * 0.00001f, (s * w.y) * 0.00001f, (s * w.z) * 0.00001f};
}

__device__ __forceinline__ void integrate_axis(const StepConsts& c, float pf, float vf, float ext, float denom,
                                               float v0, float x0, float dt, float& vel, float& pos) {
    vf = vf * c.mu;
    const float force = (pf + vf) + ext;
    const float acc = force / denom;
    const float v = v0 + acc * dt;
    vel = fminf(fmaxf(v, -c.max_speed), c.max_speed);
    pos = x0 + vel * dt;
    if (pos < c.border) {
        vel = vel * -c.damping;
        pos = c.border;
    } else if (pos > c.hi) {
        vel = vel * -c.damping;
        pos = c.hi;
    }
}

// Pressure and viscosity contributions of one accepted neighbour (update.comp:178-187).
struct ForceSums {
    float pfx, pfy, pfz, vfx, vfy, vfz;

    // Returns the pair distance.  FAST: the quotients by rho_j, by 2 rho_j and by the distance
    // come from one reciprocal each (quot); the results are the same bits as with FAST false
    // whenever every operand passes div_operand.  A zero quotient may then carry the other sign,
    // which these sums cannot show: they start at +0, and x + (+-0) = x, +0 - (+-0) = +0.
    template <bool FAST>
    __device__ __forceinline__ float add(const StepConsts& c, const float4& p, const float4& pv, const float4& q,
                                         const float4& qv) {
        const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
        const float dist = sqrtf((rx * rx + ry * ry) + rz * rz);
        float iw = 0.0f, pressure;
        if constexpr (FAST) {
            iw = 1.0f / q.w;  // RN(1 / rho_j); RN(1 / (2 rho_j)) is half of it
            pressure = quot(pv.w + qv.w, 2.0f * q.w, iw * 0.5f);
        } else {
            pressure = (pv.w + qv.w) / (2.0f * q.w);
        }
        if (pressure > 0.0f) {
            const V3 sw = spiky<FAST>(c, rx, ry, rz, dist + 1e-16f);
            const float mp = c.m * pressure;
            pfx = pfx - mp * sw.x;
            pfy = pfy - mp * sw.y;
            pfz = pfz - mp * sw.z;
        }
        const float wv = (c.h - dist) * c.visc;
        if constexpr (FAST) {
            vfx = vfx + (c.m * quot(qv.x - pv.x, q.w, iw)) * wv;
            vfy = vfy + (c.m * quot(qv.y - pv.y, q.w, iw)) * wv;
            vfz = vfz + (c.m * quot(qv.z - pv.z, q.w, iw)) * wv;
        } else {
            vfx = vfx + (c.m * ((qv.x - pv.x) / q.w)) * wv;
            vfy = vfy + (c.m * ((qv.y - pv.y) / q.w)) * wv;
            vfz = vfz + (c.m * ((qv.z - pv.z) / q.w)) * wv;
        }
        return dist;
    }

    // The same sums with the square root and the reciprocals in their short forms: every operand
    // passes div_operand (positions pos_operand), so each step rounds as in add.  The pair pressure is
    // half the quotient by rho_j, exactly, and the half goes into the mass (a power of two).
    __device__ __forceinline__ void add_in_range(const StepConsts& c, const float4& p, const float4& pv,
                                                 const float4& q, const float4& qv) {
        const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
        const float dist = sqrt_in_range((rx * rx + ry * ry) + rz * rz);
        const float iw = rcp_in_range(q.w);
        const float twice = quot(pv.w + qv.w, q.w, iw);  // twice the pair pressure
        const float mp = twice > 0.0f ? (0.5f * c.m) * twice : 0.0f;
        const float dd = dist + 1e-16f;
        const float y = rcp_in_range(dd);
        const float a = c.h - dd;
        const float s = a * a;
        pfx = pfx - mp * ((s * quot(rx, dd, y)) * c.spiky);
        pfy = pfy - mp * ((s * quot(ry, dd, y)) * c.spiky);
        pfz = pfz - mp * ((s * quot(rz, dd, y)) * c.spiky);
        const float wv = (c.h - dist) * c.visc;
        vfx = vfx + (c.m * quot(qv.x - pv.x, q.w, iw)) * wv;
        vfy = vfy + (c.m * quot(qv.y - pv.y, q.w, iw)) * wv;
        vfz = vfz + (c.m * quot(qv.z - pv.z, q.w, iw)) * wv;
    }
};

// Integration of the learned large step: the reference's update with the network's correction
// (units of g, times corr_scale) added to the acceleration of particles at least 2h from every
// wall, and the plain acceleration optionally written out (w = 1 for those particles).
// substeps = 0: one symplectic Euler step of dt (the reference's update with the correction).
// substeps = K > 0: the outcome of K symplectic Euler steps of dt / K under a force frozen at its
// current value, v = v0 + K (dt/K) a and x = x0 + (dt/K) (K v0 + K (K+1)/2 (dt/K) a), which
// removes the K (K-1)/2 (dt/K)^2 a position error of a single large step.
__device__ __forceinline__ void learned_axis(const StepConsts& c, float pf, float vf, float ext, float denom,
                                             float v0, float x0, float dt, float substeps, float corr,
                                             float& acc_plain, float& vel, float& pos) {
    vf = vf * c.mu;
    const float force = (pf + vf) + ext;
    acc_plain = force / denom;
    const float a = acc_plain + corr;
    const float v = v0 + a * dt;
    vel = fminf(fmaxf(v, -c.max_speed), c.max_speed);
    if (substeps > 0.0f) {
        const float dts = dt / substeps;
        pos = x0 + dts * (substeps * v0 + (substeps * (substeps + 1.0f) * 0.5f) * dts * a);
    } else {
        pos = x0 + vel * dt;
    }
    if (pos < c.border) {
        vel = vel * -c.damping;
        pos = c.border;
    } else if (pos > c.hi) {
        vel = vel * -c.damping;
        pos = c.hi;
    }
}

__device__ __forceinline__ bool closure_interior(const StepConsts& c, float x, float y, float z) {
    const float margin = 2.0f * c.h;
    return x > margin && y > margin && z > margin && x < c.size - margin && y < c.size - margin &&
           z < c.size - margin;
}

__device__ __forceinline__ void learned_integrate(const StepConsts& c, const ForceSums& f, const V3& ext, float denom,
                                                  const float4& p, const float4& pv, uint32_t t, float dt,
                                                  float substeps, bool have_corr, const V3& kc, float corr_scale,
                                                  float4* __restrict__ acc_out, float4& po, float4& vo) {
    float4 k = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const bool interior = closure_interior(c, p.x, p.y, p.z);
    if (have_corr && interior) k = make_float4(kc.x * corr_scale, kc.y * corr_scale, kc.z * corr_scale, 0.0f);
    float4 a;
    learned_axis(c, f.pfx, f.vfx, ext.x, denom, pv.x, p.x, dt, substeps, k.x, a.x, vo.x, po.x);
    learned_axis(c, f.pfy, f.vfy, ext.y, denom, pv.y, p.y, dt, substeps, k.y, a.y, vo.y, po.y);
    learned_axis(c, f.pfz, f.vfz, ext.z, denom, pv.z, p.z, dt, substeps, k.z, a.z, vo.z, po.z);
    a.w = interior ? 1.0f : 0.0f;
    if (acc_out) acc_out[t] = a;
}

// MODE 0: the reference's force pass.  MODE 1 (learned closure): dt comes from the argument and
// corr * corr_scale is added to the acceleration of particles at least 2h from every wall; with
// acc_out the plain acceleration is also written out.  MODE 2: as MODE 1 with the correction
// averaged over the particle and its accepted neighbours, weights h - distance (h for the
// particle itself); neighbours within 2h of a wall count with a zero correction.
// LIST: the neighbours come from the lists the density pass wrote (a particle whose list
// overflowed searches as without LIST).
template <int BLOCK, int CAP, int CHUNK, bool PLANE_DRAIN, int MODE, bool LIST>
__global__ __launch_bounds__(BLOCK) void k_update(Scenes S, const float4* __restrict__ posrho_in,
                                                  const float4* __restrict__ velp_in,
                                                  const uint32_t* __restrict__ skey,
                                                  const uint2* __restrict__ range, float4* __restrict__ posrho_out,
                                                  float4* __restrict__ velp_out,
                                                  unsigned long long* __restrict__ scene_done,
                                                  const uint32_t* __restrict__ id_sorted, uint32_t* __restrict__ id_out,
                                                  float dt_arg, const float4* __restrict__ corr, float corr_scale,
                                                  float4* __restrict__ acc_out, const uint32_t* __restrict__ nlist,
                                                  const uint32_t* __restrict__ ncount, float substeps,
                                                  const uint32_t* __restrict__ div_flags, RecordBackup backup) {
    // with neighbour lists the pass keeps no LDS (a particle whose list overflowed searches
    // without one, below), so that its occupancy is bound by registers alone
    __shared__ uint32_t s_list[LIST ? 1 : CAP * BLOCK];
    const uint32_t b = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t s = scene_of(scene_table<BLOCK>(S), S.num_scenes, b);
    const SceneDesc& d = S.desc[s];
    const StepConsts c = d.c;  // by value, as in k_density: not reloaded after each LDS store
    const uint32_t lt = (b - first_blocks<BLOCK>(S)[s]) * BLOCK + threadIdx.x;
    if (lt >= c.n) return;
    const uint32_t t = d.p_off + lt;
    const float4 p = posrho_in[t];
    const float4 pv = velp_in[t];
    if (backup.posrho) {
        backup.posrho[t] = p;
        backup.velp[t] = pv;
        if (backup.ids && id_sorted) backup.ids[t] = id_sorted[t];
    }
    const lds_ptr<uint32_t> list = (lds_ptr<uint32_t>)s_list + threadIdx.x;
    ForceSums f{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    V3 csum{0.0f, 0.0f, 0.0f};  // MODE 2: weighted sum of neighbour corrections
    float wsum = 0.0f;
    // Every neighbour's pressure and viscosity terms.  FAST (a density pass ran since the last sort
    // and found all of this step's operands in div_operand's range; a wave-uniform flag) shares
    // one reciprocal between the quotients of a neighbour; the results are the same bits either
    // way.
    auto accumulate = [&](auto fast) {
        constexpr bool FAST = decltype(fast)::value;
        auto load = [&](uint32_t u, float4& q, float4& qv) {
            q = posrho_in[u];
            qv = velp_in[u];
        };
        // MODE 2: the neighbour's correction, loaded with its records (one neighbour ahead)
        auto load_corr = [&](uint32_t u) {
            if constexpr (MODE == 2) {
                if (corr) return corr[u];
            }
            return float4{0.0f, 0.0f, 0.0f, 0.0f};
        };
        auto add_corr = [&](float dist, const float4& q, const float4& cj) {
            if constexpr (MODE == 2) {
                const float w = c.h - dist;
                if (corr && closure_interior(c, q.x, q.y, q.z)) {
                    csum.x += w * cj.x;
                    csum.y += w * cj.y;
                    csum.z += w * cj.z;
                }
                wsum += w;
            }
        };
        // neighbour k + 1's records are loaded while neighbour k's terms are formed
        auto drain = [&](int cnt) {
            if (cnt <= 0) return;
            uint32_t u = list[0];
            float4 q, qv;
            load(u, q, qv);
            float4 cj = load_corr(u);
            for (int k = 0; k < cnt; ++k) {
                const uint32_t un = list[(k + 1 < cnt ? k + 1 : k) * BLOCK];
                float4 qn, qvn;
                load(un, qn, qvn);
                const float4 cjn = load_corr(un);
                const float dist = f.template add<FAST>(c, p, pv, q, qv);
                add_corr(dist, q, cj);
                q = qn;
                qv = qvn;
                cj = cjn;
            }
        };
        bool searched = true;
        if constexpr (LIST) {
            // lists are written by the density pass; after a sort with none since, they describe
            // the previous order and the particle searches instead
            const uint32_t cnt = (div_flags[0] & kDivPending) ? kListOverflow : ncount[t];
            if (cnt != kListOverflow) {
                searched = false;
                // the same loop as the drain, over the stored list (entry k at nlist[k * total + t]):
                // entry k + 2's index and entry k + 1's records load while entry k's terms are formed,
                // so no gather waits for the index it needs
                const size_t stride = S.total_particles;
                if (cnt > 0) {
                    const uint32_t last = cnt - 1;
                    const uint32_t u0 = nlist[t];
                    uint32_t u1 = nlist[(size_t)(last < 1u ? last : 1u) * stride + t];
                    float4 q, qv;
                    load(u0, q, qv);
                    float4 cj = load_corr(u0);
                    for (uint32_t k = 0; k < cnt; ++k) {
                        const uint32_t u2 = nlist[(size_t)(k + 2 < cnt ? k + 2 : last) * stride + t];
                        float4 qn, qvn;
                        load(u1, qn, qvn);
                        const float4 cjn = load_corr(u1);
                        const float dist = f.template add<FAST>(c, p, pv, q, qv);
                        add_corr(dist, q, cj);
                        q = qn;
                        qv = qvn;
                        cj = cjn;
                        u1 = u2;
                    }
                }
            }
        }
        if (searched) {
            if constexpr (LIST) {
                // a list that overflowed (more than kNeighbourListMax neighbours), or lists older than
                // the last sort: every candidate is tested and an accepted one added at once, in
                // enumeration order, one slot at a time (rare, so no LDS list is kept for it)
                auto visit = [&](uint32_t start, uint32_t end, auto own) {
                    for (uint32_t u = start; u < end; ++u) {
                        if (decltype(own)::value && u == t) continue;
                        const float4 q = posrho_in[u];
                        const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
                        const float d2 = (rx * rx + ry * ry) + rz * rz;
                        if (d2 >= c.cut2) continue;  // dist >= h; a NaN distance is accepted, as in the search
                        const float4 qv = velp_in[u];
                        const float4 cj = load_corr(u);
                        const float dist = f.template add<FAST>(c, p, pv, q, qv);
                        add_corr(dist, q, cj);
                    }
                };
                auto nothing = []() {};
                for_each_neighbour_cell(skey[t], range + d.c_off, c, d.p_off + c.n, visit, nothing);
            } else {
                search_neighbours<BLOCK, CAP, CHUNK, PLANE_DRAIN>(skey[t], t, d.p_off + c.n, p.x, p.y, p.z,
                                                                  posrho_in, range + d.c_off, c, list, drain);
            }
        }
    };
    if (div_flags[0] == 0u)
        accumulate(std::true_type{});
    else
        accumulate(std::false_type{});

    V3 ext{c.g[0] * p.w, c.g[1] * p.w, c.g[2] * p.w};
    V3 mouse{0.0f, 0.0f, 0.0f}, wall{0.0f, 0.0f, 0.0f};
    if (c.mouse_force) mouse = mouse_force(c, p.x, p.y, p.z, pv.w);
    if (c.wall_force) wall = wall_forces(c, p.x, p.y, p.z);
    ext.x = ext.x + (mouse.x + wall.x);
    ext.y = ext.y + (mouse.y + wall.y);
    ext.z = ext.z + (mouse.z + wall.z);

    const float denom = p.w + 1e-16f;
    float4 po, vo;
    if (MODE == 0) {
        const float dt = d.dt;
        integrate_axis(c, f.pfx, f.vfx, ext.x, denom, pv.x, p.x, dt, vo.x, po.x);
        integrate_axis(c, f.pfy, f.vfy, ext.y, denom, pv.y, p.y, dt, vo.y, po.y);
        integrate_axis(c, f.pfz, f.vfz, ext.z, denom, pv.z, p.z, dt, vo.z, po.z);
    } else {
        V3 kc{0.0f, 0.0f, 0.0f};
        if (corr) {
            const float4 ct = corr[t];
            if (MODE == 2) {
                const float inv = 1.0f / (c.h + wsum);
                kc = V3{(c.h * ct.x + csum.x) * inv, (c.h * ct.y + csum.y) * inv, (c.h * ct.z + csum.z) * inv};
            } else {
                kc = V3{ct.x, ct.y, ct.z};
            }
        }
        learned_integrate(c, f, ext, denom, p, pv, t, dt_arg, substeps, corr != nullptr, kc, corr_scale, acc_out, po,
                          vo);
    }
    po.w = p.w;
    vo.w = pv.w;
    posrho_out[t] = po;
    velp_out[t] = vo;
    if (id_out) id_out[t] = id_sorted[t];
    // completion time of this wave's particles; the scene's latest wave ends its step
    if ((threadIdx.x & 63) == 0) atomicMax(&scene_done[s], (unsigned long long)wall_clock64());
}

// ------------------------------------------------------------------------------------------
// Tile passes: density and forces of one box of cells per workgroup, neighbours in LDS.
//
// The per-particle search above spends 14 VALU instructions and a 12-byte L1 return on each of the
// about 216 candidates of a particle, and the list-driven force pass waits on neighbour gathers
// through a 32 KB L1.  Here a workgroup copies the records of its box of cells and of the cells
// around it into LDS once, and
//   - the density pass forms candidate distances on the matrix cores (tile_search), which leaves one
//     VALU instruction per candidate and lane;
//   - both passes read neighbours from LDS.  The density pass leaves each particle's accepted
//     neighbours as 16-bit indices into the staged records (half the bytes of slots), and the force
//     pass, which stages the same boxes the same way, walks them.
// Sums are formed in the reference's order with the reference's operations, so results are the same
// bits as those of the per-particle passes.
//
// Measured against those (us, density + force): the 80,000-particle scene 120 + 202 -> 92 + 64, 192,089
// particles 90 + 125 -> 84 + 57, the million-particle block 265 + 217 -> 163 + 117, 17.8 million
// 3,582 + 3,762 -> 2,107 + 1,710; the work list and tables cost the sort 20 us of the million's step.
//
// The density pass is bound by VALU issue and, below 4 boxes a CU, by its chain of dependent loads; the force
// pass by LDS reads (32 bytes a neighbour) and arithmetic.  512 threads and 1,920 records let three density
// workgroups into a CU's LDS and registers (80 of them), and two force workgroups; 256 threads and 2,304
// records suit boxes of at most 256 particles and cells of up to 85, at 4 and 2.
// ------------------------------------------------------------------------------------------
// The box's table into sh: as k_gather formed it, or formed here for entries past its memory.
template <int BLOCK>
__device__ __forceinline__ void box_open(BoxShared& sh, const Box& b, const SceneDesc& d,
                                         const uint2* __restrict__ range, const BoxTable* __restrict__ tables,
                                         uint32_t item, uint32_t table_cap) {
    if (threadIdx.x == 0) sh.rho = 0u;
    if (item < table_cap) {  // workgroup-uniform
        for (uint32_t k = threadIdx.x; k < sizeof(BoxTable) / 16; k += BLOCK)
            reinterpret_cast<uint4*>(static_cast<BoxTable*>(&sh))[k] = reinterpret_cast<const uint4*>(tables + item)[k];
    } else {
        box_cells<BLOCK>(sh, b, d, range);
    }
}

// The work of a pass: the sparse particles in chunks of BLOCK first (a single scene's without entries of their own),
// dealt round to the XCDs, then the listed boxes, neighbours on one XCD.
struct TileItems {
    uint32_t boxes, sparse, chunks, lead, all;  // lead: items of the chunks, a multiple of kNumXcd
    uint32_t cap;
};
template <int BLOCK>
__device__ __forceinline__ TileItems tile_items(const Scenes& S, const uint32_t* __restrict__ count, uint32_t cap) {
    TileItems t;
    t.boxes = min(count[0], cap);
    t.sparse = S.num_scenes == 1 ? min(count[1], S.total_particles) : 0u;
    t.chunks = S.num_scenes == 1 ? (t.sparse + BLOCK - 1) / BLOCK : min(count[kSceneSparse - 1], cap - t.boxes);
    t.cap = cap;
    t.lead = (t.chunks + kNumXcd - 1) / kNumXcd * kNumXcd;
    t.all = t.lead + t.boxes;
    return t;
}
template <int BLOCK>
__device__ __forceinline__ uint4 tile_item(const TileItems& t, const uint4* __restrict__ tiles, uint32_t item,
                                           uint32_t& at_list) {
    at_list = 0u;
    if (item < t.lead) {
        if (item >= t.chunks) return make_uint4(0u, kEntryDirect, 0u, 0u);  // an entry of no particles
        if (t.sparse == 0u) return tiles[t.cap - 1u - item];
        const uint32_t first = item * BLOCK;
        return make_uint4(0u, kEntryDirect | kEntrySparse | min((uint32_t)BLOCK, t.sparse - first) << 13, 0u, first);
    }
    at_list = item - t.lead;
    if (t.all <= gridDim.x) at_list = xcd_block(at_list, t.boxes);
    return tiles[at_list];
}

// Copies the box's records: store(LDS index, record, slot) for each.  Eight lanes take a cell, neighbours in
// x side by side, with up to 16 records of kFlight cells in flight.  The table is read where box_open reads it,
// without waiting for sh.
template <int BLOCK, typename Load, typename Store>
__device__ __forceinline__ void box_stage_from(const Box& b, const BoxTable* table, uint32_t cap, Load load,
                                               Store store) {
    constexpr int kFlight = 3, kGroups = BLOCK / 8;
    const uint32_t sub = threadIdx.x & 7u;
    const int ncell = b.hx * b.hy * b.hz;
    using Rec = decltype(load(0u));
    for (int i0 = (int)(threadIdx.x >> 3); i0 < ncell; i0 += kGroups * kFlight) {
        Rec v[kFlight][2];
        uint32_t at[kFlight], end[kFlight], slot[kFlight];
#pragma unroll
        for (int k = 0; k < kFlight; ++k) {
            const int i = i0 + k * kGroups, c = table_cell(b, min(i, ncell - 1));
            const uint32_t e = table->cell[c];
            slot[k] = table->slot[c];
            at[k] = (e & 0xffffu) + sub;
            end[k] = i < ncell ? min(e >> 16, cap) : 0u;
        }
#pragma unroll
        for (int k = 0; k < kFlight; ++k) {
            if (at[k] < end[k]) v[k][0] = load(at[k] + slot[k]);
            if (at[k] + 8u < end[k]) v[k][1] = load(at[k] + 8u + slot[k]);
        }
#pragma unroll
        for (int k = 0; k < kFlight; ++k) {
            if (at[k] < end[k]) store(at[k], v[k][0], at[k] + slot[k]);
            if (at[k] + 8u < end[k]) store(at[k] + 8u, v[k][1], at[k] + 8u + slot[k]);
        }
        for (int k = 0; k < kFlight; ++k)  // cells of more than 16 records
            for (uint32_t a = at[k] + 16u; a < end[k]; a += 8u) store(a, load(a + slot[k]), a + slot[k]);
    }
}

template <int BLOCK, typename Load, typename Store>
__device__ __forceinline__ void box_stage(const BoxShared& sh, const Box& b, const BoxTable* __restrict__ tables,
                                          uint32_t item, uint32_t table_cap, uint32_t cap, Load load, Store store) {
    if (item < table_cap)
        box_stage_from<BLOCK>(b, tables + item, cap, load, store);
    else
        box_stage_from<BLOCK>(b, &sh, cap, load, store);
}

// The lane's particle: lane `at` of the box's `sh.own` numbering (lanes past a column's or the box's last
// particle repeat it).
struct BoxLane {
    uint32_t idx;   // its record in LDS
    uint32_t slot;
    int cell;       // its halo cell
    bool valid;
};
__device__ __forceinline__ BoxLane box_lane(const BoxShared& sh, const Box& b, uint32_t at, const SceneDesc& d) {
    const uint32_t all = sh.own[kMaxBox * kMaxBox];
    const uint32_t a = min(at, all - 1u);
    int q = -1;  // the last column that starts at or before `a` (empty ones after it start past it or hold no lane)
#pragma unroll
    for (int k = 0; k < kMaxBox * kMaxBox; ++k) q += a >= sh.own[k] ? 1 : 0;
    const int c0 = own_column(b, q);
    const uint32_t st = sh.cell[c0 + 1] & 0xffffu, n = (sh.cell[c0 + b.nz] >> 16) - st;
    uint32_t li = a - sh.own[q];
    BoxLane L;
    L.valid = at < all && li < n;
    li = min(li, n - 1u);
    L.idx = st + li;
    L.cell = c0 + 1;
    for (int k = 2; k <= b.nz; ++k) L.cell += L.idx >= (sh.cell[c0 + k] & 0xffffu) ? 1 : 0;
    L.slot = L.idx + sh.slot[L.cell];
    L.valid = L.valid && L.slot - d.p_off < d.c.n;  // always, unless the scan failed
    return L;
}

// Candidates of a wave's particles, on the matrix cores.
//
// v_mfma_f32_4x4x1 (16 blocks) forms, for each group of four lanes, a 4x4 outer product: lane 4g + i
// supplies row i (a candidate), lane 4g + j column j (its own particle), and lane 4g + j receives
// column j in four registers.  Four of them (x, y, z, 1) accumulate
//     C + sum_k (-2 a'_k) b_k + n_b,   C = n_a + 2 sum_k a'_k o_k - cut2 - margin,
// with a' = a - o, n_a = |a'|^2, n_b = |b - o|^2 (staged beside the record) and o the box's centre:
// that is |a - b|^2 - cut2 - margin, rounded.  Its sign bit marks a candidate; one v_alignbit per
// register shifts it into the lane's mask.  The four lanes of a group are consecutive particles of a
// column of cells along z, so their candidates in a neighbouring column lie in one window of three or
// four cells (more where cells hold fewer than four).
//
// Rounding, in units of bin^2: |a'_k| and |b_k - o_k| are at most 3 (boxes with a particle further out search
// directly), o lies in the grid of R cells a side, so |b_k| <= R + 3, whatever the cube's `size` is.  n_a and n_b are
// at most 27, 2 sum a'_k o_k and the three products 18 R and 18 (R + 3), and a cutoff over 108 accepts every pair.  So
// no partial sum exceeds 18 R + 220, and with the inputs' own rounding the sum errs by less than 2^-24 (144 R + 2,010)
// < 1.2e-5 (R + 10): with that margin the marked candidates are a superset of the accepted ones (measured: 0.2 of it at
// most), and the drain applies the exact test.
//
// A lane appends its marked candidates to its list in enumeration order: cells in NEIGHBORHOOD order,
// candidates in slot order.
typedef float mfma_f4 __attribute__((ext_vector_type(4)));
constexpr int kPosPad = 32 + 8;      // records read past a window's end

__device__ __forceinline__ uint32_t group_first(uint32_t x) {  // of the group of four lanes
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x00, 0xf, 0xf, true);
}
__device__ __forceinline__ uint32_t group_last(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xff, 0xf, 0xf, true);
}

// Eight candidates from q (4 lanes' worth at q and at q + 4) into the low bits of mask, the first highest.
__device__ __forceinline__ uint32_t mark_eight(const float4* q, float b0, float b1, float b2, const mfma_f4& cc,
                                               uint32_t mask) {
    const float4 p = q[0], r = q[4];
    mfma_f4 u = __builtin_amdgcn_mfma_f32_4x4x1f32(p.w, 1.0f, cc, 0, 0, 0);
    mfma_f4 v = __builtin_amdgcn_mfma_f32_4x4x1f32(r.w, 1.0f, cc, 0, 0, 0);
    u = __builtin_amdgcn_mfma_f32_4x4x1f32(p.x, b0, u, 0, 0, 0);
    v = __builtin_amdgcn_mfma_f32_4x4x1f32(r.x, b0, v, 0, 0, 0);
    u = __builtin_amdgcn_mfma_f32_4x4x1f32(p.y, b1, u, 0, 0, 0);
    v = __builtin_amdgcn_mfma_f32_4x4x1f32(r.y, b1, v, 0, 0, 0);
    u = __builtin_amdgcn_mfma_f32_4x4x1f32(p.z, b2, u, 0, 0, 0);
    v = __builtin_amdgcn_mfma_f32_4x4x1f32(r.z, b2, v, 0, 0, 0);
#pragma unroll
    for (int k = 0; k < 4; ++k) mask = __builtin_amdgcn_alignbit(mask, __float_as_uint(u[k]), 31);
#pragma unroll
    for (int k = 0; k < 4; ++k) mask = __builtin_amdgcn_alignbit(mask, __float_as_uint(v[k]), 31);
    return mask;
}

// One column (dx, dy) of three cells at a time, in NEIGHBORHOOD order: append(bits, first) receives a window's
// marked candidates 32 at a time, bit 31 - k for record first + k.
template <typename Append>
__device__ __forceinline__ void tile_search(const BoxShared& sh, const Box& b, const float4* s_pos, const BoxLane& L,
                                            float b0, float b1, float b2, float c0, Append append) {
    const uint32_t sub = lane_id() & 3u;
    const mfma_f4 cc = {c0, c0, c0, c0};
    const int sy = b.hz, sx = b.hy * b.hz;
    const lds_ptr<const uint32_t> table = (lds_ptr<const uint32_t>)sh.cell + (L.cell - 1 - sy - sx);
    uint32_t lo = table[0], hi = table[2];
#pragma unroll 1
    for (int dx = 0; dx < 3; ++dx) {
#pragma unroll 1
        for (int dy = 0; dy < 3; ++dy) {
            const uint32_t st = lo & 0xffffu, en = hi >> 16;
            // the next column's entries (past the last, some entries of the table)
            const int next = dy < 2 ? dx * sx + (dy + 1) * sy : (dx < 2 ? (dx + 1) * sx : 0);
            lo = table[next];
            hi = table[next + 2];
            const uint32_t w0 = group_first(st), len = group_last(en) - w0;
            for (uint32_t w = 0; __any(w < len); w += 32u) {
                const float4* const q = s_pos + w0 + min(w, len) + sub;
                uint32_t mask = mark_eight(q, b0, b1, b2, cc, 0u);
                int got = 24;
                if (__any(len > w + 8u)) {  // wave-uniform, as below
                    mask = mark_eight(q + 8, b0, b1, b2, cc, mask);
                    got = 16;
                    if (__any(len > w + 16u)) {
                        mask = mark_eight(q + 16, b0, b1, b2, cc, mask);
                        got = 8;
                        if (__any(len > w + 24u)) {
                            mask = mark_eight(q + 24, b0, b1, b2, cc, mask);
                            got = 0;
                        }
                    }
                }
                mask <<= got;  // candidate w0 + w + k at bit 31 - k
                // the lane's own three cells
                const uint32_t from = max(st, w0 + w);
                const int n = (int)(min(en, w0 + w + 32u) - from);
                uint32_t m = n > 0 ? mask << (from - w0 - w) & (uint32_t)((int)0x80000000u >> (n - 1)) : 0u;
                if (dx == 1 && dy == 1) {  // not the particle itself
                    const uint32_t self = L.idx - from;
                    m &= self < 32u ? ~(0x80000000u >> self) : ~0u;
                }
                append(m, from);
            }
        }
    }
}

template <int BLOCK, int CAP, int WPE, bool GLOBAL>
__global__ __launch_bounds__(BLOCK, WPE) void k_density_tile(Scenes S, const uint4* __restrict__ tiles,
                                                        const uint32_t* __restrict__ tile_count, uint32_t tile_cap,
                                                        const BoxTable* __restrict__ tables, uint32_t table_cap,
                                                        const uint32_t* __restrict__ sparse,
                                                        float4* __restrict__ posrho, float4* __restrict__ velp,
                                                        const uint32_t* __restrict__ skey,
                                                        const uint2* __restrict__ range, uint32_t* __restrict__ rho_max,
                                                        uint16_t* __restrict__ llist, uint16_t* __restrict__ lcount,
                                                        uint32_t list_cap, uint32_t list_chunks,
                                                        uint32_t* __restrict__ nlist,
                                                        uint32_t* __restrict__ ncount) {
    constexpr uint32_t kFar = CAP + kPosPad;
    __shared__ float4 s_pos[CAP + kPosPad + 1];
    __shared__ uint32_t s_slot[GLOBAL ? CAP + kPosPad : 1];
    __shared__ BoxShared sh;
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAnd(&rho_max[1], ~kDivPending);
    const TileItems items = tile_items<BLOCK>(S, tile_count, tile_cap);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (threadIdx.x == 0) s_pos[kFar] = make_float4(1e30f, 1e30f, 1e30f, 1e30f);
    for (uint32_t item = blockIdx.x; item < items.all; item += gridDim.x) {
        uint32_t at_list;
        const uint4 e = tile_item<BLOCK>(items, tiles, item, at_list);
        if (e.y == kEntryDirect) continue;  // no particles, and no scene's
        const SceneDesc& d = S.desc[e.z];
        const StepConsts c = d.c;
        uint32_t top = 0;  // largest density of the lane's particles, as bits (NaN ranks highest)
        auto finish = [&](uint32_t t, const float4& p, float rho) {
            const float wall = c.wall_density ? wall_density(c, p.x, p.y, p.z) : 0.0f;
            const float density = rho + wall;
            const float pressure = eos(c, rho);
            reinterpret_cast<float*>(posrho)[4 * (size_t)t + 3] = density;
            reinterpret_cast<float*>(velp)[4 * (size_t)t + 3] = pressure;
            const bool ok = pos_operand(p.x) && pos_operand(p.y) && pos_operand(p.z) && div_operand(pressure) &&
                            div_operand(density) && density != 0.0f;
            if (!ok) atomicOr(&rho_max[1], kDivUnsafe);
            top = max(top, __float_as_uint(density) & 0x7fffffffu);
        };
        // a particle of a box with irregular positions: every candidate tested from HBM, added at once
        auto direct = [&](uint32_t t) {
            const float4 p = posrho[t];
            float rho = c.m * poly6(c, 0.0f);
            uint32_t written = 0;
            auto visit = [&](uint32_t start, uint32_t end, auto own) {
                for (uint32_t u = start; u < end; ++u) {
                    if (decltype(own)::value && u == t) continue;
                    const float4 q = posrho[u];
                    const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
                    const float d2 = (rx * rx + ry * ry) + rz * rz;
                    if (d2 >= c.cut2) continue;
                    rho += c.m * poly6(c, sqrtf(d2));
                    if (GLOBAL && written < kNeighbourListMax) nlist[(size_t)written * S.total_particles + t] = u;
                    ++written;
                }
            };
            auto nothing = []() {};
            for_each_neighbour_cell(skey[t], range + d.c_off, c, d.p_off + c.n, visit, nothing);
            if (GLOBAL) ncount[t] = written <= kNeighbourListMax ? written : kListOverflow;
            finish(t, p, rho);
        };
        if (e.y & kEntryDirect) {
            if (threadIdx.x == 0) sh.rho = 0u;
            __syncthreads();
            using Entry = typename std::conditional<GLOBAL, uint32_t, float>::type;
            // the search's lists take the records' place
            constexpr int kFit = (int)(sizeof(float4) * CAP / (BLOCK * sizeof(Entry)));
            constexpr int kDirectCap = kFit < 40 ? kFit : 40;
            const lds_ptr<Entry> found = (lds_ptr<Entry>)reinterpret_cast<Entry*>(s_pos) + threadIdx.x;
            for (uint32_t i = threadIdx.x; i < e.y >> 13; i += BLOCK) {
                const uint32_t t = e.y & kEntrySparse ? sparse[min(e.w + i, S.total_particles - 1u)] : e.w + i;
                if (t - d.p_off >= c.n) continue;  // only after a failed scan
                const float4 p = posrho[t];
                float rho = c.m * poly6(c, 0.0f);
                uint32_t written = 0;
                auto drain = [&](int cnt) {
                    for (int k = 0; k < cnt; ++k) {
                        if constexpr (GLOBAL) {
                            const uint32_t u = found[k * BLOCK];
                            const float4 q = posrho[u];
                            const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
                            const float d2 = (rx * rx + ry * ry) + rz * rz;
                            rho += c.m * poly6(c, sqrtf(d2));
                            if (written < kNeighbourListMax) nlist[(size_t)written * S.total_particles + t] = u;
                            ++written;
                        } else {
                            rho += c.m * poly6(c, sqrtf(found[k * BLOCK]));
                        }
                    }
                };
                search_neighbours<BLOCK, kDirectCap, 4, false>(skey[t], t, d.p_off + c.n, p.x, p.y, p.z, posrho,
                                                               range + d.c_off, c, found, drain);
                if (GLOBAL) ncount[t] = written <= kNeighbourListMax ? written : kListOverflow;
                finish(t, p, rho);
            }
        } else {
            const Box b = box_of(e);
            box_open<BLOCK>(sh, b, d, range, tables, at_list, table_cap);
            const float ox = ((float)b.x + 0.5f * (float)b.nx) * c.bin, oy = ((float)b.y + 0.5f * (float)b.ny) * c.bin,
                        oz = ((float)b.z + 0.5f * (float)b.nz) * c.bin;
            const float reach = 3.001f * c.bin;
            bool bad = false;
            box_stage<BLOCK>(
                sh, b, tables, at_list, table_cap, CAP,
                [&](uint32_t slot) { return posrho[min(slot, d.p_off + c.n - 1u)]; },
                [&](uint32_t at, float4 q, uint32_t slot) {
                    const float x = q.x - ox, y = q.y - oy, z = q.z - oz;
                    bad |= !(fabsf(x) <= reach && fabsf(y) <= reach && fabsf(z) <= reach && pos_operand(q.x) &&
                             pos_operand(q.y) && pos_operand(q.z));
                    q.w = (x * x + y * y) + z * z;
                    s_pos[at] = q;
                    if (GLOBAL) s_slot[at] = slot;
                });
            const bool irregular = __syncthreads_or(bad ? 1 : 0) != 0;
            if (sh.records > CAP) {  // only after a failed scan
                __syncthreads();
                continue;
            }
            const uint32_t lanes = sh.own[kMaxBox * kMaxBox];
            const float cut = c.cut2 + 1.2e-5f * c.bin * (c.bin * (float)(c.R + 10));
            const bool room = e.w + (lanes + 63u) / 64u <= list_chunks, listable = room && !irregular;
            bool overflowed = false;
            for (uint32_t ch = (uint32_t)wave; ch * 64u < lanes; ch += BLOCK / 64) {
                const BoxLane L = box_lane(sh, b, ch * 64u + lane_id(), d);
                const float4 p = s_pos[L.idx];
                char* const list =
                    reinterpret_cast<char*>(llist) + (size_t)(e.w + ch) * (list_cap * 128u) + lane_id() * 2u;
                uint32_t cnt = list_cap + 1u;  // no list: as an overflowed one
                if (listable) {                // workgroup-uniform
                    const float ax = p.x - ox, ay = p.y - oy, az = p.z - oz;
                    // lanes that repeat a particle mark nothing
                    const float c0 = L.valid ? (p.w - cut) + 2.0f * ((ax * ox + ay * oy) + az * oz) : 1e30f;
                    // Candidates go to the particle's list: a queue in LDS would take 4 KB a wave, and half the
                    // waves of a CU with it.  Past the list's end they are only counted.
                    char* const list_end = list + list_cap * 128u;
                    char* next = list;
                    auto append = [&](uint32_t m, uint32_t first) {
                        if (__any(next + 32 * 128 > list_end)) {  // wave-uniform
                            for (; m != 0u; next += 128) {
                                const uint32_t k = (uint32_t)__builtin_clz(m);
                                m ^= 0x80000000u >> k;
                                if (next < list_end) *reinterpret_cast<uint16_t*>(next) = (uint16_t)((first + k) << 4);
                            }
                        } else {
                            for (; m != 0u; next += 128) {
                                const uint32_t k = (uint32_t)__builtin_clz(m);
                                m ^= 0x80000000u >> k;
                                *reinterpret_cast<uint16_t*>(next) = (uint16_t)((first + k) << 4);
                            }
                        }
                    };
                    tile_search(sh, b, s_pos, L, -2.0f * ax, -2.0f * ay, -2.0f * az, c0, append);
                    cnt = (uint32_t)(next - list) / 128u;
                }
                if (!L.valid) continue;
                if (room) lcount[(e.w + ch) * 64u + lane_id()] = (uint16_t)min(cnt, list_cap + 1u);
                if (cnt > list_cap) {
                    overflowed = true;
                    continue;
                }
                // The exact test and the sum, in order, kAhead candidates a round with the next round's in
                // flight.  Past its list a lane takes the record kFar, out of everything's reach.
                constexpr uint32_t kAhead = 4;
                const char* const rec = reinterpret_cast<const char*>(s_pos);
                auto entry = [&](uint32_t k) { return (uint32_t)*reinterpret_cast<const uint16_t*>(list + k * 128u); };
                auto dist2 = [&](uint32_t o) {
                    const float4 q = *reinterpret_cast<const float4*>(rec + o);
                    const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
                    return (rx * rx + ry * ry) + rz * rz;
                };
                float rho = c.m * poly6(c, 0.0f);
                uint32_t written = 0;  // accepted so far
                uint32_t off[kAhead];
#pragma unroll
                for (uint32_t j = 0; j < kAhead; ++j) off[j] = entry(j);
                for (uint32_t k = 0; __any(k < cnt); k += kAhead) {
                    uint32_t cur[kAhead];
#pragma unroll
                    for (uint32_t j = 0; j < kAhead; ++j) cur[j] = k + j < cnt ? off[j] : kFar << 4;
                    const uint32_t ahead = min(k + kAhead, list_cap - kAhead);  // wave-uniform
#pragma unroll
                    for (uint32_t j = 0; j < kAhead; ++j) off[j] = entry(ahead + j);
                    const uint32_t before = written;
#pragma unroll
                    for (uint32_t j = 0; j < kAhead; ++j) {
                        const float d2 = dist2(cur[j]);
                        const float sum = rho + c.m * poly6(c, sqrt_in_range(d2));
                        const bool in = d2 < c.cut2;
                        rho = in ? sum : rho;
                        if (GLOBAL && in && written < kNeighbourListMax)
                            nlist[(size_t)written * S.total_particles + L.slot] = s_slot[cur[j] >> 4];
                        written += in ? 1u : 0u;
                    }
                    // a rejected candidate (one within the margin) becomes the particle itself, which adds
                    // nothing to the force sums
                    if (__any(k < cnt && written - before != min(cnt - k, kAhead))) {
#pragma unroll
                        for (uint32_t j = 0; j < kAhead; ++j)
                            if (k + j < cnt && !(dist2(cur[j]) < c.cut2))
                                *reinterpret_cast<uint16_t*>(list + (k + j) * 128u) = (uint16_t)(L.idx << 4);
                    }
                }
                if (GLOBAL) ncount[L.slot] = written <= kNeighbourListMax ? written : kListOverflow;
                finish(L.slot, p, rho);
            }
            // Lanes without a list, after the others: the search's state next to theirs would spill.
            if (__any(overflowed)) {
                for (uint32_t ch = (uint32_t)wave; ch * 64u < lanes; ch += BLOCK / 64) {
                    const BoxLane L = box_lane(sh, b, ch * 64u + lane_id(), d);
                    if (L.valid && (!room || lcount[(e.w + ch) * 64u + lane_id()] > list_cap)) direct(L.slot);
                }
            }
        }
        for (int k = 32; k >= 1; k >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, k));
        if (lane_id() == 0) atomicMax(&sh.rho, top);
        __syncthreads();
        if (threadIdx.x == 0) atomicMax(rho_max, sh.rho);
        __syncthreads();
    }
}

// Forces + integration of one box per workgroup.  MODE 0 and 1 as in k_update.
template <int BLOCK, int CAP, int WPE, int MODE>
__global__ __launch_bounds__(BLOCK, WPE) void k_update_tile(Scenes S, const uint4* __restrict__ tiles,
                                                       const uint32_t* __restrict__ tile_count, uint32_t tile_cap,
                                                       const BoxTable* __restrict__ tables, uint32_t table_cap,
                                                       const uint32_t* __restrict__ sparse,
                                                       const float4* __restrict__ posrho_in,
                                                       const float4* __restrict__ velp_in,
                                                       const uint32_t* __restrict__ skey,
                                                       const uint2* __restrict__ range, float4* __restrict__ posrho_out,
                                                       float4* __restrict__ velp_out,
                                                       unsigned long long* __restrict__ scene_done,
                                                       const uint32_t* __restrict__ id_sorted,
                                                       uint32_t* __restrict__ id_out,
                                                       const uint16_t* __restrict__ llist,
                                                       const uint16_t* __restrict__ lcount, uint32_t list_cap,
                                                       uint32_t list_chunks,
                                                       const uint32_t* __restrict__ div_flags, float dt_arg,
                                                       const float4* __restrict__ corr, float corr_scale,
                                                       float4* __restrict__ acc_out, float substeps,
                                                       RecordBackup backup) {
    __shared__ float4 s_rec[2 * CAP];
    float4* const s_pos = s_rec;
    float4* const s_vel = s_rec + CAP;
    __shared__ BoxShared sh;
    const TileItems items = tile_items<BLOCK>(S, tile_count, tile_cap);
    const uint32_t flags = div_flags[0];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (uint32_t item = blockIdx.x; item < items.all; item += gridDim.x) {
        uint32_t at_list;
        const uint4 e = tile_item<BLOCK>(items, tiles, item, at_list);
        if (e.y == kEntryDirect) continue;  // no particles, and no scene's
        const SceneDesc& d = S.desc[e.z];
        const StepConsts c = d.c;
        auto finish = [&](uint32_t t, const float4& p, const float4& pv, const ForceSums& f) {
            if (backup.posrho) {
                backup.posrho[t] = p;
                backup.velp[t] = pv;
                if (backup.ids && id_sorted) backup.ids[t] = id_sorted[t];
            }
            V3 ext{c.g[0] * p.w, c.g[1] * p.w, c.g[2] * p.w};
            V3 mouse{0.0f, 0.0f, 0.0f}, wall{0.0f, 0.0f, 0.0f};
            if (c.mouse_force) mouse = mouse_force(c, p.x, p.y, p.z, pv.w);
            if (c.wall_force) wall = wall_forces(c, p.x, p.y, p.z);
            ext.x = ext.x + (mouse.x + wall.x);
            ext.y = ext.y + (mouse.y + wall.y);
            ext.z = ext.z + (mouse.z + wall.z);
            const float denom = p.w + 1e-16f;
            float4 po, vo;
            if (MODE == 0) {
                const float dt = d.dt;
                integrate_axis(c, f.pfx, f.vfx, ext.x, denom, pv.x, p.x, dt, vo.x, po.x);
                integrate_axis(c, f.pfy, f.vfy, ext.y, denom, pv.y, p.y, dt, vo.y, po.y);
                integrate_axis(c, f.pfz, f.vfz, ext.z, denom, pv.z, p.z, dt, vo.z, po.z);
            } else {
                V3 kc{0.0f, 0.0f, 0.0f};
                if (corr) {
                    const float4 ct = corr[t];
                    kc = V3{ct.x, ct.y, ct.z};
                }
                learned_integrate(c, f, ext, denom, p, pv, t, dt_arg, substeps, corr != nullptr, kc, corr_scale,
                                  acc_out, po, vo);
            }
            po.w = p.w;
            vo.w = pv.w;
            posrho_out[t] = po;
            velp_out[t] = vo;
            if (id_out) id_out[t] = id_sorted[t];
        };
        // a particle without a list: every candidate tested from HBM, added at once
        auto direct = [&](uint32_t t) {
            const float4 p = posrho_in[t], pv = velp_in[t];
            ForceSums f{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            auto visit = [&](uint32_t start, uint32_t end, auto own) {
                for (uint32_t u = start; u < end; ++u) {
                    if (decltype(own)::value && u == t) continue;
                    const float4 q = posrho_in[u];
                    const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
                    const float d2 = (rx * rx + ry * ry) + rz * rz;
                    if (d2 >= c.cut2) continue;
                    f.template add<false>(c, p, pv, q, velp_in[u]);
                }
            };
            auto nothing = []() {};
            for_each_neighbour_cell(skey[t], range + d.c_off, c, d.p_off + c.n, visit, nothing);
            finish(t, p, pv, f);
        };
        if (e.y & kEntryDirect) {
            // the search's lists take the records' place
            constexpr int kFit = (int)(2 * sizeof(float4) * CAP / (BLOCK * sizeof(uint32_t)));
            constexpr int kDirectCap = kFit < 40 ? kFit : 40;
            const lds_ptr<uint32_t> found = (lds_ptr<uint32_t>)reinterpret_cast<uint32_t*>(s_rec) + threadIdx.x;
            for (uint32_t i = threadIdx.x; i < e.y >> 13; i += BLOCK) {
                const uint32_t t = e.y & kEntrySparse ? sparse[min(e.w + i, S.total_particles - 1u)] : e.w + i;
                if (t - d.p_off >= c.n) continue;  // only after a failed scan
                const float4 p = posrho_in[t], pv = velp_in[t];
                ForceSums f{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                auto drain = [&](int cnt) {
                    for (int k = 0; k < cnt; ++k) {
                        const uint32_t u = found[k * BLOCK];
                        if (flags == 0u)
                            f.add_in_range(c, p, pv, posrho_in[u], velp_in[u]);
                        else
                            f.template add<false>(c, p, pv, posrho_in[u], velp_in[u]);
                    }
                };
                search_neighbours<BLOCK, kDirectCap, 4, false>(skey[t], t, d.p_off + c.n, p.x, p.y, p.z, posrho_in,
                                                               range + d.c_off, c, found, drain);
                finish(t, p, pv, f);
            }
        } else {
            const Box b = box_of(e);
            box_open<BLOCK>(sh, b, d, range, tables, at_list, table_cap);
            struct Rec {
                float4 p, v;
            };
            box_stage<BLOCK>(
                sh, b, tables, at_list, table_cap, CAP,
                [&](uint32_t slot) {
                    const uint32_t u = min(slot, d.p_off + c.n - 1u);
                    return Rec{posrho_in[u], velp_in[u]};
                },
                [&](uint32_t at, const Rec& r, uint32_t) {
                    s_pos[at] = r.p;
                    s_vel[at] = r.v;
                });
            __syncthreads();
            if (sh.records > CAP) {  // only after a failed scan
                __syncthreads();
                continue;
            }
            const uint32_t lanes = sh.own[kMaxBox * kMaxBox];
            const bool listed_box = !(flags & kDivPending) && e.w + (lanes + 63u) / 64u <= list_chunks;
            for (uint32_t ch = (uint32_t)wave; ch * 64u < lanes; ch += BLOCK / 64) {
                const BoxLane L = box_lane(sh, b, ch * 64u + lane_id(), d);
                if (!L.valid) continue;
                const uint32_t cnt = listed_box ? (uint32_t)lcount[(e.w + ch) * 64u + lane_id()] : list_cap + 1u;
                if (cnt > list_cap) {
                    direct(L.slot);
                    continue;
                }
                const float4 p = s_pos[L.idx], pv = s_vel[L.idx];
                ForceSums f{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                const char* const list =
                    reinterpret_cast<const char*>(llist) + (size_t)(e.w + ch) * (list_cap * 128u) + lane_id() * 2u;
                const char* const rec_p = reinterpret_cast<const char*>(s_pos);
                const char* const rec_v = reinterpret_cast<const char*>(s_vel);
                auto entry = [&](uint32_t k) {
                    return (uint32_t)*reinterpret_cast<const uint16_t*>(list + k * 128u);
                };
                auto pos = [&](uint32_t off) { return *reinterpret_cast<const float4*>(rec_p + off); };
                auto vel = [&](uint32_t off) { return *reinterpret_cast<const float4*>(rec_v + off); };
                if (flags == 0u) {
                    // All lanes run to the longest list of the wave, kAhead entries a round, the next round's
                    // offsets in flight.  Past its list a lane takes its own record, which adds nothing: the
                    // differences are 0, and every sum keeps its bits (it starts at +0, see ForceSums).
                    constexpr uint32_t kAhead = 4;
                    const uint32_t self = L.idx << 4;
                    uint32_t off[kAhead];
#pragma unroll
                    for (uint32_t j = 0; j < kAhead; ++j) off[j] = entry(j);
                    for (uint32_t k = 0; __any(k < cnt); k += kAhead) {
                        uint32_t cur[kAhead];
#pragma unroll
                        for (uint32_t j = 0; j < kAhead; ++j) cur[j] = k + j < cnt ? off[j] : self;
                        const uint32_t ahead = min(k + kAhead, list_cap - kAhead);  // wave-uniform
#pragma unroll
                        for (uint32_t j = 0; j < kAhead; ++j) off[j] = entry(ahead + j);
#pragma unroll
                        for (uint32_t j = 0; j < kAhead; ++j) f.add_in_range(c, p, pv, pos(cur[j]), vel(cur[j]));
                    }
                } else {
                    for (uint32_t k = 0; k < cnt; ++k) {
                        const uint32_t u = min(entry(k), (sh.records - 1u) << 4);
                        if (u == L.idx << 4) continue;  // a rejected candidate
                        f.template add<false>(c, p, pv, pos(u), vel(u));
                    }
                }
                finish(L.slot, p, pv, f);
            }
        }
        __syncthreads();  // the box's last particle is done
        if (threadIdx.x == 0) atomicMax(&scene_done[e.z], (unsigned long long)wall_clock64());
    }
}


// ------------------------------------------------------------------------------------------
// advect.comp:20-59 (the reference compiles it but Fluid::update never dispatches it): a
// position-only step on buffer 1, x += v dt, then the cube clamp with the shader's own border
// 0.01 and damping 0.3 (advect.comp:30-31), in place.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kHashBlock) void k_advect(Scenes S, float4* __restrict__ posrho,
                                                       float4* __restrict__ velp, float dt) {
    const uint32_t b = blockIdx.x;
    const uint32_t s = scene_of(S.scene256, S.num_scenes, b);
    const SceneDesc& d = S.desc[s];
    const uint32_t lt = (b - S.blk256[s]) * kHashBlock + threadIdx.x;
    if (lt >= d.c.n) return;
    const uint32_t i = d.p_off + lt;
    float4 x = posrho[i], v = velp[i];
    const float damping = 0.3f, border = 0.01f;
    const float hi = d.c.size - border;
    x.x = x.x + v.x * dt;
    x.y = x.y + v.y * dt;
    x.z = x.z + v.z * dt;
    auto clamp_axis = [&](float& xa, float& va) {
        if (xa < border) {
            va = va * -damping;
            xa = border;
        } else if (xa > hi) {
            va = va * -damping;
            xa = hi;
        }
    };
    clamp_axis(x.x, v.x);
    clamp_axis(x.y, v.y);
    clamp_axis(x.z, v.z);
    posrho[i] = x;
    velp[i] = v;
}

// ------------------------------------------------------------------------------------------
// Learned closure features (single-scene contexts).  For every requested slot of the sorted
// buffer: its 32 nearest neighbours inside the kernel radius (the density pass's acceptance
// test; nearest by squared distance, among equal distances the earlier in NEIGHBORHOOD
// enumeration order), listed in enumeration order, each as ((x_j - x_i) / h, v_j - v_i);
// then rho_i / rho0 - 1 scaled by 10, the step multiplier / 4 and the fraction of the 32 places
// filled; zero padded to 208 bf16 values.
// ------------------------------------------------------------------------------------------
constexpr int kFeatBlock = 64;
constexpr int kFeatCap = 40;    // accepted neighbours held per particle between selections
constexpr int kFeatChunk = 4;   // candidate slots loaded per step of a lane's walk

// Removes the `drop` farthest of a lane's `cnt` listed neighbours (largest squared distance;
// of equal ones the later), keeping the rest in order.  Squared distances compare as their bit
// patterns: non-negative floats order like the integers, and NaN, which the acceptance test
// lets through, ranks above every number.
__device__ __forceinline__ int drop_farthest(lds_ptr<uint32_t> key, lds_ptr<uint32_t> slot, int cnt, int drop) {
    // the lane's keys into registers (all loads in flight), the `drop` largest marked one at a
    // time (of equal keys the later entry), then one pass that closes the gaps in order -- the
    // same entries, in the same order, as dropping and shifting one at a time
    uint32_t kv[kFeatCap];
#pragma unroll
    for (int k = 0; k < kFeatCap; ++k) kv[k] = k < cnt ? key[k * kFeatBlock] : 0u;
    uint64_t gone = 0;
    for (int m = 0; m < drop; ++m) {
        uint32_t best = 0;
        int at = 0;
#pragma unroll
        for (int k = 0; k < kFeatCap; ++k) {
            const bool ge = k < cnt && !((gone >> k) & 1ull) && kv[k] >= best;
            best = ge ? kv[k] : best;
            at = ge ? k : at;
        }
        gone |= 1ull << at;
    }
    int w = 0;
#pragma unroll
    for (int k = 0; k < kFeatCap; ++k) {
        if (k < cnt && !((gone >> k) & 1ull)) {  // w <= k: a move never overwrites an unread entry
            key[w * kFeatBlock] = kv[k];
            slot[w * kFeatBlock] = slot[k * kFeatBlock];
            ++w;
        }
    }
    return w;
}

// two floats -> two bf16 (round to nearest even) in one word, lo in the low half: one
// v_cvt_pk_bf16_f32 on gfx950
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// One feature row: the kept neighbours' relative positions (/ h) and velocities, in
// bf16, then the scaled density deviation, dt multiplier and filled fraction.  slot_of(k) gives
// the k-th kept neighbour's slot, k < cnt.
// Software-pipelined: the gathers of group g + 1 are issued before group g is formed, and the
// scheduling barrier keeps the compiler from interleaving them with waits.  Positions k >= cnt
// load the particle's own record t and write zeros.
template <typename SlotOf>
__device__ __forceinline__ void write_feature_row(uint4* __restrict__ row, const StepConsts& c, uint32_t t, float4 p,
                                                  float4 pv, int cnt, SlotOf slot_of,
                                                  const float4* __restrict__ posrho, const float4* __restrict__ velp,
                                                  float dt_mult) {
    const float inv_h = 1.0f / c.h;
    float4 q[4], qv[4];
    auto load_group = [&](int g) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = g * 4 + j;
            const uint32_t u = k < cnt ? slot_of(k) : t;
            q[j] = posrho[u];
            qv[j] = velp[u];
        }
    };
    load_group(0);
    // eight groups of four neighbours: 24 values = three 16-byte stores
#pragma unroll
    for (int g = 0; g < kClosureNeighbours / 4; ++g) {
        float4 cq[4], cqv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            cq[j] = q[j];
            cqv[j] = qv[j];
        }
        if (g + 1 < kClosureNeighbours / 4) load_group(g + 1);
        __builtin_amdgcn_sched_barrier(0);
        float v[24];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            // zeros past cnt by masking the bits; the mask is opaque to the optimizer, which would
            // otherwise turn a select into a branch around the loads
            uint32_t m = g * 4 + j < cnt ? ~0u : 0u;
            asm("" : "+v"(m));
            auto keep = [m](float x) { return __uint_as_float(__float_as_uint(x) & m); };
            v[6 * j + 0] = keep((cq[j].x - p.x) * inv_h);
            v[6 * j + 1] = keep((cq[j].y - p.y) * inv_h);
            v[6 * j + 2] = keep((cq[j].z - p.z) * inv_h);
            v[6 * j + 3] = keep(cqv[j].x - pv.x);
            v[6 * j + 4] = keep(cqv[j].y - pv.y);
            v[6 * j + 5] = keep(cqv[j].z - pv.z);
        }
#pragma unroll
        for (int e = 0; e < 3; ++e)
            row[g * 3 + e] = make_uint4(pack_bf16(v[8 * e + 0], v[8 * e + 1]), pack_bf16(v[8 * e + 2], v[8 * e + 3]),
                                        pack_bf16(v[8 * e + 4], v[8 * e + 5]), pack_bf16(v[8 * e + 6], v[8 * e + 7]));
    }
    const float rho_rel = (p.w / c.rho0 - 1.0f) * 10.0f;
    row[24] = make_uint4(pack_bf16(rho_rel, dt_mult * 0.25f), pack_bf16((float)cnt * (1.0f / kClosureNeighbours), 0.0f),
                         0u, 0u);
    row[25] = make_uint4(0u, 0u, 0u, 0u);
}

__global__ void k_clear_word(uint32_t* __restrict__ w) {
    if (threadIdx.x == 0) *w = 0u;
}

// Lists a lane selects from by its threshold network (k_closure_select) hold up to kSelRegCap
// entries; longer ones are selected by bisection or by the wave, and lists that overflowed go
// through k_closure_features on kHeavyBlocks workgroups.
constexpr int kSelRegCap = 40;
constexpr int kHeavyBlocks = 64;
static_assert(kSelRegCap <= (int)kNeighbourListMax, "the selection's loads stay inside the lists");

// Loads at a wave-uniform base plus a per-lane 32-bit byte offset, the form global loads take with
// the base in scalar registers (one VGPR per address instead of two).  Slots are below 2^28.
__device__ __forceinline__ uint32_t load_at(const uint32_t* base, uint32_t slot) {
    return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(base) + (slot << 2));
}
__device__ __forceinline__ float3 load_pos_at(const float4* base, uint32_t slot) {
    const float* f = reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + (slot << 4));
    return float3{f[0], f[1], f[2]};
}

// The kClosureNeighbours nearest of the m listed neighbours of slot t, kClosureNeighbours < m <=
// CAP <= kClosureNeighbours + 8, in list order, to sel_out at the particle's slot.
// - The list entries load 8 at a time, two groups ahead of the neighbours' positions, which load 8
//   at a time, one group ahead of the distances formed from them.  The key of an entry is its
//   squared distance's bits, so NaN ranks farthest; entries past m take key 0.
// - The D = m - kClosureNeighbours largest keys, each as often as it occurs, come out of an
//   insertion network of 8 (two instructions per key and level, no indexing); the D-th largest, T,
//   is the threshold.  Every key above T is dropped, and of the keys equal to T the last
//   D - #{above} in list order: what dropping the largest key, of equal ones the later entry, D
//   times drops.
// - The entries are read again, the dropped ones removed in registers (each closes its gap, the
//   last first), and the kClosureNeighbours kept ones written in list order, entry j of slot t at
//   sel_out[t * kClosureNeighbours + j]: one whole 128-byte line per row, in 16-byte stores.
template <int CAP>
__device__ __forceinline__ void select_by_threshold(uint32_t t, uint32_t m, uint32_t n,
                                                    const float4* __restrict__ posrho,
                                                    const uint32_t* __restrict__ nlist, size_t stride,
                                                    uint32_t* __restrict__ sel_out) {
    constexpr int kTop = 8, kGroup = 8, kGroups = CAP / kGroup;
    static_assert(CAP <= (int)kNeighbourListMax && CAP - kClosureNeighbours <= kTop, "one network of 8");
    static_assert(CAP % kGroup == 0 && kGroups >= 2, "whole groups");
    const float4 p = posrho[t];
    auto entries = [&](int g, uint32_t (&u)[kGroup]) {
#pragma unroll
        for (int j = 0; j < kGroup; ++j) u[j] = load_at(nlist + (size_t)(g * kGroup + j) * stride, t);
    };
    // entries past m may be stale: one out of range is replaced by the particle's own slot
    auto gather = [&](int g, const uint32_t (&u)[kGroup], float3 (&q)[kGroup]) {
#pragma unroll
        for (int j = 0; j < kGroup; ++j) {
            q[j] = load_pos_at(posrho, u[j] < n ? u[j] : t);
        }
    };
    uint32_t key[CAP];
    uint32_t ua[kGroup];
    float3 cur[kGroup], nxt[kGroup];
    entries(0, ua);
    gather(0, ua, cur);
    entries(1, ua);
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        if (g + 1 < kGroups) gather(g + 1, ua, nxt);
        if (g + 2 < kGroups) entries(g + 2, ua);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kGroup; ++j) {
            const float rx = p.x - cur[j].x, ry = p.y - cur[j].y, rz = p.z - cur[j].z;
            uint32_t kk = __float_as_uint((rx * rx + ry * ry) + rz * rz);
            kk = (uint32_t)(g * kGroup + j) < m ? kk : 0u;
            // keeps the distance here, between the group's loads: left free, the instruction
            // selector moves all of them after the last group, with every position held meanwhile
            asm volatile("" : "+v"(kk));
            key[g * kGroup + j] = kk;
        }
#pragma unroll
        for (int j = 0; j < kGroup; ++j) cur[j] = nxt[j];
    }
    // top[0] >= top[1] >= ... >= top[7]: the 8 largest keys, each as often as it occurs
    uint32_t top[kTop];
#pragma unroll
    for (int i = 0; i < kTop; ++i) top[i] = 0u;
#pragma unroll
    for (int k = 0; k < CAP; ++k) {
        uint32_t x = key[k];
#pragma unroll
        for (int i = 0; i < kTop; ++i) {
            const uint32_t hi = max(top[i], x);
            x = min(top[i], x);
            top[i] = hi;
        }
    }
    const uint32_t drop = m - (uint32_t)kClosureNeighbours;  // 1 ... CAP - kClosureNeighbours
    uint32_t thr = top[0];
#pragma unroll
    for (int i = 1; i < kTop; ++i) thr = drop == (uint32_t)(i + 1) ? top[i] : thr;
    uint32_t above = 0;  // entries past m (key 0) are never above
#pragma unroll
    for (int k = 0; k < CAP; ++k) above += key[k] > thr ? 1u : 0u;
    // Keys equal to T are dropped from the end of the list.  With T = 0 the entries past m, last
    // in the list and of key 0, come first: they take CAP - m of the drops, on top of the real ones.
    uint32_t ties = drop - above + (thr == 0u ? (uint32_t)CAP - m : 0u);
    uint64_t gone = 0;
#pragma unroll
    for (int k = CAP - 1; k >= 0; --k) {
        const bool eq = key[k] == thr && ties != 0u;
        ties -= eq ? 1u : 0u;
        gone |= (key[k] > thr || eq) ? (1ull << k) : 0ull;
    }
    // the dropped entries before m (entries past m follow every kept one and need no removal)
    uint64_t dropped = gone & ((1ull << m) - 1ull);  // m <= CAP < 64
    __builtin_amdgcn_sched_barrier(0);
    // read the entries again rather than hold them through the selection (registers); the pointer
    // is passed through an empty asm statement so the loads are not merged with the first ones
    const uint32_t* again = nlist;
    asm volatile("" : "+s"(again));
    uint32_t u[CAP];
#pragma unroll
    for (int k = 0; k < CAP; ++k) u[k] = load_at(again + (size_t)k * stride, t);
    // at most CAP - kClosureNeighbours drops; a lane with fewer shifts nothing in the later rounds
#pragma unroll
    for (int r = 0; r < CAP - kClosureNeighbours; ++r) {
        if (__ballot(dropped != 0) == 0) break;  // wave-uniform
        const uint32_t g = dropped != 0 ? 63u - (uint32_t)__clzll((long long)dropped) : 64u;
        dropped &= ~(1ull << (g & 63u));
#pragma unroll
        for (int i = 0; i + 1 < CAP; ++i) u[i] = (uint32_t)i >= g ? u[i + 1] : u[i];
    }
    uint4* row = reinterpret_cast<uint4*>(sel_out + (size_t)t * kClosureNeighbours);
#pragma unroll
    for (int j = 0; j < kClosureNeighbours / 4; ++j)
        row[j] = make_uint4(u[4 * j], u[4 * j + 1], u[4 * j + 2], u[4 * j + 3]);
}

// The kClosureNeighbours nearest of the m listed neighbours of slot t, kSelRegCap < m <=
// kNeighbourListMax, in list order, to sel_out at the particle's slot (as select_by_threshold).
// - Keys are formed as there (entries past m take the largest key, 0xFFFFFFFF).
// - v, the kClosureNeighbours-th smallest key with multiplicity (the least v with at least
//   kClosureNeighbours keys <= v), is found by bisection over the 32-bit key range: 32 rounds of
//   one compare and one add per key, no indexing.
// - Kept: every key below v, and of the keys equal to v the first kClosureNeighbours - #{below} in
//   list order -- the kClosureNeighbours smallest by (key, list position), which is what dropping
//   the largest key, of equal ones the later entry, m - kClosureNeighbours times leaves.  Entries
//   past m follow every real one, so they are never among them.
// - The entries are read again and written to the lane's row of LDS at its next free word, which
//   advances only past a kept entry (a dropped entry is overwritten by the next kept one, or lands
//   in the row's spare last word); the row's kClosureNeighbours words then go out as 16-byte
//   stores, one 128-byte line.
constexpr int kSelStageWords = kClosureNeighbours + 1;  // per lane: odd, so lanes' rows fall in different banks
__device__ __forceinline__ void select_by_bisection(uint32_t t, uint32_t m, uint32_t n,
                                                    const float4* __restrict__ posrho,
                                                    const uint32_t* __restrict__ nlist, size_t stride,
                                                    uint32_t* __restrict__ sel_out, lds_ptr<uint32_t> stage) {
    constexpr int CAP = (int)kNeighbourListMax, kGroup = 4, kGroups = CAP / kGroup;  // 64 keys held: smaller groups
    static_assert(CAP <= 64 && CAP % kGroup == 0, "one 64-bit mask, whole groups");
    const float4 p = posrho[t];
    // the list's columns in order, through one advancing scalar pointer (the empty asm keeps the
    // compiler from holding every column's address in scalar registers)
    const uint32_t* col = nlist;
    auto entries = [&](int, uint32_t (&u)[kGroup]) {
#pragma unroll
        for (int j = 0; j < kGroup; ++j) {
            u[j] = load_at(col, t);
            col += stride;
            asm volatile("" : "+s"(col));
        }
    };
    auto gather = [&](const uint32_t (&u)[kGroup], float3 (&q)[kGroup]) {
#pragma unroll
        for (int j = 0; j < kGroup; ++j) q[j] = load_pos_at(posrho, u[j] < n ? u[j] : t);
    };
    uint32_t key[CAP];
    uint32_t ua[kGroup];
    float3 cur[kGroup], nxt[kGroup];
    entries(0, ua);
    gather(ua, cur);
    entries(1, ua);
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        if (g + 1 < kGroups) gather(ua, nxt);
        if (g + 2 < kGroups) entries(g + 2, ua);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kGroup; ++j) {
            const float rx = p.x - cur[j].x, ry = p.y - cur[j].y, rz = p.z - cur[j].z;
            uint32_t kk = __float_as_uint((rx * rx + ry * ry) + rz * rz);
            kk = (uint32_t)(g * kGroup + j) < m ? kk : 0xFFFFFFFFu;
            asm volatile("" : "+v"(kk));  // formed here, between the group's loads
            key[g * kGroup + j] = kk;
        }
#pragma unroll
        for (int j = 0; j < kGroup; ++j) cur[j] = nxt[j];
    }
    uint32_t lo = 0u, hi = 0xFFFFFFFFu;
#pragma unroll 1
    for (int round = 0; round < 32; ++round) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        uint32_t c = 0;
#pragma unroll
        for (int k = 0; k < CAP; ++k) c += key[k] <= mid ? 1u : 0u;
        const bool enough = c >= (uint32_t)kClosureNeighbours;
        hi = enough ? mid : hi;
        lo = enough ? lo : mid + 1u;
    }
    const uint32_t v = lo;
    uint32_t below = 0;
#pragma unroll
    for (int k = 0; k < CAP; ++k) below += key[k] < v ? 1u : 0u;
    uint32_t quota = (uint32_t)kClosureNeighbours - below;
    uint64_t keep = 0;
#pragma unroll
    for (int k = 0; k < CAP; ++k) {
        const bool eq = key[k] == v && quota != 0u;
        quota -= eq ? 1u : 0u;
        keep |= (key[k] < v || eq) ? (1ull << k) : 0ull;
    }
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t* again = nlist;  // read again, not merged with the first loads (registers)
    uint32_t w = 0;
#pragma unroll
    for (int k = 0; k < CAP; ++k) {
        asm volatile("" : "+s"(again));
        stage[w] = load_at(again, t);
        again += stride;
        w += (uint32_t)(keep >> k) & 1u;
    }
    uint4* row = reinterpret_cast<uint4*>(sel_out + (size_t)t * kClosureNeighbours);
#pragma unroll
    for (int j = 0; j < kClosureNeighbours / 4; ++j)
        row[j] = make_uint4(stage[4 * j], stage[4 * j + 1], stage[4 * j + 2], stage[4 * j + 3]);
}

// One row of kSelRegCap + 1 ... kNeighbourListMax entries selected by the whole wave: slot t
// (uniform), its m listed neighbours (uniform), the lane's entry u (entry `lane`; the row's own
// slot past m) and that entry's position q.  Lane k ranks entry k among the row's m entries by
// (squared distance bits, list position), reading the others' keys lane by lane; the
// kClosureNeighbours lowest ranks are kept, in list order (the same entries as
// select_by_bisection keeps).  For waves with a few such rows: one row costs the wave about as
// much as the bisection costs each lane, but only the rows there are.
constexpr int kSelWaveRowsMax = 8;
struct WaveRow {
    uint32_t t, m, u;
    float3 q;
};
__device__ __forceinline__ void select_row_by_wave(const WaveRow& w, const float4* __restrict__ posrho,
                                                   uint32_t* __restrict__ sel_out) {
    static_assert(kNeighbourListMax == 64, "one entry per lane");
    const uint32_t lane = threadIdx.x & 63;
    const float4 p = posrho[w.t];
    const float rx = p.x - w.q.x, ry = p.y - w.q.y, rz = p.z - w.q.z;
    const uint32_t key = __float_as_uint((rx * rx + ry * ry) + rz * rz);
    uint32_t rank = 0;
    for (uint32_t j = 0; j < w.m; ++j) {
        const uint32_t kj = (uint32_t)__builtin_amdgcn_readlane((int)key, (int)j);
        rank += (kj < key || (kj == key && j < lane)) ? 1u : 0u;
    }
    const bool keep = lane < w.m && rank < (uint32_t)kClosureNeighbours;
    const uint64_t km = __ballot(keep);
    if (keep) sel_out[(size_t)w.t * kClosureNeighbours + (uint32_t)__popcll(km & ((1ull << lane) - 1ull))] = w.u;
}

// Selection of the kept neighbours of every slot whose list is longer than kClosureNeighbours:
// lists of up to kSelRegCap entries by each lane's threshold network; longer ones up to
// kNeighbourListMax by each lane's bisection in a wave that has more than kSelWaveRowsMax of them,
// else by the whole wave one row at a time; overflowed lists are appended to `heavy` (one atomic
// per wave that has any) for k_closure_features' walk.  Rows of at most kClosureNeighbours need no
// selection.
__global__ __launch_bounds__(256) void k_closure_select(const float4* __restrict__ posrho, uint32_t n,
                                                        const uint32_t* __restrict__ nlist,
                                                        const uint32_t* __restrict__ ncount, size_t stride,
                                                        uint32_t* __restrict__ sel_out, uint32_t* __restrict__ heavy,
                                                        uint32_t* __restrict__ heavy_count) {
    __shared__ uint32_t s_stage[256 * kSelStageWords];
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    const uint32_t m = t < n ? ncount[t] : 0u;
    const bool is_heavy = m > kNeighbourListMax;  // kListOverflow
    const uint64_t hm = __ballot(is_heavy);
    if (hm != 0) {  // wave-uniform
        const uint32_t lane = threadIdx.x & 63;
        const uint32_t leader = (uint32_t)__ffsll((unsigned long long)hm) - 1u;
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(heavy_count, (uint32_t)__popcll(hm));
        base = __shfl(base, (int)leader);
        if (is_heavy) heavy[base + (uint32_t)__popcll(hm & ((1ull << lane) - 1ull))] = t;
    }
    if (m > (uint32_t)kClosureNeighbours && m <= (uint32_t)kSelRegCap)
        select_by_threshold<kSelRegCap>(t, m, n, posrho, nlist, stride, sel_out);
    const bool longer = m > (uint32_t)kSelRegCap && !is_heavy;
    uint64_t rows = __ballot(longer);
    if (__popcll(rows) > kSelWaveRowsMax) {  // wave-uniform
        if (longer)
            select_by_bisection(t, m, n, posrho, nlist, stride, sel_out,
                                (lds_ptr<uint32_t>)s_stage + threadIdx.x * kSelStageWords);
        return;
    }
    // A few longer rows: every lane of the wave takes part in each, one after another, while the
    // next row's positions and the one after's list entries are in flight.
    const uint32_t lane = threadIdx.x & 63;
    auto next_row = [&](WaveRow& w) {  // wave-uniform; issues the row's list loads
        if (rows == 0) return false;
        const int l = __ffsll((unsigned long long)rows) - 1;
        rows &= rows - 1;
        w.t = (uint32_t)__builtin_amdgcn_readlane((int)t, l);
        w.m = (uint32_t)__builtin_amdgcn_readlane((int)m, l);
        w.u = lane < w.m ? nlist[(size_t)lane * stride + w.t] : w.t;
        return true;
    };
    auto positions = [&](WaveRow& w) {
        const float* f = reinterpret_cast<const float*>(posrho + w.u);
        w.q = float3{f[0], f[1], f[2]};
    };
    WaveRow a{}, b{}, c{};
    bool have_a = next_row(a), have_b = false;
    if (have_a) {
        positions(a);
        have_b = next_row(b);
    }
    while (have_a) {  // wave-uniform
        bool have_c = false;
        if (have_b) {
            positions(b);
            have_c = next_row(c);
        }
        select_row_by_wave(a, posrho, sel_out);
        a = b;
        b = c;
        have_a = have_b;
        have_b = have_c;
    }
}

// Rows whose particle has at most kClosureNeighbours listed neighbours keep all of them, in list
// order: written straight from the density pass's lists, with no distances and no LDS.  Other
// rows are left to k_closure_features.
__global__ __launch_bounds__(256) void k_closure_features_short(Scenes S, const float4* __restrict__ posrho,
                                                                const float4* __restrict__ velp,
                                                                const uint32_t* __restrict__ rows, uint32_t nrows,
                                                                float dt_mult, uint16_t* __restrict__ X,
                                                                const uint32_t* __restrict__ nlist,
                                                                const uint32_t* __restrict__ ncount) {
    const uint32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= nrows) return;
    const SceneDesc& d = S.desc[0];
    const StepConsts& c = d.c;
    const uint32_t t = rows ? rows[r] : d.p_off + r;
    uint4* row = reinterpret_cast<uint4*>(X + (size_t)r * kClosureFeatures);
    if (t - d.p_off >= c.n) {
        for (int q = 0; q < kClosureFeatures / 8; ++q) row[q] = make_uint4(0u, 0u, 0u, 0u);
        return;
    }
    const uint32_t listed = ncount[t];
    if (listed > (uint32_t)kClosureNeighbours) return;  // more than are kept, or overflowed
    // all listed slots first (coalesced across the wave, in flight together)
    const size_t stride = S.total_particles;
    uint32_t u[kClosureNeighbours];
#pragma unroll
    for (int k = 0; k < kClosureNeighbours; ++k) u[k] = (uint32_t)k < listed ? nlist[(size_t)k * stride + t] : t;
    write_feature_row(row, c, t, posrho[t], velp[t], (int)listed, [&](int k) { return u[k]; }, posrho, velp, dt_mult);
}

// One row of k_closure_features.
__device__ __forceinline__ void closure_row(const Scenes& S, const float4* __restrict__ posrho,
                                            const float4* __restrict__ velp, const uint32_t* __restrict__ skey,
                                            const uint2* __restrict__ range, const uint32_t* __restrict__ rows,
                                            uint32_t r, float dt_mult, uint16_t* __restrict__ X,
                                            const uint32_t* __restrict__ nlist, const uint32_t* __restrict__ ncount,
                                            bool skip_short, uint32_t* __restrict__ sel_out, lds_ptr<uint32_t> key,
                                            lds_ptr<uint32_t> slot) {
    const SceneDesc& d = S.desc[0];
    const StepConsts& c = d.c;
    const uint32_t t = rows ? rows[r] : d.p_off + r;
    uint4* row = X ? reinterpret_cast<uint4*>(X + (size_t)r * kClosureFeatures) : nullptr;  // null: slots to sel_out
    if (t - d.p_off >= c.n) {
        if (row)
            for (int q = 0; q < kClosureFeatures / 8; ++q) row[q] = make_uint4(0u, 0u, 0u, 0u);
        return;
    }
    // rows of short lists are written by k_closure_features_short
    if (skip_short && ncount[t] <= (uint32_t)kClosureNeighbours) return;
    const float4 p = posrho[t];
    const float4 pv = velp[t];
    int cnt = 0;
    auto visit = [&](uint32_t start, uint32_t end, auto own) {
        for (uint32_t u = start; u < end; u += kFeatChunk) {
            if (cnt > kFeatCap - kFeatChunk) cnt = drop_farthest(key, slot, cnt, cnt - kClosureNeighbours);
            const uint32_t left = end - u;
            const float4* q = posrho + u;  // the buffers are padded past the last particle
            float4 v[kFeatChunk];
#pragma unroll
            for (int j = 0; j < kFeatChunk; ++j) v[j] = q[j];
#pragma unroll
            for (int j = 0; j < kFeatChunk; ++j) {
                const float rx = p.x - v[j].x, ry = p.y - v[j].y, rz = p.z - v[j].z;
                const float d2 = (rx * rx + ry * ry) + rz * rz;
                bool ok = ((uint32_t)j < left) & !(d2 >= c.cut2);
                if constexpr (decltype(own)::value) ok &= (u + (uint32_t)j != t);
                key[cnt * kFeatBlock] = __float_as_uint(d2);
                slot[cnt * kFeatBlock] = u + (uint32_t)j;
                cnt += ok ? 1 : 0;
            }
        }
    };
    auto nothing = []() {};
    // With the density pass's neighbour lists the accepted neighbours are read in the same order
    // instead of searched for (a list that overflowed is searched for as without lists).
    const uint32_t listed = ncount ? ncount[t] : kListOverflow;
    if (listed != kListOverflow) {
        const size_t stride = S.total_particles;
        for (uint32_t k = 0; k < listed; k += kFeatChunk) {
            if (cnt > kFeatCap - kFeatChunk) cnt = drop_farthest(key, slot, cnt, cnt - kClosureNeighbours);
            uint32_t u[kFeatChunk];
            float4 v[kFeatChunk];
#pragma unroll
            for (int j = 0; j < kFeatChunk; ++j) u[j] = nlist[(size_t)min(k + (uint32_t)j, listed - 1) * stride + t];
#pragma unroll
            for (int j = 0; j < kFeatChunk; ++j) v[j] = posrho[u[j]];
#pragma unroll
            for (int j = 0; j < kFeatChunk; ++j) {
                const float rx = p.x - v[j].x, ry = p.y - v[j].y, rz = p.z - v[j].z;
                const float d2 = (rx * rx + ry * ry) + rz * rz;
                key[cnt * kFeatBlock] = __float_as_uint(d2);
                slot[cnt * kFeatBlock] = u[j];
                cnt += (k + (uint32_t)j < listed) ? 1 : 0;
            }
        }
    } else {
        for_each_neighbour_cell(skey[t], range + d.c_off, c, d.p_off + c.n, visit, nothing);
    }
    if (cnt > kClosureNeighbours) cnt = drop_farthest(key, slot, cnt, cnt - kClosureNeighbours);

    if (sel_out) {
        // the kept neighbours' slots instead of the row, entry k of slot t at
        // sel_out[t * kClosureNeighbours + k] as the selection writes them, for inference that
        // forms the values itself
        for (int k = 0; k < cnt; ++k) sel_out[(size_t)(t - d.p_off) * kClosureNeighbours + k] = slot[k * kFeatBlock];
        return;
    }
    write_feature_row(row, c, t, p, pv, cnt, [&](int k) { return slot[k * kFeatBlock]; }, posrho, velp, dt_mult);
}

__global__ __launch_bounds__(kFeatBlock) void k_closure_features(Scenes S, const float4* __restrict__ posrho,
                                                                 const float4* __restrict__ velp,
                                                                 const uint32_t* __restrict__ skey,
                                                                 const uint2* __restrict__ range,
                                                                 const uint32_t* __restrict__ rows, uint32_t nrows,
                                                                 float dt_mult, uint16_t* __restrict__ X,
                                                                 const uint32_t* __restrict__ nlist,
                                                                 const uint32_t* __restrict__ ncount,
                                                                 bool skip_short, uint32_t* __restrict__ sel_out,
                                                                 const uint32_t* __restrict__ nrows_dev) {
    static_assert(kFeatChunk <= (int)kRecordPad + 1, "chunked loads may run kFeatChunk - 1 records past a cell");
    static_assert(kFeatCap >= kClosureNeighbours + kFeatChunk, "a chunk must fit after a selection");
    __shared__ uint32_t s_key[kFeatCap * kFeatBlock];
    __shared__ uint32_t s_slot[kFeatCap * kFeatBlock];
    if (nrows_dev) nrows = *nrows_dev;  // a count an earlier kernel wrote
    // rows r, r + the grid, ...: one row per lane when the grid covers them all
    for (uint32_t r = blockIdx.x * kFeatBlock + threadIdx.x; r < nrows; r += gridDim.x * kFeatBlock)
        closure_row(S, posrho, velp, skey, range, rows, r, dt_mult, X, nlist, ncount, skip_short, sel_out,
                    (lds_ptr<uint32_t>)s_key + threadIdx.x, (lds_ptr<uint32_t>)s_slot + threadIdx.x);
}

// ------------------------------------------------------------------------------------------
// After the host rewrites the particle buffers or the parameters: the cell key of every slot of
// buffer 2 is recomputed from its position with the current constants (the neighbour passes
// read it where the reference recomputes clamp(ivec3(p / binSize)), density.comp:88,
// update.comp:141), the neighbour lists are marked overflowed (so every reader searches), and
// the force pass's division operands are marked unchecked.  The cell ranges stay those of the
// last sort, as the reference's counts and offsets do.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kHashBlock) void k_invalidate(Scenes S, const float4* __restrict__ posrho,
                                                           uint32_t* __restrict__ skey, uint32_t* __restrict__ ncount,
                                                           uint32_t* __restrict__ div_flags) {
    const uint32_t b = blockIdx.x;
    if (b == 0 && threadIdx.x == 0) atomicOr(div_flags, kDivPending | kDivUnsafe);
    if (b >= S.blocks256) return;
    const uint32_t s = scene_of(S.scene256, S.num_scenes, b);
    const SceneDesc& d = S.desc[s];
    const uint32_t lt = (b - S.blk256[s]) * kHashBlock + threadIdx.x;
    if (lt >= d.c.n) return;
    const uint32_t t = d.p_off + lt;
    const float4 p = posrho[t];
    skey[t] = cell_key(d.c, p.x, p.y, p.z);
    if (ncount) ncount[t] = kListOverflow;
}

// ------------------------------------------------------------------------------------------
// Allocation-free step: the scene's constants and block tables go into the library's fixed
// scratch array (from kernel arguments, so nothing is copied from host memory), and what a step
// expects to start at zero is cleared: the cell counts (a step whose scan failed leaves some
// behind) and the failure word.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kHashBlock) void k_noalloc_setup(SceneDesc d, uint4 t0, uint4 t1,
                                                              SceneDesc* __restrict__ desc,
                                                              uint32_t* __restrict__ tables,
                                                              uint32_t* __restrict__ counts, uint32_t ncells,
                                                              uint32_t* __restrict__ error_flag) {
    const uint32_t g = blockIdx.x * kHashBlock + threadIdx.x;
    if (g == 0) {
        *desc = d;
        reinterpret_cast<uint4*>(tables)[0] = t0;
        reinterpret_cast<uint4*>(tables)[1] = t1;
        *error_flag = 0u;
    }
    for (uint32_t i = g; i < ncells; i += gridDim.x * kHashBlock) counts[i] = 0u;
}

// ------------------------------------------------------------------------------------------
// Record <-> split-half conversion.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kHashBlock) void k_split(const float4* __restrict__ rec, float4* __restrict__ posrho,
                                                      float4* __restrict__ velp, uint32_t n) {
    const uint32_t i = blockIdx.x * kHashBlock + threadIdx.x;
    if (i >= n) return;
    posrho[i] = rec[2 * (size_t)i];
    velp[i] = rec[2 * (size_t)i + 1];
}

__global__ __launch_bounds__(kHashBlock) void k_join(const float4* __restrict__ posrho,
                                                     const float4* __restrict__ velp, float4* __restrict__ rec,
                                                     uint32_t n) {
    const uint32_t i = blockIdx.x * kHashBlock + threadIdx.x;
    if (i >= n) return;
    rec[2 * (size_t)i] = posrho[i];
    rec[2 * (size_t)i + 1] = velp[i];
}

inline unsigned blocks_for(size_t n, unsigned per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

hipError_t launch_hash(const DeviceBuffers& b, bool tiles, hipStream_t s) {
    const Scenes& S = b.sc;
    size_t blocks = S.blocks256;
    const size_t reset = blocks_for(S.total_tiles > S.num_scenes ? S.total_tiles : S.num_scenes, kHashBlock);
    if (reset > blocks) blocks = reset;
    if (blocks == 0) blocks = 1;  // still resets the step clock
    hipLaunchKernelGGL(k_hash, dim3((unsigned)blocks), dim3(kHashBlock), 0, s, S, b.posrho[0], b.key, b.rank,
                       b.counts, b.scan_status, b.scene_done, b.step_start, b.rho_max, b.crowd_count,
                       tiles ? b.tile_count : nullptr);
    return hipGetLastError();
}

hipError_t launch_scan(const DeviceBuffers& b, hipStream_t s) {
    if (b.sc.total_tiles == 0) return hipSuccess;
    hipLaunchKernelGGL(k_scan, dim3(b.sc.total_tiles), dim3(kScanThreads), 0, s, b.sc, b.counts, b.range,
                       b.scan_status, b.error_flag);
    return hipGetLastError();
}

static unsigned tile_grid(const DeviceBuffers& b) {
    // About one workgroup per box where boxes hold 8 particles a cell, and the chip's fill where most hold
    // fewer; a longer list is walked with this stride.
    const uint64_t most = (uint64_t)b.sc.total_particles / (8 * b.sc.bx * b.sc.by * b.sc.bz) + 512;
    return (unsigned)(b.tile_cap < most ? b.tile_cap : most);
}

static TileWork tile_work(const DeviceBuffers& b, const TileShape* t) {
    TileWork w{};
    if (!t) return w;
    w.tiles = b.tiles;
    w.count = b.tile_count;
    w.cap = b.tile_cap;
    w.rec_cap = (uint32_t)t->cap;
    w.chunk = (uint32_t)t->block;
    w.tables = b.tables;
    w.table_cap = b.table_cap;
    w.sparse = b.sparse;
    w.sparse_max = sparse_records(b.sc.total_particles) * (uint32_t)((t->x + 2) * (t->y + 2) * (t->z + 2));
    return w;
}

hipError_t launch_place(const DeviceBuffers& b, const TileShape* tiles, hipStream_t s) {
    if (b.sc.blocks256 == 0) return hipSuccess;
    const unsigned extra = tiles ? b.sc.tblocks : 0u;
    hipLaunchKernelGGL(tiles ? k_place<true> : k_place<false>, dim3(b.sc.blocks256 + extra), dim3(kHashBlock), 0, s,
                       b.sc, b.key, b.rank, b.range, b.slot_tmp, b.crowd, b.crowd_count, b.crowd_cap, b.error_flag,
                       tile_work(b, tiles));
    return hipGetLastError();
}

hipError_t launch_gather(const DeviceBuffers& b, const TileShape* tiles, hipStream_t s) {
    if (b.sc.blocks256 == 0) return hipSuccess;
    static_assert(kCrowdBlocks % kNumXcd == 0, "the leading workgroups keep the XCD mapping of the others");
    const unsigned extra = tiles ? tile_grid(b) : 0u;
    hipLaunchKernelGGL(tiles ? k_gather<true> : k_gather<false>, dim3(b.sc.blocks256 + kCrowdBlocks + extra),
                       dim3(kHashBlock), 0, s, b.sc, b.slot_tmp, b.key, b.range, b.posrho[0], b.velp[0], b.posrho[1],
                       b.velp[1], b.sorted, b.skey, b.ids[0], b.ids[1], b.rho_max + 1, b.crowd, b.crowd_count,
                       b.crowd_cap, tile_work(b, tiles));
    return hipGetLastError();
}

// Tuning variants of the two neighbour passes: (block size, LDS list entries per lane, slots
// in flight per lane, drain after every dx plane).  Every variant computes identical bits.
#define WC_VARIANTS(X)     \
    X(256, 32, 4, true)    \
    X(128, 32, 4, true)    \
    X(64, 32, 4, true)     \
    X(64, 32, 8, true)     \
    X(64, 40, 4, false)    \
    X(64, 48, 4, false)    \
    X(64, 64, 4, false)    \
    X(128, 48, 4, false)   \
    X(128, 32, 2, true)    \
    X(64, 40, 8, false)    \
    X(128, 32, 8, true)

static const PassVariant kVariants[] = {
#define WC_ROW(B, C, K, P) {B, C, K, P},
    WC_VARIANTS(WC_ROW)
#undef WC_ROW
    {0, 0, 0, false},  // the tile passes: no particle a lane, workgroup and lists by the context's box and size
};

int num_variants() { return (int)(sizeof(kVariants) / sizeof(kVariants[0])); }
int tile_variant() { return num_variants() - 1; }
PassVariant variant(int v) { return kVariants[(v >= 0 && v < num_variants()) ? v : 0]; }

static unsigned pass_blocks(const Scenes& S, int block) {
    return block == 64 ? S.blocks64 : (block == 128 ? S.blocks128 : S.blocks256);
}

hipError_t launch_density(const DeviceBuffers& b, int v, bool list, hipStream_t s) {
    const PassVariant pv = variant(v);
    const unsigned blocks = pass_blocks(b.sc, pv.block);
    if (blocks == 0) return hipSuccess;
    if (list && (!b.nlist || !b.ncount)) return hipErrorInvalidValue;
#define WC_LAUNCH(B, C, K, P)                                                                             \
    if (pv.block == B && pv.list_cap == C && pv.chunk == K && pv.plane_drain == P) {                     \
        if (list)                                                                                         \
            hipLaunchKernelGGL((k_density<B, C, K, P, true>), dim3(blocks), dim3(B), 0, s, b.sc, b.posrho[1], \
                               b.velp[1], b.skey, b.range, b.rho_max, b.nlist, b.ncount);                  \
        else                                                                                              \
            hipLaunchKernelGGL((k_density<B, C, K, P, false>), dim3(blocks), dim3(B), 0, s, b.sc, b.posrho[1],\
                               b.velp[1], b.skey, b.range, b.rho_max, nullptr, nullptr);                   \
        return hipGetLastError();                                                                         \
    }
    WC_VARIANTS(WC_LAUNCH)
#undef WC_LAUNCH
    return hipErrorInvalidValue;
}

hipError_t launch_update(const DeviceBuffers& b, int v, bool list, hipStream_t s) {
    const PassVariant pv = variant(v);
    const unsigned blocks = pass_blocks(b.sc, pv.block);
    if (blocks == 0) return hipSuccess;
    if (list && (!b.nlist || !b.ncount)) return hipErrorInvalidValue;
#define WC_LAUNCH(B, C, K, P)                                                                             \
    if (pv.block == B && pv.list_cap == C && pv.chunk == K && pv.plane_drain == P) {                     \
        if (list)                                                                                         \
            hipLaunchKernelGGL((k_update<B, C, K, P, 0, true>), dim3(blocks), dim3(B), 0, s, b.sc,         \
                               b.posrho[1], b.velp[1], b.skey, b.range, b.posrho[0], b.velp[0],            \
                               b.scene_done, b.ids[1], b.ids[0], 0.0f, nullptr, 0.0f, nullptr, b.nlist,    \
                               b.ncount, 0.0f, b.rho_max + 1, RecordBackup{});                                  \
        else                                                                                              \
            hipLaunchKernelGGL((k_update<B, C, K, P, 0, false>), dim3(blocks), dim3(B), 0, s, b.sc,        \
                               b.posrho[1], b.velp[1], b.skey, b.range, b.posrho[0], b.velp[0],            \
                               b.scene_done, b.ids[1], b.ids[0], 0.0f, nullptr, 0.0f, nullptr, nullptr,    \
                               nullptr, 0.0f, b.rho_max + 1, RecordBackup{});                                   \
        return hipGetLastError();                                                                         \
    }
    WC_VARIANTS(WC_LAUNCH)
#undef WC_LAUNCH
    return hipErrorInvalidValue;
}

// The two sizes of a tile workgroup: threads, staged records (then: waves per SIMD to compile for).
#define WC_TILE_LARGE kTileLargeBlock, kTileLargeCap
#define WC_TILE_SMALL kTileSmallBlock, kTileSmallCap

template <int BLOCK, int CAP, int WPE>
static void density_tile(const DeviceBuffers& b, bool list, hipStream_t s) {
    if (list)
        hipLaunchKernelGGL((k_density_tile<BLOCK, CAP, WPE, true>), dim3(tile_grid(b)), dim3(BLOCK), 0, s, b.sc,
                           b.tiles, b.tile_count, b.tile_cap, reinterpret_cast<const BoxTable*>(b.tables), b.table_cap,
                           b.sparse, b.posrho[1], b.velp[1], b.skey, b.range, b.rho_max, b.llist, b.lcount, b.list_cap,
                           b.list_chunks, b.nlist, b.ncount);
    else
        hipLaunchKernelGGL((k_density_tile<BLOCK, CAP, WPE, false>), dim3(tile_grid(b)), dim3(BLOCK), 0, s, b.sc,
                           b.tiles, b.tile_count, b.tile_cap, reinterpret_cast<const BoxTable*>(b.tables), b.table_cap,
                           b.sparse, b.posrho[1], b.velp[1], b.skey, b.range, b.rho_max, b.llist, b.lcount, b.list_cap,
                           b.list_chunks, nullptr, nullptr);
}

hipError_t launch_density_tile(const DeviceBuffers& b, const TileShape& t, bool list, hipStream_t s) {
    if (list && (!b.nlist || !b.ncount)) return hipErrorInvalidValue;
    if (t.block == kTileLargeBlock)
        density_tile<WC_TILE_LARGE, 6>(b, list, s);
    else
        density_tile<WC_TILE_SMALL, 3>(b, list, s);
    return hipGetLastError();
}

template <int BLOCK, int CAP, int WPE, int MODE>
static void update_tile(const DeviceBuffers& b, const TileUpdate& u, hipStream_t s) {
    hipLaunchKernelGGL((k_update_tile<BLOCK, CAP, WPE, MODE>), dim3(tile_grid(b)), dim3(BLOCK), 0, s, b.sc, b.tiles,
                       b.tile_count, b.tile_cap, reinterpret_cast<const BoxTable*>(b.tables), b.table_cap, b.sparse,
                       b.posrho[1], b.velp[1], b.skey, b.range, b.posrho[0], b.velp[0], b.scene_done, b.ids[1],
                       b.ids[0], b.llist, b.lcount, b.list_cap, b.list_chunks, b.rho_max + 1, u.dt,
                       reinterpret_cast<const float4*>(u.corr), u.corr_scale, reinterpret_cast<float4*>(u.acc_out),
                       u.substeps, u.backup);
}

hipError_t launch_update_tile(const DeviceBuffers& b, const TileShape& t, const TileUpdate& u, hipStream_t s) {
    if (t.block == kTileLargeBlock && u.learned)
        update_tile<WC_TILE_LARGE, 2, 1>(b, u, s);
    else if (t.block == kTileLargeBlock)
        update_tile<WC_TILE_LARGE, 2, 0>(b, u, s);
    else if (u.learned)
        update_tile<WC_TILE_SMALL, 2, 1>(b, u, s);
    else
        update_tile<WC_TILE_SMALL, 2, 0>(b, u, s);
    return hipGetLastError();
}

hipError_t launch_closure_features(const DeviceBuffers& b, const uint32_t* rows, uint32_t nrows, float dt_mult,
                                   uint16_t* X, bool lists, hipStream_t s) {
    if (nrows == 0) return hipSuccess;
    if (lists && (!b.nlist || !b.ncount)) return hipErrorInvalidValue;
    if (lists) {
        hipLaunchKernelGGL(k_closure_features_short, dim3(blocks_for(nrows, 256)), dim3(256), 0, s, b.sc, b.posrho[1],
                           b.velp[1], rows, nrows, dt_mult, X, b.nlist, b.ncount);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_closure_features, dim3(blocks_for(nrows, kFeatBlock)), dim3(kFeatBlock), 0, s, b.sc,
                       b.posrho[1], b.velp[1], b.skey, b.range, rows, nrows, dt_mult, X,
                       lists ? b.nlist : nullptr, lists ? b.ncount : nullptr, lists, nullptr, nullptr);
    return hipGetLastError();
}

hipError_t launch_closure_selection(const DeviceBuffers& b, uint32_t n, uint32_t* sel, uint32_t* heavy,
                                    uint32_t* heavy_count, hipStream_t s) {
    if (n == 0) return hipSuccess;
    if (!b.nlist || !b.ncount || !sel || !heavy || !heavy_count) return hipErrorInvalidValue;
    // a kernel clears the count (no memset node in a captured graph); the register selection runs
    // on every slot and lists the rare longer rows, which the walk then takes on a small grid
    hipLaunchKernelGGL(k_clear_word, dim3(1), dim3(64), 0, s, heavy_count);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_closure_select, dim3(blocks_for(n, 256)), dim3(256), 0, s, b.posrho[1], n, b.nlist, b.ncount,
                       (size_t)b.sc.total_particles, sel, heavy, heavy_count);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_closure_features, dim3(kHeavyBlocks), dim3(kFeatBlock), 0, s, b.sc, b.posrho[1], b.velp[1],
                       b.skey, b.range, heavy, n, 0.0f, nullptr, b.nlist, b.ncount, true, sel, heavy_count);
    return hipGetLastError();
}

hipError_t launch_closure_update(const DeviceBuffers& b, float dt, const float* corr, float corr_scale,
                                 float* acc_out, bool smooth, float substeps, bool lists, hipStream_t s,
                                 const RecordBackup& backup) {
    if (b.sc.blocks64 == 0) return hipSuccess;
    if (lists && (!b.nlist || !b.ncount)) return hipErrorInvalidValue;
    if (lists) {
        if (smooth)
            hipLaunchKernelGGL((k_update<64, 32, 4, true, 2, true>), dim3(b.sc.blocks64), dim3(64), 0, s, b.sc,
                               b.posrho[1], b.velp[1], b.skey, b.range, b.posrho[0], b.velp[0], b.scene_done,
                               b.ids[1], b.ids[0], dt, reinterpret_cast<const float4*>(corr), corr_scale,
                               reinterpret_cast<float4*>(acc_out), b.nlist, b.ncount, substeps, b.rho_max + 1, backup);
        else
            hipLaunchKernelGGL((k_update<64, 32, 4, true, 1, true>), dim3(b.sc.blocks64), dim3(64), 0, s, b.sc,
                               b.posrho[1], b.velp[1], b.skey, b.range, b.posrho[0], b.velp[0], b.scene_done,
                               b.ids[1], b.ids[0], dt, reinterpret_cast<const float4*>(corr), corr_scale,
                               reinterpret_cast<float4*>(acc_out), b.nlist, b.ncount, substeps, b.rho_max + 1, backup);
        return hipGetLastError();
    }
    if (smooth)
        hipLaunchKernelGGL((k_update<64, 32, 4, true, 2, false>), dim3(b.sc.blocks64), dim3(64), 0, s, b.sc,
                           b.posrho[1], b.velp[1], b.skey, b.range, b.posrho[0], b.velp[0], b.scene_done, b.ids[1],
                           b.ids[0], dt, reinterpret_cast<const float4*>(corr), corr_scale,
                           reinterpret_cast<float4*>(acc_out), nullptr, nullptr, substeps, b.rho_max + 1, backup);
    else
        hipLaunchKernelGGL((k_update<64, 32, 4, true, 1, false>), dim3(b.sc.blocks64), dim3(64), 0, s, b.sc,
                           b.posrho[1], b.velp[1], b.skey, b.range, b.posrho[0], b.velp[0], b.scene_done, b.ids[1],
                           b.ids[0], dt, reinterpret_cast<const float4*>(corr), corr_scale,
                           reinterpret_cast<float4*>(acc_out), nullptr, nullptr, substeps, b.rho_max + 1, backup);
    return hipGetLastError();
}

hipError_t launch_noalloc_setup(const SceneDesc& d, const uint32_t tables_host[8], SceneDesc* desc,
                                uint32_t* tables, uint32_t* counts, uint32_t ncells, uint32_t* error_flag,
                                hipStream_t s) {
    const uint4 t0 = make_uint4(tables_host[0], tables_host[1], tables_host[2], tables_host[3]);
    const uint4 t1 = make_uint4(tables_host[4], tables_host[5], tables_host[6], tables_host[7]);
    unsigned blocks = blocks_for(ncells, kHashBlock);
    blocks = blocks < 1 ? 1 : (blocks > 256 ? 256 : blocks);
    hipLaunchKernelGGL(k_noalloc_setup, dim3(blocks), dim3(kHashBlock), 0, s, d, t0, t1, desc, tables, counts, ncells,
                       error_flag);
    return hipGetLastError();
}

hipError_t launch_invalidate(const DeviceBuffers& b, hipStream_t s) {
    const unsigned blocks = b.sc.blocks256 ? b.sc.blocks256 : 1;  // block 0 always marks the flags
    hipLaunchKernelGGL(k_invalidate, dim3(blocks), dim3(kHashBlock), 0, s, b.sc, b.posrho[1], b.skey, b.ncount,
                       b.rho_max + 1);
    return hipGetLastError();
}

hipError_t launch_advect(const DeviceBuffers& b, float dt, hipStream_t s) {
    if (b.sc.blocks256 == 0) return hipSuccess;
    hipLaunchKernelGGL(k_advect, dim3(b.sc.blocks256), dim3(kHashBlock), 0, s, b.sc, b.posrho[0], b.velp[0], dt);
    return hipGetLastError();
}

hipError_t launch_split_records(const wc_particle* rec, float4* posrho, float4* velp, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_split, dim3(blocks_for(n, kHashBlock)), dim3(kHashBlock), 0, s,
                       reinterpret_cast<const float4*>(rec), posrho, velp, n);
    return hipGetLastError();
}

hipError_t launch_join_records(const float4* posrho, const float4* velp, wc_particle* rec, uint32_t n,
                               hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_join, dim3(blocks_for(n, kHashBlock)), dim3(kHashBlock), 0, s, posrho, velp,
                       reinterpret_cast<float4*>(rec), n);
    return hipGetLastError();
}

}  // namespace wc
