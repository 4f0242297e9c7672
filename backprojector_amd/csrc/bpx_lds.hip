// LDS-staged confocal gather with polynomial quotients (gfx950): flat wall, voxel columns
// along the wall normal.
//
// A 256-lane work-group owns a 16 x 16 x KZ voxel tile, a lane one (x, y) column of KZ voxels.
// Per pair the tile's bin window is copied from the fused rows to LDS by direct-to-LDS loads,
// and every update reads its element (threshold, both candidate samples) from there.
//
// The approximate quotient of an update only has to come within 1/2 of the exact one: the
// threshold comparison then decides the bin exactly from the update's own squared distance.
// Along a column the quotient is smooth, q(rho) = inv2 sqrt(axy + (u - rho step)^2) + w with rho
// the voxel's offset from the column's centre, so one reciprocal square root per (lane, pair)
// gives its Taylor coefficients and each update evaluates a polynomial in a compile-time rho
// (1.5 or 2 v_fmamk_f32, the even and odd parts shared by rho and -rho) instead of a
// v_sqrt_f32 and a v_fma_f32.  The host bounds the polynomial's error (lds_poly_shape).
#include <algorithm>
#include <cmath>

#include "bpx_lds.hpp"

// dst = VCC ? high half of src : low half of src, zero-extended
#define SEL16(dst, src)                                                                         \
    "v_cndmask_b32_sdwa " dst ", " src ", " src ", vcc dst_sel:DWORD dst_unused:UNUSED_PAD "   \
    "src0_sel:WORD_0 src1_sel:WORD_1"

namespace bpx {

namespace {

// Count rows: samples are integers 0 .. 2048 (16 bits each), summed as integers: exact in any
// order, one register per voxel and no compensation.  column() adds KZ updates: element e[i] =
// (S, lo | hi << 16) of voxel r = column_order(i) gives lo where s < S and hi elsewhere, s = axy + dz2[r].  Each update is a
// compare, a select whose SDWA word selects move the chosen half into place, an add, and the add
// that makes the next update's s; written in one chain so that the two wait states the select
// needs after the compare (and the one the add needs after the select) hold the neighbours' adds.
struct CountRows {
    using acc_t = uint32_t;
    template <int KZ>
    __device__ static __forceinline__ void column(acc_t (&acc)[KZ], const uint2 (&e)[KZ], float axy,
                                                  const float (&dz2)[KZ]) {
        float s = axy + dz2[column_order<KZ>(0)];
        uint32_t h;
        asm("v_cmp_ge_f32_e32 vcc, %1, %2\n\ts_nop 1\n\t" SEL16("%0", "%3")
            : "=v"(h) : "v"(s), "v"(e[0].x), "v"(e[0].y) : "vcc");
#pragma unroll
        for (int i = 1; i < KZ; ++i) {
            const int r = column_order<KZ>(i), prev = column_order<KZ>(i - 1);
            s = axy + dz2[r];
            uint32_t hn;
            asm("v_cmp_ge_f32_e32 vcc, %2, %3\n\t"
                "v_add_u32_e32 %0, %0, %5\n\t"
                "s_nop 0\n\t" SEL16("%1", "%4")
                : "+&v"(acc[prev]), "=v"(hn) : "v"(s), "v"(e[i].x), "v"(e[i].y), "v"(h) : "vcc");
            h = hn;
        }
        acc[column_order<KZ>(KZ - 1)] += h;
    }
};

}  // namespace

// Pairs per part of a listed tile: the launch's work-groups spread over the listed tiles, at most
// 8 parts of at least 128 pairs.
__device__ __forceinline__ uint32_t list_part_pairs(uint32_t P, uint32_t count, uint32_t groups) {
    const uint32_t parts = max(1u, min(min(groups / max(count, 1u), 8u), P / 128u));
    return ((P + parts - 1u) / parts + 3u) / 4u * 4u;
}

template <class Fz, int KZ, int DEG, bool TILES>
__global__ __launch_bounds__(256, 4) void confocal_lds_kernel_poly(LdsPolyArgs a) {
    constexpr uint32_t NW = 4, PS = NW;   // waves; pairs per stage (one per wave)
    using Off = ElemOffset<8>;
    using acc_t = typename Fz::acc_t;
    if (!rows_wanted(a.c)) return;
    extern __shared__ char smem[];   // [2][PS][seg] 8-byte elements, then [2][PS] pair records
    const uint32_t slot_bytes = a.seg * 8u, lds0 = lds_offset(smem);
    float4* const meta = reinterpret_cast<float4*>(smem + 2u * PS * slot_bytes);
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const Grid& g = a.c.g;
    const uint32_t n0 = g.n[0], n1 = g.n[1], n2 = g.n[2], tiles = poly_tiles(g, KZ);
    // every tile of the grid, or those of a list whose length is on the device (then the launch is
    // fixed and its work-groups are shared out here)
    const uint32_t count = TILES ? __builtin_amdgcn_readfirstlane(*a.n_tiles) : tiles;
    const uint32_t part_pairs = TILES ? list_part_pairs(a.c.P, count, gridDim.x) : a.part_pairs;
    const uint32_t part = count ? blockIdx.x / count : 0u, index = count ? blockIdx.x % count : 0u;
    if (TILES && (count == 0u || part * part_pairs >= a.c.P)) return;
    const uint32_t tile = TILES ? __builtin_amdgcn_readfirstlane(a.tiles[index]) : xcd_remap(index, tiles);
    const uint32_t p0 = part * part_pairs, p1 = min(p0 + part_pairs, a.c.P);
    const ColumnTile<KZ> t(g, tile, w, lane);
    float dz2[KZ];   // uniform
#pragma unroll
    for (int r = 0; r < KZ; ++r) {
        float v[3];
        voxel_position(g, t.cx, t.cy, t.iz0 + r, v);
        const float dz = a.c.lz - v[2];
        dz2[r] = uniform_f32(dz * dz);
    }
    const float u = t.centre(g, a.c.lz), u2 = u * u;
    const TileBox<KZ> box(g, t, a.c.lz);
    const uint32_t row_bytes = a.c.ldh * 8u;
    const uint32_t nstage = (p1 - p0 + PS - 1u) / PS;

    // Windows and pair records, 64 stages of this wave at a time (one pair per lane): lane L holds
    // the wave's pair of stage base + L.
    float mx = 0.0f, my = 0.0f, mw = 0.0f;
    int mjl = 0, mcnt = 0;
    auto plan_windows = [&](uint32_t base) {
        const uint32_t st = base + lane, p = p0 + st * PS + w;
        mcnt = 0;
        mjl = 0;
        if (p < p1) {
            const float4 pr = a.c.pairs[p];
            float smin, smax;
            box.distances(pr.x, pr.y, smin, smax);
            // 2 elements of margin each way; the start even, so that a 16-byte load never
            // straddles a row end
            const int jl = ((int)__builtin_fmaf(__builtin_amdgcn_sqrtf(smin), a.c.inv2, pr.w) - 2) & ~1;
            const int jh = (int)__builtin_fmaf(__builtin_amdgcn_sqrtf(smax), a.c.inv2, pr.w) + 2;
            mjl = jl;
            mcnt = min(jh + 2 - jl, (int)a.seg);
            mx = pr.x;
            my = pr.y;
            mw = pr.w + (float)(int)((((st & 1u) * PS + w) * a.seg) - (uint32_t)jl + (lds0 >> 3) + (uint32_t)Off::kBias);
        }
    };
    auto stage = [&](uint32_t b) {
        const uint32_t sl = b & 63u;
        if (sl == 0u) plan_windows(b);
        const uint32_t slot = (b & 1u) * PS + w;
        const int jl = __builtin_amdgcn_readlane(mjl, sl), cnt = __builtin_amdgcn_readlane(mcnt, sl);
        if (lane == sl) meta[slot] = make_float4(mx, my, mw, 0.0f);
        const __amdgpu_buffer_rsrc_t rr =
            make_rsrc(static_cast<const char*>(a.c.H) + (size_t)(p0 + b * PS + w) * row_bytes, row_bytes);
        const int vo = jl * 8 + (int)lane * 16;
        const uint32_t base = lds0 + slot * slot_bytes;
        for (int m = 0; m < cnt; m += 128) load_lds16(rr, base + (uint32_t)m * 8u, vo + m * 8);
    };

    acc_t acc[KZ];
#pragma unroll
    for (int r = 0; r < KZ; ++r) acc[r] = 0;
    auto pair_step = [&](const float4 m) {
        const float dx = m.x - t.vx, dy = m.y - t.vy;
        const float axy = dx * dx + dy * dy;
        const ColumnQuotient<KZ, DEG> q(axy, u, u2, a.c.inv2, a.k1, a.k2, a.k3, m.z);
        uint2 e[KZ];
#pragma unroll
        for (int i = 0; i < KZ; ++i) e[i] = lds_read8(Off::of(q.at(i)));
        __builtin_amdgcn_sched_barrier(0);
        Fz::template column<KZ>(acc, e, axy, dz2);
    };
    if (nstage) stage(0u);
    wait_loads();
    __syncthreads();
    for (uint32_t b = 0; b < nstage; ++b) {
        if (b + 1u < nstage) stage(b + 1u);
        const float4* mb = meta + (b & 1u) * PS;
        const uint32_t np = min(PS, p1 - p0 - b * PS);
        float4 m = mb[0];
#pragma unroll 1
        for (uint32_t i = 0; i < np; ++i) {
            const float4 next = mb[i + 1u < PS ? i + 1u : i];
            pair_step(m);
            m = next;
        }
        wait_loads();
        __syncthreads();
    }
    if (TILES) {   // [work-group = part x listed tiles + index][voxel of the column][lane]
        uint32_t* o = a.parts + (size_t)blockIdx.x * (256u * KZ) + threadIdx.x;
#pragma unroll
        for (int r = 0; r < KZ; ++r) o[256u * r] = acc[r];
    } else if (t.ix < n0 && t.iy < n1) {
        const size_t id = t.id(g);
        if (a.parts) {
            uint32_t* o = a.parts + (size_t)part * n0 * n1 * n2 + id;
#pragma unroll
            for (int r = 0; r < KZ; ++r) o[r] = acc[r];
        } else {
            float* o = static_cast<float*>(a.c.out) + id;
#pragma unroll
            for (int r = 0; r < KZ; ++r) o[r] = (float)acc[r];
        }
    }
}

// The volume from the integer partial sums of every part.
__global__ __launch_bounds__(256) void lds_parts_sum_kernel(LdsPolyArgs a, uint32_t parts, uint64_t n) {
    if (!rows_wanted(a.c)) return;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t v = 0;
        for (uint32_t k = 0; k < parts; ++k) v += a.parts[(size_t)k * n + i];
        static_cast<float*>(a.c.out)[i] = (float)v;
    }
}

// Voxel (x, y, z) in the tiles of the kernel above: tile, lane of its column and place in it.
struct TileVoxel {
    uint32_t tile, lane, r;
};
template <int KZ>
__device__ __forceinline__ TileVoxel tile_voxel(const Grid& g, uint32_t x, uint32_t y, uint32_t z) {
    const uint32_t ntz = (g.n[2] + KZ - 1u) / KZ, nty = (g.n[1] + 15u) / 16u;
    const uint32_t tz = z / KZ;
    TileVoxel t;
    t.tile = ((x >> 4) * nty + (y >> 4)) * ntz + tz;
    t.lane = (((y >> 3) & 1u) * 2u + ((x >> 3) & 1u)) * 64u + (y & 7u) * 8u + (x & 7u);
    t.r = z - min(tz * KZ, g.n[2] - KZ);
    return t;
}

// Marks the listed voxels: one bit per voxel (16 per column of a tile) and the number per tile.
// Lists follow the octree's blocks, so a wave's voxels share few tiles; the counters are updated
// once per (wave, tile).
template <int KZ>
__global__ __launch_bounds__(256) void tile_mark_kernel(TileListArgs a, const uint32_t* __restrict__ voxels, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    TileVoxel t{0xffffffffu, 0u, 0u};
    if (i < n) {
        const uint32_t v = voxels[i];
        t = tile_voxel<KZ>(a.g, v & 1023u, (v >> 10) & 1023u, v >> 20);
        const uint32_t col = t.tile * 256u + t.lane;
        atomicOr(&a.mask[col >> 1], 1u << (t.r + 16u * (col & 1u)));
    }
    bool left = i < n;
    while (__ballot(left) != 0ull) {
        const uint32_t first = (uint32_t)__builtin_ctzll(__ballot(left));
        const uint32_t tile = __builtin_amdgcn_readlane(t.tile, first);
        const bool mine = left && t.tile == tile;
        const uint64_t m = __ballot(mine);
        if ((threadIdx.x & 63u) == first) atomicAdd(&a.fill[tile], (uint32_t)__builtin_popcountll(m));
        left = left && !mine;
    }
}
// Tiles with at least `dense` listed voxels, in any order (each is computed by itself).
__global__ __launch_bounds__(256) void tile_pick_kernel(TileListArgs a, uint32_t tiles, uint32_t dense) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < tiles && a.fill[i] >= dense) a.tiles[atomicAdd(&a.counts[0], 1u)] = i;
}
// The listed voxels of the other tiles, 64 neighbours of the list at a time.
template <int KZ>
__global__ __launch_bounds__(256) void tile_rest_kernel(TileListArgs a, const uint32_t* __restrict__ voxels, uint32_t n,
                                                        uint32_t dense) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63u;
    uint32_t v = 0;
    bool rest = false;
    if (i < n) {
        v = voxels[i];
        rest = a.fill[tile_voxel<KZ>(a.g, v & 1023u, (v >> 10) & 1023u, v >> 20).tile] < dense;
    }
    const uint64_t m = __ballot(rest);
    uint32_t base = 0;
    if (lane == 0u && m) base = atomicAdd(&a.counts[1], (uint32_t)__builtin_popcountll(m));
    base = __builtin_amdgcn_readfirstlane(base);
    if (rest) a.rest[base + (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1ull))] = v;
}
// Volume values of the marked voxels of the listed tiles from their integer partial sums.
template <int KZ>
__global__ __launch_bounds__(256) void tile_store_kernel(TileListArgs a, LdsPolyArgs p, uint32_t groups) {
    const uint32_t count = a.counts[0];
    if (blockIdx.x >= count) return;
    const uint32_t part_pairs = list_part_pairs(p.c.P, count, groups), parts = (p.c.P + part_pairs - 1u) / part_pairs;
    const uint32_t tile = a.tiles[blockIdx.x], col = tile * 256u + threadIdx.x;
    const uint32_t bits = a.mask[col >> 1] >> (16u * (col & 1u)) & 0xffffu;
    if (!bits) return;
    const uint32_t ntz = (a.g.n[2] + KZ - 1u) / KZ, nty = (a.g.n[1] + 15u) / 16u;
    const uint32_t tz = tile % ntz, ty = tile / ntz % nty, tx = tile / ntz / nty, w = threadIdx.x >> 6;
    const uint32_t ix = tx * 16u + (w & 1u) * 8u + (threadIdx.x & 7u), iy = ty * 16u + (w >> 1) * 8u + ((threadIdx.x >> 3) & 7u);
    float* out = static_cast<float*>(p.c.out) + ((size_t)ix * a.g.n[1] + iy) * a.g.n[2] + min(tz * KZ, a.g.n[2] - KZ);
    for (int r = 0; r < KZ; ++r)
        if (bits >> r & 1u) {
            uint32_t v = 0;
            for (uint32_t k = 0; k < parts; ++k)
                v += p.parts[((size_t)k * count + blockIdx.x) * (256u * KZ) + 256u * r + threadIdx.x];
            out[r] = (float)v;
        }
}

template <int KZ, int DEG, bool TILES>
static hipError_t poly_launch(const LdsPolyArgs& a, uint32_t groups, hipStream_t s) {
    const auto fn = confocal_lds_kernel_poly<CountRows, KZ, DEG, TILES>;
    const size_t lds = 2u * 4u * ((size_t)a.seg * 8u + sizeof(float4));
    if (lds > 64u * 1024u) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3(groups), dim3(256), lds, s, a);
    return hipGetLastError();
}
template <bool TILES>
static hipError_t poly_launch_shape(const LdsPolyArgs& a, const LdsPolyShape& sh, uint32_t groups, hipStream_t s) {
    if (sh.kz == 16) return sh.deg == 2 ? poly_launch<16, 2, TILES>(a, groups, s) : poly_launch<16, 3, TILES>(a, groups, s);
    return sh.deg == 2 ? poly_launch<8, 2, TILES>(a, groups, s) : poly_launch<8, 3, TILES>(a, groups, s);
}
LdsPolyArgs lds_poly_args(const ConfocalArgs& c, const LdsPolyShape& sh) {
    LdsPolyArgs a{};
    a.c = c;
    a.seg = sh.seg;
    const double step = c.g.inc[8], A = c.inv2;
    a.k1 = (float)(-A * step);
    a.k2 = (float)(A * step * step / 2.0);
    a.k3 = (float)(A * step * step * step / 2.0);
    return a;
}
hipError_t launch_lds_counts(const LdsPolyArgs& a, const LdsPolyShape& sh, uint32_t parts, hipStream_t s) {
    const hipError_t e = poly_launch_shape<false>(a, sh, (uint32_t)poly_tiles(a.c.g, sh.kz) * parts, s);
    if (e != hipSuccess || !a.parts) return e;
    const uint64_t n = (uint64_t)a.c.g.n[0] * a.c.g.n[1] * a.c.g.n[2];
    hipLaunchKernelGGL(lds_parts_sum_kernel, dim3((uint32_t)std::min<uint64_t>((n + 255u) / 256u, 4096u)), dim3(256), 0,
                       s, a, parts, n);
    return hipGetLastError();
}

uint64_t lds_tile_count(const Grid& g, const LdsPolyShape& sh) { return poly_tiles(g, sh.kz); }

template <int KZ>
static hipError_t tile_lists(const TileListArgs& a, const uint32_t* const lists[2], const uint32_t n[2], uint32_t dense,
                             hipStream_t s) {
    const uint32_t tiles = (uint32_t)poly_tiles(a.g, KZ);
    for (int k = 0; k < 2; ++k)
        if (n[k]) hipLaunchKernelGGL(tile_mark_kernel<KZ>, dim3((n[k] + 255u) / 256u), dim3(256), 0, s, a, lists[k], n[k]);
    hipLaunchKernelGGL(tile_pick_kernel, dim3((tiles + 255u) / 256u), dim3(256), 0, s, a, tiles, dense);
    for (int k = 0; k < 2; ++k)
        if (n[k])
            hipLaunchKernelGGL(tile_rest_kernel<KZ>, dim3((n[k] + 255u) / 256u), dim3(256), 0, s, a, lists[k], n[k], dense);
    return hipGetLastError();
}
hipError_t launch_tile_lists(const TileListArgs& a, const LdsPolyShape& sh, const uint32_t* const lists[2],
                             const uint32_t n[2], uint32_t dense, hipStream_t s) {
    return sh.kz == 16 ? tile_lists<16>(a, lists, n, dense, s) : tile_lists<8>(a, lists, n, dense, s);
}
hipError_t launch_lds_counts_tiles(LdsPolyArgs a, const LdsPolyShape& sh, const TileListArgs& t, uint32_t max_tiles,
                                   uint32_t groups, hipStream_t s) {
    a.tiles = t.tiles;
    a.n_tiles = t.counts;
    const hipError_t e = poly_launch_shape<true>(a, sh, groups, s);
    if (e != hipSuccess) return e;
    if (sh.kz == 16) hipLaunchKernelGGL(tile_store_kernel<16>, dim3(max_tiles), dim3(256), 0, s, t, a, groups);
    else hipLaunchKernelGGL(tile_store_kernel<8>, dim3(max_tiles), dim3(256), 0, s, t, a, groups);
    return hipGetLastError();
}

// Error of the column polynomial against the quotient, in bins.  With f(z) = sqrt(a + z^2),
// g = 1 / f and t = z g, the third derivative over 6 is -t (1 - t^2) g^2 / 2 and the fourth over 24
// (1 - t^2)(5 t^2 - 1) g^3 / 8; g = t / z, so over every a >= 0 they stay within 0.0930 / z^2 and
// 0.0559 / z^3.  A column of half length h around its centre, at least zmin from the wall: the cubic
// Taylor polynomial is within 0.0559 h^4 / zmin^3 (Lagrange's remainder), and replacing c3 rho^3 by
// its best linear approximation adds c3 h^3 / 4.  In use the polynomial's value rounds to 1/8 four
// times (w, c0, the even part, the sum: 1/16 each), so the bound on the approximate quotient
// (`bound`, which covers the arithmetic of its terms) and the polynomial's error must stay below
// 1/4 together (`budget`; the window kernel's end edge rounds a fifth time: 3/16).
LdsPolyShape lds_poly_shape(const Grid& g, float inv2, float lz, double bound, double max_path, double budget) {
    LdsPolyShape none;
    // column along z alone; coordinates whose squares and reciprocals stay normal floats
    if (g.inc[2] != 0.0f || g.inc[5] != 0.0f || g.inc[6] != 0.0f || g.inc[7] != 0.0f) return none;
    const double step = std::fabs((double)g.inc[8]), A = std::fabs((double)inv2);
    const double za = (double)lz - g.zero[2], zb = za - (double)g.inc[8] * (double)(g.n[2] - 1u);
    const double zmin = std::min(std::fabs(za), std::fabs(zb)) * (1.0 - 1e-5);
    if (!(za * zb > 0.0) || !(zmin > 1e-12) || !(max_path < 1e12) || !(step > 0.0)) return none;
    for (int kz : {16, 8}) {
        if (g.n[2] < (uint32_t)kz) continue;
        const double h = 0.5 * (kz - 1) * step;
        const double e3 = A * 0.0559 * h * h * h * h / (zmin * zmin * zmin);
        const double e2 = e3 + A * 0.0930 * h * h * h / (4.0 * zmin * zmin);
        const double limit = budget - bound;
        const int deg = e2 <= limit ? 2 : e3 <= limit ? 3 : 0;
        if (!deg) continue;
        double d2 = 0.0;
        for (int k = 0; k < 3; ++k) {
            const double r = 15.0 * (std::fabs((double)g.inc[k]) + std::fabs((double)g.inc[3 + k])) +
                             (kz - 1.0) * std::fabs((double)g.inc[6 + k]);
            d2 += r * r;
        }
        // as confocal_lds_fits, with one more element for the even start
        const double need = std::ceil(std::sqrt(d2) * A * (1.0 + 1e-6)) + 9.0;
        if (!(need <= (double)kPolySegMax)) continue;
        LdsPolyShape sh;
        sh.kz = kz;
        sh.deg = deg;
        sh.seg = ((uint32_t)need + 127u) / 128u * 128u;
        return sh;
    }
    return none;
}

// Parts the pairs are split into (integer sums are exact, so the split does not change the
// volume): towards 4,096 work-groups while each keeps 128 pairs, and 1,024 (4 on each of 256 CUs)
// while each keeps 32; at most 64 MiB of partial sums.  Measured: 16,384 pairs into 128^3 (512
// tiles) 8.65 ms in 1 part, 6.85 in 2, 6.42 in 4, 6.08 in 8, 6.11 in 16 -- more rounds of resident
// work-groups even out the last one; 1,961 pairs into 45 x 61 x 38 (60 tiles) 0.107 ms in 9 parts,
// 0.082 in 18, 0.087 in 61.
uint32_t lds_poly_parts(const Grid& g, const LdsPolyShape& sh, uint32_t P, uint32_t sum_bytes, uint32_t* part_pairs) {
    const uint64_t tiles = poly_tiles(g, sh.kz), vox = (uint64_t)g.n[0] * g.n[1] * g.n[2];
    uint64_t parts = std::max(std::min<uint64_t>((4096u + tiles - 1u) / tiles, P / 128u),
                              std::min<uint64_t>((1024u + tiles - 1u) / tiles, P / 32u));
    parts = std::max<uint64_t>(1u, std::min<uint64_t>(parts, (64ull << 20) / (sum_bytes * vox)));
    *part_pairs = (uint32_t)(((P + parts - 1u) / parts + 3u) / 4u * 4u);
    return std::max(1u, (P + *part_pairs - 1u) / *part_pairs);
}

}  // namespace bpx
