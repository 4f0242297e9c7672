// LDS-staged gather of non-confocal captures (laser and SPAD points apart), single tap: exhaustive
// laser x SPAD grids and arbitrary pair lists, real samples.
//
// A 256-lane work-group owns a 16 x 16 x KZ voxel tile, a lane one (x, y) column.  The bin of an
// update is decided by its exact fp32 path ((lw + d1) + d2) + cw against the path-length thresholds
// Z (kept whole in LDS), as in grid_kernel and pairs_kernel; the samples come from LDS copies of
// each pair's bin window over the tile (the tile's nearest and farthest points from both legs bound
// it), made by direct-to-LDS loads straight from the unpadded rows: bins outside the row lie
// outside the row's buffer descriptor and read as 0.
//
// What bounds it: an update is two 4-byte LDS reads (threshold, then sample: 8 to 13 LDS cycles a
// wave) and about 36 cycles of arithmetic; pair lists add two correctly rounded roots (exact_root:
// 25 cycles each, against about 60 for the compiler's sequence, which also covers arguments that
// cannot occur here).  The texture-path kernels are held by 22 texture-address cycles a wave.
// Pairs are split over work-groups where the tiles alone leave the chip idle; parts are added in
// double.
#include <algorithm>
#include <cmath>

#include "bpx_lds.hpp"

namespace bpx {

namespace {

// sqrtf correctly rounded for s in [2^-100, 2^100]: one Newton step on s rsqrt(s), its residual
// exact in the first fma, one rounding in the second.  Compared on gfx950 with the root in double,
// rounded, for each of the 1.7e9 floats of that range: no difference.
__device__ __forceinline__ float exact_root(float s) {
    const float r = __builtin_amdgcn_rsqf(s);
    const float g = s * r, h = 0.5f * r;
    const float e = __builtin_fmaf(-g, g, s);
    return __builtin_fmaf(e, h, g);
}

__device__ __forceinline__ float lds_read_f32(uint32_t off) {
    return *(const __attribute__((address_space(3))) float*)(uintptr_t)off;
}

// Distances of a box's nearest and farthest point from a point.
__device__ __forceinline__ void box_range(const float bmin[3], const float bmax[3], float x, float y, float z, float& dmin,
                                          float& dmax) {
    const float c[3] = {x, y, z};
    float a = 0.0f, b = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float e = c[k] - fminf(fmaxf(c[k], bmin[k]), bmax[k]), f = fmaxf(fabsf(c[k] - bmin[k]), fabsf(c[k] - bmax[k]));
        a += e * e;
        b += f * f;
    }
    dmin = __builtin_amdgcn_sqrtf(a);
    dmax = __builtin_amdgcn_sqrtf(b);
}

}  // namespace

// GRID: pair p = l C + c; a part takes a range of lasers and, 8 SPADs at a time, walks its lasers with
// the 8 SPAD legs of its voxels in registers.  Otherwise a part takes a range of pairs, both legs per
// update.  A stage is 8 pairs, two copied by each wave, double-buffered.  FINE: compensated adds within a
// grid's stages, for blocks of fewer than 8 pairs.
template <bool GRID, int KZ, bool FINE>
__global__ __launch_bounds__(256, GRID ? 2 : 3) void paths_lds_kernel(PathsLdsArgs a) {
    constexpr uint32_t CS = 8;
    constexpr int kNoWindow = (int)0x80000000;
    using Off = ElemOffset<8>;
    // [2][CS][seg] samples, Z [Tc + 1], then seg floats that hold the windows' records: a guess up to
    // a window's length before the row or past its end still reads inside the allocation
    extern __shared__ char smem[];
    const uint32_t zlen = (a.Tc + 1u + 63u) / 64u * 64u;
    const uint32_t rows0 = lds_offset(smem), z0 = rows0 + 2u * CS * a.seg * 4u;
    float* const zs = reinterpret_cast<float*>(smem) + 2u * CS * a.seg;
    int2* const win = reinterpret_cast<int2*>(zs + zlen);            // [2][CS]: W, threshold distance
    float4* const rec = reinterpret_cast<float4*>(win + 2u * CS);    // [2][CS][2], pair lists only
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    for (uint32_t j = threadIdx.x; j <= a.Tc; j += 256u) zs[j] = a.Z[j];
    const uint32_t tiles = poly_tiles(a.g, KZ), part = blockIdx.x / tiles;
    const ColumnTile<KZ> t(a.g, xcd_remap(blockIdx.x % tiles, tiles), w, lane);
    float vz[KZ];
#pragma unroll
    for (int r = 0; r < KZ; ++r) {
        float v[3];
        voxel_position(a.g, t.cx, t.cy, t.iz0 + r, v);
        vz[r] = v[2];
    }
    const TileBox<KZ> box(a.g, t, 0.0f);
    // stages of this part: GRID [chunk of 8 SPADs][laser], else [8 pairs]
    const uint32_t first = part * a.part_units, end = min(first + a.part_units, GRID ? a.L : a.P);
    if (first >= end) return;
    const uint32_t lasers = end - first, nstage = GRID ? (a.C + CS - 1u) / CS * lasers : (end - first + CS - 1u) / CS;
    // pair of slot c of stage st, and its points (laser, SPAD; w: wall distances)
    auto pair_of = [&](uint32_t st, uint32_t c, float4& lp, float4& cp) -> uint32_t {
        if (GRID) {
            const uint32_t l = first + st % lasers, s = st / lasers * CS + c;
            if (s >= a.C) return 0xffffffffu;
            lp = a.lasers[l];
            cp = a.spads[s];
            return l * a.C + s;
        }
        const uint32_t p = first + st * CS + c;
        if (p >= end) return 0xffffffffu;
        const float* q = a.pairs + 8u * (size_t)p;
        cp = make_float4(q[0], q[1], q[2], q[6]);
        lp = make_float4(q[3], q[4], q[5], q[7]);
        return p;
    };
    // the windows of this wave's two pairs of 32 stages, one pair a lane: pair, first bin + 1, count
    uint32_t mp = 0;
    int mjl = 0, mcnt = 0;
    float4 mlp = make_float4(0, 0, 0, 0), mcp = make_float4(0, 0, 0, 0);
    auto plan_windows = [&](uint32_t st0) {
        const uint32_t st = st0 + (lane >> 1), c = 2u * w + (lane & 1u);
        mp = st < nstage ? pair_of(st, c, mlp, mcp) : 0xffffffffu;
        mcnt = 0;
        mjl = 0;
        if (mp != 0xffffffffu) {
            float n1, f1, n2, f2;
            box_range(box.bmin, box.bmax, mlp.x, mlp.y, mlp.z, n1, f1);
            box_range(box.bmin, box.bmax, mcp.x, mcp.y, mcp.z, n2, f2);
            const float walls = mlp.w + mcp.w;
            // padded element j (bin j - 1) and its neighbour, 2 elements of margin each way; raw
            // sample index j - 1 a multiple of 4, so that no 16-byte load straddles the row's start
            const int jl = (((int)__builtin_fmaf(walls + (n1 + n2), a.inv, a.c1) - 4) & ~3) + 1;
            const int jh = (int)__builtin_fmaf(walls + (f1 + f2), a.inv, a.c1) + 3;
            mjl = jl;
            // (windows wholly before or past the row add nothing: count 0)
            if (jh >= 0 && jl <= (int)a.Tc + 1) mcnt = min(jh + 2 - jl, (int)a.seg);
        }
    };
    auto stage = [&](uint32_t b) {
        if ((b & 31u) == 0u) plan_windows(b);
#pragma unroll
        for (uint32_t k = 0; k < 2; ++k) {
            const uint32_t src = 2u * (b & 31u) + k, slot = (b & 1u) * CS + 2u * w + k;
            const uint32_t p = __builtin_amdgcn_readlane(mp, src);
            const int jl = __builtin_amdgcn_readlane(mjl, src), cnt = __builtin_amdgcn_readlane(mcnt, src);
            const uint32_t to = rows0 + slot * a.seg * 4u;
            if (lane == src) {
                // W: biased quotient -> the window's element in LDS; distance from there to Z[j]
                const float W = a.c1 + (float)(int)((to >> 2) - (uint32_t)jl + (uint32_t)Off::kBias);
                win[slot] = make_int2(__float_as_int(W), cnt > 0 ? (int)(z0 - to) + jl * 4 : kNoWindow);
                if (!GRID) {
                    rec[2u * slot] = mlp;
                    rec[2u * slot + 1u] = mcp;
                }
            }
            const __amdgpu_buffer_rsrc_t r =
                make_rsrc(reinterpret_cast<const char*>(a.rows) + (size_t)(cnt > 0 ? p : 0u) * a.Tc * 4u, a.Tc * 4u);
            const int vo = (jl - 1) * 4 + (int)lane * 16;
            for (int m = 0; m < cnt; m += 256) load_lds16(r, to + (uint32_t)m * 4u, vo + m * 4);
        }
    };

    float sum[KZ], comp[KZ], blk[KZ];
#pragma unroll
    for (int r = 0; r < KZ; ++r) sum[r] = comp[r] = blk[r] = 0.0f;
    uint32_t since = 0;
    auto settle = [&](uint32_t n) {
        since += n;
        if (since >= a.kahan_block) {
            since = 0;
#pragma unroll
            for (int r = 0; r < KZ; ++r) {
                kahan_add(sum[r], comp[r], blk[r]);
                blk[r] = 0.0f;
            }
        }
    };
    // One pair's updates from its exact paths: padded element j = floor(q) of the pair's window (not
    // clamped: elements outside the row are 0) from the mantissa of the biased quotient, whose two
    // roundings to 1/8 come on top of the quotient's bound (< 1/4); element j + [total >= Z[j]].
    auto taps = [&](const float (&total)[KZ], int2 m) {
        uint32_t o[KZ];
        float z[KZ];
#pragma unroll
        for (int r = 0; r < KZ; ++r) {
            o[r] = Off::of(__builtin_fmaf(total[r], a.inv, __int_as_float(m.x))) >> 1;
            z[r] = lds_read_f32(o[r] + (uint32_t)m.y);
        }
        float h[KZ];
#pragma unroll
        for (int r = 0; r < KZ; ++r) h[r] = lds_read_f32(o[r] + (total[r] >= z[r] ? 4u : 0u));
#pragma unroll
        for (int r = 0; r < KZ; ++r) blk[r] = blk[r] + h[r];
    };
    float d2[GRID ? CS : 1][KZ], cw[GRID ? CS : 1];
    stage(0u);
    wait_loads();
    __syncthreads();
    for (uint32_t b = 0; b < nstage; ++b) {
        if (b + 1u < nstage) stage(b + 1u);
        const uint32_t sl = (b & 1u) * CS;
        if constexpr (GRID) {
            const uint32_t chunk = b / lasers, l = first + b % lasers;
            if (b % lasers == 0u && !t.idle) {
#pragma unroll
                for (uint32_t c = 0; c < CS; ++c) {
                    const float4 sp = a.spads[min(chunk * CS + c, a.C - 1u)];
                    cw[c] = sp.w;
                    const float x = t.vx - sp.x, y = t.vy - sp.y, xy = x * x + y * y;
#pragma unroll
                    for (int r = 0; r < KZ; ++r) {
                        const float z = vz[r] - sp.z;
                        d2[c][r] = exact_root(xy + z * z);
                    }
                }
            }
            const float4 lp = a.lasers[l];
            const float x = lp.x - t.vx, y = lp.y - t.vy, xy = x * x + y * y;
            float d1[KZ];
#pragma unroll
            for (int r = 0; r < KZ; ++r) {
                const float z = lp.z - vz[r];
                d1[r] = lp.w + exact_root(xy + z * z);
            }
            const uint32_t n = t.idle ? 0u : min(CS, a.C - chunk * CS);
#pragma unroll
            for (uint32_t c = 0; c < CS; ++c)
                if (const int2 m = win[sl + c]; c < n && __builtin_amdgcn_readfirstlane(m.y) != kNoWindow) {
                    float total[KZ];
#pragma unroll
                    for (int r = 0; r < KZ; ++r) {
                        total[r] = d1[r] + d2[c][r];
                        total[r] = total[r] + cw[c];
                    }
                    taps(total, m);
                    if (FINE) settle(1u);
                }
            if (!FINE) settle(n);
        } else {
            const uint32_t n = t.idle ? 0u : min(CS, end - first - b * CS);
#pragma unroll 1
            for (uint32_t c = 0; c < n; ++c) {
                const int2 m = win[sl + c];
                const float4 lp = rec[2u * (sl + c)], cp = rec[2u * (sl + c) + 1u];
                if (__builtin_amdgcn_readfirstlane(m.y) == kNoWindow) continue;
                const float x1 = lp.x - t.vx, y1 = lp.y - t.vy, xy1 = x1 * x1 + y1 * y1;
                const float x2 = t.vx - cp.x, y2 = t.vy - cp.y, xy2 = x2 * x2 + y2 * y2;
                float total[KZ];
#pragma unroll
                for (int r = 0; r < KZ; ++r) {
                    const float z1 = lp.z - vz[r], z2 = vz[r] - cp.z;
                    total[r] = lp.w + exact_root(xy1 + z1 * z1);
                    total[r] = total[r] + exact_root(xy2 + z2 * z2);
                    total[r] = total[r] + cp.w;
                }
                taps(total, m);
                settle(1u);
            }
        }
        wait_loads();
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < KZ; ++r) kahan_add(sum[r], comp[r], blk[r]);
    if (t.ix < a.g.n[0] && t.iy < a.g.n[1]) {
        const size_t id = t.id(a.g), n = (size_t)a.g.n[0] * a.g.n[1] * a.g.n[2];
#pragma unroll
        for (int r = 0; r < KZ; ++r) {
            if (a.parts) a.parts[(size_t)part * n + id + r] = (double)sum[r] - (double)comp[r];
            else a.out[id + r] = kahan_result(sum[r], comp[r]) * a.scale;
        }
    }
}

__global__ __launch_bounds__(256) void paths_parts_sum_kernel(const double* __restrict__ parts, uint32_t count, uint64_t n,
                                                              float scale, float* __restrict__ out) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        double v = parts[i];
        for (uint32_t k = 1; k < count; ++k) v += parts[(size_t)k * n + i];
        out[i] = (float)v * scale;
    }
}

// 16-bit storage: the rows as the storage format holds them, back in fp32.
__global__ __launch_bounds__(256) void quantise_rows_kernel(const float* __restrict__ src, uint64_t n, int format,
                                                            float inv_scale, float* __restrict__ dst) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const float x = src[i] * inv_scale;
        if (format == kF16) {
            dst[i] = (float)(_Float16)x;
        } else {
            const uint32_t u = __float_as_uint(x);
            const uint32_t q = (u & 0x7fffffffu) > 0x7f800000u ? (u | 0x400000u) : u + 0x7fffu + ((u >> 16) & 1u);
            dst[i] = __uint_as_float(q & 0xffff0000u);
        }
    }
}
hipError_t launch_quantise_rows(const float* src, uint64_t n, int format, float inv_scale, float* dst, hipStream_t s) {
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((n + 255u) / 256u, 16384u);
    hipLaunchKernelGGL(quantise_rows_kernel, dim3(blocks), dim3(256), 0, s, src, n, format, inv_scale, dst);
    return hipGetLastError();
}

size_t paths_lds_bytes(const PathsLdsArgs& a) {
    // (the records take 640 bytes of the last seg floats)
    return 4u * ((size_t)((a.Tc + 1u + 63u) / 64u * 64u) + 17u * (size_t)a.seg);
}

template <bool GRID, bool FINE>
static hipError_t paths_launch(const PathsLdsArgs& a, uint32_t parts, hipStream_t s) {
    const auto fn = paths_lds_kernel<GRID, 8, FINE>;
    const size_t lds = paths_lds_bytes(a);
    if (lds > 64u * 1024u) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3(poly_tiles(a.g, 8) * parts), dim3(256), lds, s, a);
    if (hipError_t e = hipGetLastError(); e != hipSuccess || !a.parts) return e;
    const uint64_t n = (uint64_t)a.g.n[0] * a.g.n[1] * a.g.n[2];
    hipLaunchKernelGGL(paths_parts_sum_kernel, dim3((uint32_t)std::min<uint64_t>((n + 255u) / 256u, 4096u)), dim3(256), 0, s,
                       a.parts, parts, n, a.scale, a.out);
    return hipGetLastError();
}
hipError_t launch_paths_lds(const PathsLdsArgs& a, uint32_t parts, hipStream_t s) {
    if (!a.L) return paths_launch<false, false>(a, parts, s);
    return a.kahan_block < 8u ? paths_launch<true, true>(a, parts, s) : paths_launch<true, false>(a, parts, s);
}

}  // namespace bpx
