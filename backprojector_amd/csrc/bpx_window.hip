// CPU-path semantics (backproject.hpp:75-96) for confocal pairs, a flat wall and voxel columns along
// its normal: the LDS-staged form of window_kernel, with the same window edges and prefix sums.
//
// Per pair and voxel the edges are bins of total = (lw + float(2 d)) + cw, d = sqrt(s) correctly
// rounded from the double s = (x x + y y) + z z of float differences: both edges are monotone step
// functions of s.  window_table_kernel finds, per pair and bin, the smallest double s that reaches
// the bin (the start's and the end's edge), so the gather neither takes a double root nor rounds a
// path: it forms s with one double add, guesses both bins with the polynomial quotient of
// bpx_lds.hip, settles each with one double comparison, and reads the two prefix sums.
//
// Per pair a 16 x 16 x KZ voxel tile stages three windows in LDS by direct-to-LDS loads: the two
// threshold tables and the prefix sums between the first start and the last end.  An update costs
// four 8-byte LDS reads, about as long as its arithmetic (both near 70 cycles per 64 updates, 98
// measured); the double root and the scattered prefix reads of window_kernel cost 417.  9,216 pairs
// into 96^3: 21.6 -> 5.07 ms, and 0.18 ms for the tables.
#include <algorithm>
#include <cmath>

#include "bpx_lds.hpp"

namespace bpx {

namespace {

// The smallest float path wvw with (lw + wvw) + cw >= z.
struct PathPred {
    float lw, cw, z;
    __device__ bool operator()(uint32_t key) const {
        float total = lw + fkey_inv(key);
        total = total + cw;
        return total >= z;
    }
};

__device__ __forceinline__ double next_up(double x, int64_t k) {   // k units in the last place, x > 0
    return __longlong_as_double(__double_as_longlong(x) + k);
}

// The smallest double s >= 0 with (lw + float(2 sqrt_rn(s))) + cw >= z.
__device__ double window_threshold(float lw, float cw, float z) {
    const double gd = ((double)z - (double)lw) - (double)cw;
    const float g = gd > 0.0 ? (float)gd : 0.0f;
    const float w = fkey_inv(min_true_key_near(PathPred{lw, cw, z}, fkey(g), fkey(0.0f), fkey(__builtin_inff())));
    if (!(w > 0.0f)) return 0.0;
    if (!(w <= 0x1p60f)) return __builtin_inf();
    // smallest double D = 2 d with float(D) >= w: the midpoint m below w (exact in double) when
    // ties go to w (even mantissa), else the double above it
    const float below = __uint_as_float(__float_as_uint(w) - 1u);
    const double m = 0.5 * ((double)w + (double)below);
    const double d = 0.5 * ((__float_as_uint(w) & 1u) ? next_up(m, 1) : m);
    // smallest s with sqrt_rn(s) >= d: within a few units of d d (its predecessor's square is
    // d d - d ulp(d), 1 to 2 units away)
    const double s0 = d * d;
    if (!(s0 > 0x1p-900)) return 0.0;   // below any distance the plan admits
    int64_t lo = -4, hi = 4;
    while (__builtin_sqrt(next_up(s0, lo)) >= d) lo -= 4;
    while (!(__builtin_sqrt(next_up(s0, hi)) >= d)) hi += 4;
    while (hi - lo > 1) {
        const int64_t mid = (lo + hi) >> 1;
        if (__builtin_sqrt(next_up(s0, mid)) >= d) hi = mid;
        else lo = mid;
    }
    return next_up(s0, hi);
}

}  // namespace

// Slo / Shi [P][pitch], entries of bins 1 .. T - 1 that some voxel of the grid can guess (the bins
// over the grid's bounding box, 6 wider each way); the others are never compared with.
__global__ __launch_bounds__(256) void window_table_kernel(WindowLdsArgs a, double* Slo, double* Shi) {
    const uint32_t p = blockIdx.x;
    const float4 pr = a.pairs[p];
    const float lw = a.pair8[8u * p + 7u], cw = a.pair8[8u * p + 6u];
    float near2 = 0.0f, far2 = 0.0f;
    const float c[3] = {pr.x, pr.y, a.lz};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float v0 = a.g.zero[k], v1 = a.g.zero[k] + a.g.inc[4 * k] * (float)(a.g.n[k] - 1u);
        const float lo = fminf(v0, v1), hi = fmaxf(v0, v1);
        const float e = c[k] - fminf(fmaxf(c[k], lo), hi), f = fmaxf(fabsf(c[k] - lo), fabsf(c[k] - hi));
        near2 += e * e;
        far2 += f * f;
    }
    const float qn = sqrtf(near2) * a.inv2 * 0.9999f + pr.w, qf = sqrtf(far2) * a.inv2 * 1.0001f + pr.w;
    for (int kind = 0; kind < 2; ++kind) {
        const float* Z = kind ? a.Zhi : a.Zlo;
        double* S = (kind ? Shi : Slo) + (size_t)p * a.pitch;
        const float shift = kind ? a.width_bins : 0.0f;
        const int j0 = (int)fminf(fmaxf(qn + shift - 6.0f, 1.0f), (float)a.T);
        const int j1 = (int)fminf(fmaxf(qf + shift + 6.0f, 0.0f), (float)a.T - 1.0f);
        for (int j = j0 + (int)threadIdx.x; j <= j1; j += 256) S[j] = window_threshold(lw, cw, Z[j]);
    }
}

template <int KZ, int DEG>
__global__ __launch_bounds__(256, 3) void window_lds_kernel(WindowLdsArgs a) {
    constexpr uint32_t PS = 2;   // pairs per stage: two waves copy one pair's windows
    using Off = ElemOffset<8>;
    extern __shared__ char smem[];   // [2][PS] slots of (2 seg + seg_sums) doubles, then [2][PS] records
    const uint32_t slot_elems = 2u * a.seg + a.seg_sums, lds0 = lds_offset(smem);
    float4* const meta = reinterpret_cast<float4*>(smem + 2u * PS * slot_elems * 8u);
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t n0 = a.g.n[0], n1 = a.g.n[1];
    const uint32_t tiles = poly_tiles(a.g, KZ), part = blockIdx.x / tiles;
    const ColumnTile<KZ> t(a.g, xcd_remap(blockIdx.x % tiles, tiles), w, lane);
    const uint32_t p0 = part * a.part_pairs, p1 = min(p0 + a.part_pairs, a.P);
    double z2[KZ];   // uniform
#pragma unroll
    for (int r = 0; r < KZ; ++r) {
        float v[3];
        voxel_position(a.g, t.cx, t.cy, t.iz0 + r, v);
        const double dz = (double)(a.lz - v[2]);
        z2[r] = uniform_f64(dz * dz);
    }
    const float u = t.centre(a.g, a.lz), u2 = u * u;
    const TileBox<KZ> box(a.g, t, a.lz);
    const uint32_t nstage = (p1 - p0 + PS - 1u) / PS;

    float mx = 0.0f, my = 0.0f, mw = 0.0f, on = 0.0f;
    int mjl = 0, mcnt = 0;
    auto plan_windows = [&](uint32_t base) {
        const uint32_t st = base + lane, k = w >> 1, p = p0 + st * PS + k;
        mcnt = 0;
        on = 0.0f;
        if (p < p1) {
            const float4 pr = a.pairs[p];
            float smin, smax;
            box.distances(pr.x, pr.y, smin, smax);
            const int jl = ((int)__builtin_fmaf(__builtin_amdgcn_sqrtf(smin), a.inv2, pr.w) - 2) & ~1;
            const int jh = (int)__builtin_fmaf(__builtin_amdgcn_sqrtf(smax), a.inv2, pr.w) + 2;
            // every window wholly before bin 0 or past the last bin: both edges clamp to the same
            // bin and the pair adds nothing
            if (jl <= (int)a.T && jh + (int)a.shift + 4 >= 0) {
                mjl = jl;
                mcnt = min(jh + 2 - jl, (int)a.seg);
                on = 1.0f;
            }
            mx = pr.x;
            my = pr.y;
            mw = pr.w + (float)(int)((((st & 1u) * PS + k) * slot_elems) - (uint32_t)jl + (lds0 >> 3) + (uint32_t)Off::kBias);
        }
    };
    auto stage = [&](uint32_t b) {
        const uint32_t sl = b & 63u, k = w >> 1;
        if (sl == 0u) plan_windows(b);
        const uint32_t slot = (b & 1u) * PS + k;
        const int jl = __builtin_amdgcn_readlane(mjl, sl), cnt = __builtin_amdgcn_readlane(mcnt, sl);
        if (lane == sl && !(w & 1u)) meta[slot] = make_float4(mx, my, mw, on);
        if (cnt == 0) return;
        const size_t p = p0 + b * PS + k;
        const uint32_t base = lds0 + slot * slot_elems * 8u;
        auto copy = [&](const double* row, uint32_t row_elems, int first, int count, uint32_t to) {
            const __amdgpu_buffer_rsrc_t r = make_rsrc(row, row_elems * 8u);
            const int vo = first * 8 + (int)lane * 16;
            for (int m = 0; m < count; m += 128) load_lds16(r, to + (uint32_t)m * 8u, vo + m * 8);
        };
        if (w & 1u) {   // sums from two bins before the first start's, to the last end's
            copy(a.PS + p * a.ldp, a.ldp, jl - 2, min(cnt + (int)a.shift + 6, (int)a.seg_sums), base + a.seg * 16u);
        } else {
            copy(a.Slo + p * a.pitch, a.pitch, jl, cnt, base);
            copy(a.Shi + p * a.pitch, a.pitch, jl + (int)a.shift, cnt, base + a.seg * 8u);
        }
    };

    double acc[KZ];
#pragma unroll
    for (int r = 0; r < KZ; ++r) acc[r] = 0.0;
    // byte distance from a threshold's element to the sum of the bin below it, and of its bin
    const uint32_t dlo = (2u * a.seg + 1u) * 8u, dhi = (a.seg + a.shift + 1u) * 8u;
    auto pair_step = [&](const float4 m) {
        const float dx = m.x - t.vx, dy = m.y - t.vy;
        const double ddx = (double)dx, ddy = (double)dy, axy = ddx * ddx + ddy * ddy;
        const ColumnQuotient<KZ, DEG> q(dx * dx + dy * dy, u, u2, a.inv2, a.k1, a.k2, a.k3, m.z);
#pragma unroll
        for (int half = 0; half < KZ; half += 8) {
            uint32_t olo[8], ohi[8];
            double slo[8], shi[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float y = q.at(half + i);
                olo[i] = Off::of(y);
                ohi[i] = Off::of(y + a.hi_offset);
                slo[i] = lds_read_f64(olo[i]);
                shi[i] = lds_read_f64(ohi[i]);
            }
            __builtin_amdgcn_sched_barrier(0);
            double first[8], last[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const double s = axy + z2[column_order<KZ>(half + i)];
                first[i] = lds_read_f64(olo[i] + (s >= slo[i] ? dlo + 8u : dlo));
                last[i] = lds_read_f64(ohi[i] + (s >= shi[i] ? dhi + 8u : dhi));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[column_order<KZ>(half + i)] += last[i] - first[i];
        }
    };
    if (nstage) stage(0u);
    wait_loads();
    __syncthreads();
    for (uint32_t b = 0; b < nstage; ++b) {
        if (b + 1u < nstage) stage(b + 1u);
        const float4* mb = meta + (b & 1u) * PS;
        const uint32_t np = t.idle ? 0u : min(PS, p1 - p0 - b * PS);
#pragma unroll 1
        for (uint32_t i = 0; i < np; ++i) {
            const float4 m = mb[i];
            if (__builtin_amdgcn_readfirstlane(__float_as_uint(m.w))) pair_step(m);
        }
        wait_loads();
        __syncthreads();
    }
    if (t.ix < n0 && t.iy < n1) {
        const size_t id = t.id(a.g), n = (size_t)n0 * n1 * a.g.n[2];
#pragma unroll
        for (int r = 0; r < KZ; ++r) {
            if (a.parts) a.parts[(size_t)part * n + id + r] = acc[r];
            else a.out[id + r] = (float)acc[r];
        }
    }
}

__global__ __launch_bounds__(256) void window_parts_sum_kernel(const double* __restrict__ parts, uint32_t count,
                                                               uint64_t n, float* __restrict__ out) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        double v = parts[i];
        for (uint32_t k = 1; k < count; ++k) v += parts[(size_t)k * n + i];
        out[i] = (float)v;
    }
}

size_t window_lds_bytes(const WindowLdsArgs& a) { return 4u * ((2u * (size_t)a.seg + a.seg_sums) * 8u + sizeof(float4)); }

template <int KZ, int DEG>
static hipError_t window_launch(const WindowLdsArgs& a, uint32_t parts, hipStream_t s) {
    const auto fn = window_lds_kernel<KZ, DEG>;
    const size_t lds = window_lds_bytes(a);
    if (lds > 64u * 1024u) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, dim3(poly_tiles(a.g, KZ) * parts), dim3(256), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_window_tables(const WindowLdsArgs& a, double* Slo, double* Shi, hipStream_t s) {
    hipLaunchKernelGGL(window_table_kernel, dim3(a.P), dim3(256), 0, s, a, Slo, Shi);
    return hipGetLastError();
}
hipError_t launch_window_lds(const WindowLdsArgs& a, const LdsPolyShape& sh, uint32_t parts, hipStream_t s) {
    const hipError_t e = sh.kz == 16 ? (sh.deg == 2 ? window_launch<16, 2>(a, parts, s) : window_launch<16, 3>(a, parts, s))
                                     : (sh.deg == 2 ? window_launch<8, 2>(a, parts, s) : window_launch<8, 3>(a, parts, s));
    if (e != hipSuccess || !a.parts) return e;
    const uint64_t n = (uint64_t)a.g.n[0] * a.g.n[1] * a.g.n[2];
    hipLaunchKernelGGL(window_parts_sum_kernel, dim3((uint32_t)std::min<uint64_t>((n + 255u) / 256u, 4096u)), dim3(256), 0,
                       s, a.parts, parts, n, a.out);
    return hipGetLastError();
}

}  // namespace bpx
