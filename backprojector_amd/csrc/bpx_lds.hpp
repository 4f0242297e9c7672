// Device pieces of the LDS-staged gathers whose work-groups own 16 x 16 x KZ voxel tiles, a lane one
// (x, y) column of KZ voxels along the wall normal: tile geometry, bin windows, the polynomial
// quotient of a column, direct-to-LDS loads.
#pragma once
#include "bpx_device.hpp"

namespace bpx {

typedef __attribute__((address_space(3))) void lds_void;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t lds_offset(const void* p) { return (uint32_t)(uintptr_t)(lds_void*)p; }
__device__ __forceinline__ uint2 lds_read8(uint32_t off) {
    const u32x2 v = *(const __attribute__((address_space(3))) u32x2*)(uintptr_t)off;
    return make_uint2(v[0], v[1]);
}
__device__ __forceinline__ float lds_read4(uint32_t off) {
    return *(const __attribute__((address_space(3))) float*)(uintptr_t)off;
}
__device__ __forceinline__ double lds_read_f64(uint32_t off) {
    return *(const __attribute__((address_space(3))) double*)(uintptr_t)off;
}
__device__ __forceinline__ float uniform_f32(float x) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
}
__device__ __forceinline__ double uniform_f64(double x) {
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b), hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}

// 16 bytes per lane from the buffer at byte offset `off` (0 past its end) to LDS at
// lds_base + 16 lane.  The load has no register output; its issuer waits for vmcnt before the
// barrier that publishes the data.  (Written out because the compiler orders the builtin's load
// before every later LDS read it cannot tell apart, which would drain the loads of the next stage
// before the current stage's gathers.)
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, uint32_t lds_base, int off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :: "s"(lds_base), "v"(off), "s"(r) : "m0", "memory");
}
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__host__ __device__ inline uint32_t poly_tiles(const Grid& g, int kz) {
    return ((g.n[0] + 15u) / 16u) * ((g.n[1] + 15u) / 16u) * ((g.n[2] + (uint32_t)kz - 1u) / (uint32_t)kz);
}

// A tile and one lane's column in it.
template <int KZ>
struct ColumnTile {
    uint32_t tx, ty, ix, iy, iz0, cx, cy;
    float vx, vy;
    // The wave's 8 x 8 columns all lie past the grid (uniform): it stages with the others and skips
    // the updates, which leaves its issue slots to them.
    bool idle;
    __device__ __forceinline__ ColumnTile(const Grid& g, uint32_t tile, uint32_t w, uint32_t lane) {
        const uint32_t ntz = (g.n[2] + KZ - 1u) / KZ, nty = (g.n[1] + 15u) / 16u;
        const uint32_t tz = tile % ntz, txy = tile / ntz;
        ty = txy % nty;
        tx = txy / nty;
        ix = tx * 16u + (w & 1u) * 8u + (lane & 7u);
        iy = ty * 16u + (w >> 1) * 8u + (lane >> 3);
        idle = tx * 16u + (w & 1u) * 8u >= g.n[0] || ty * 16u + (w >> 1) * 8u >= g.n[1];
        iz0 = min(tz * KZ, g.n[2] - KZ);   // the last slab reaches back over its neighbour
        cx = min(ix, g.n[0] - 1u);
        cy = min(iy, g.n[1] - 1u);
        float v[3];
        voxel_position(g, cx, cy, iz0, v);
        vx = v[0];
        vy = v[1];
    }
    // wall distance (signed) of the columns' centre, uniform
    __device__ __forceinline__ float centre(const Grid& g, float lz) const {
        return lz - (g.zero[2] + g.inc[8] * ((float)iz0 + 0.5f * (float)(KZ - 1)));
    }
    __device__ __forceinline__ size_t id(const Grid& g) const { return ((size_t)ix * g.n[1] + iy) * g.n[2] + iz0; }
};

// Bounding box of a tile's voxels (coordinates are monotone in each index, so the extremes are at
// the corners) and the squared distances of its nearest and farthest point from a wall point.
template <int KZ>
struct TileBox {
    float bmin[3], bmax[3], ez2, fz2;
    __device__ __forceinline__ TileBox(const Grid& g, const ColumnTile<KZ>& t, float lz) {
        const uint32_t x0 = min(t.tx * 16u, g.n[0] - 1u), x1 = min(t.tx * 16u + 15u, g.n[0] - 1u);
        const uint32_t y0 = min(t.ty * 16u, g.n[1] - 1u), y1 = min(t.ty * 16u + 15u, g.n[1] - 1u);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            bmin[k] = __builtin_inff();
            bmax[k] = -__builtin_inff();
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            float v[3];
            voxel_position(g, (c & 1) ? x1 : x0, (c & 2) ? y1 : y0, (c & 4) ? t.iz0 + KZ - 1u : t.iz0, v);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                bmin[k] = fminf(bmin[k], v[k]);
                bmax[k] = fmaxf(bmax[k], v[k]);
            }
        }
        const float ez = lz - fminf(fmaxf(lz, bmin[2]), bmax[2]);
        const float fz = fmaxf(fabsf(lz - bmin[2]), fabsf(lz - bmax[2]));
        ez2 = ez * ez;
        fz2 = fz * fz;
    }
    __device__ __forceinline__ void distances(float x, float y, float& smin, float& smax) const {
        const float ex = x - fminf(fmaxf(x, bmin[0]), bmax[0]), ey = y - fminf(fmaxf(y, bmin[1]), bmax[1]);
        const float fx = fmaxf(fabsf(x - bmin[0]), fabsf(x - bmax[0])), fy = fmaxf(fabsf(y - bmin[1]), fabsf(y - bmax[1]));
        smin = (ex * ex + ey * ey) + ez2;
        smax = (fx * fx + fy * fy) + fz2;
    }
};

// Voxels of a column from the centre outwards.
template <int KZ>
__device__ constexpr int column_order(int i) {
    return (i & 1) ? KZ / 2 - 1 - i / 2 : KZ / 2 + i / 2;
}

// The approximate quotient inv2 sqrt(axy + (u - rho step)^2) + w along a column, rho the offset from
// its centre in voxels: Taylor coefficients from one reciprocal square root (k1 .. k3: LdsPolyArgs),
// evaluated at compile-time rho, the even part shared by rho and -rho.  at(i): the value of
// voxel column_order(i).
template <int KZ, int DEG>
struct ColumnQuotient {
    float c0, c1, c2, c3;
    __device__ __forceinline__ ColumnQuotient(float axy, float u, float u2, float inv2, float k1, float k2, float k3, float w) {
        const float s0 = axy + u2;
        const float gi = __builtin_amdgcn_rsqf(s0);
        const float t = u * gi;                    // cosine to the wall normal
        const float q = gi - (t * t) * gi;         // (1 - t^2) / d
        c0 = __builtin_fmaf(s0 * gi, inv2, w);
        c2 = q * k2;
        c3 = (q * t) * (gi * k3);
        c1 = t * k1;
        constexpr float kTop = 0.5f * (float)(KZ - 1);
        if (DEG == 2) c1 = __builtin_fmaf(c3, 0.75f * kTop * kTop, c1);   // best linear part of c3 rho^3
    }
    __device__ __forceinline__ float at(int i) const {
        const float rho = 0.5f + (float)(i / 2);
        const float ev = __builtin_fmaf(c2, rho * rho, c0);
        const float od = DEG == 3 ? __builtin_fmaf(c3, rho * rho, c1) : c1;
        return __builtin_fmaf(od, (i & 1) ? -rho : rho, ev);
    }
};

}  // namespace bpx
