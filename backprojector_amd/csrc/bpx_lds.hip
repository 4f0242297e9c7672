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
// the same into the high half of dst, zero below
#define SEL16_HIGH(dst, src)                                                                    \
    "v_cndmask_b32_sdwa " dst ", " src ", " src ", vcc dst_sel:WORD_1 dst_unused:UNUSED_PAD "  \
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
    static constexpr int kFormat = kCount;
    using part_t = uint32_t;
    template <int KZ>
    struct Acc {
        uint32_t sum[KZ];
        __device__ __forceinline__ void end_pair(uint32_t) {}
        __device__ __forceinline__ void finish() {}
        __device__ __forceinline__ uint32_t part(int r) const { return sum[r]; }
        __device__ __forceinline__ void store(const ConfocalArgs& a, size_t id, int r) const {
            static_cast<float*>(a.out)[id] = (float)sum[r];
        }
    };
    template <int KZ>
    __device__ static __forceinline__ void column(Acc<KZ>& acc, const uint2 (&e)[KZ], float axy,
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
                : "+&v"(acc.sum[prev]), "=v"(hn) : "v"(s), "v"(e[i].x), "v"(e[i].y), "v"(h) : "vcc");
            h = hn;
        }
        acc.sum[column_order<KZ>(KZ - 1)] += h;
    }
    template <int KZ, int DEG>
    __device__ static __forceinline__ void pair(Acc<KZ>& acc, const ColumnQuotient<KZ, DEG>& q, float axy,
                                                const float (&dz2)[KZ], uint32_t) {
        uint2 e[KZ];
#pragma unroll
        for (int i = 0; i < KZ; ++i) e[i] = lds_read8(ElemOffset<8>::of(q.at(i)));
        __builtin_amdgcn_sched_barrier(0);
        column<KZ>(acc, e, axy, dz2);
    }
};

// Real and complex rows keep the sums of the other confocal kernels: fp32 partials of kahan_block
// pairs, added to a compensated fp32 sum.  With the pairs in one part the volume is theirs bit for
// bit; more parts add up in double.
template <int KZ>
struct RealAcc {
    float sum[KZ], comp[KZ], blk[KZ];
    uint32_t n;
    __device__ __forceinline__ void flush() {
#pragma unroll
        for (int r = 0; r < KZ; ++r) {
            kahan_add(sum[r], comp[r], blk[r]);
            blk[r] = 0.0f;
        }
        n = 0u;
    }
    __device__ __forceinline__ void end_pair(uint32_t kahan_block) {
        if (++n == kahan_block) flush();
    }
    __device__ __forceinline__ void finish() {
        if (n) flush();
    }
    __device__ __forceinline__ double part(int r) const { return (double)sum[r] - (double)comp[r]; }
    __device__ __forceinline__ void store(const ConfocalArgs& a, size_t id, int r) const {
        static_cast<float*>(a.out)[id] = kahan_result(sum[r], comp[r]) * a.scale;
    }
};
struct RealRowsBase {
    using part_t = double;
    template <int KZ>
    using Acc = RealAcc<KZ>;
};
// fp32 rows, thresholds and samples apart (kF32Split): S is read first and the comparison picks the
// address of the one sample that is needed.  Two 4-byte reads at a stride of 4 bytes an update; an
// (S, sample) element takes an 8- and a 4-byte read at a stride of 8.  Measured at 9,216 pairs into
// 128 x 120 x 100: 5.06 ms against 5.74.
struct F32Rows : RealRowsBase {
    static constexpr int kFormat = kF32Split;
    template <int KZ, int DEG>
    __device__ static __forceinline__ void pair(Acc<KZ>& acc, const ColumnQuotient<KZ, DEG>& q, float axy,
                                                const float (&dz2)[KZ], uint32_t samples) {
        uint32_t o[KZ];
        float S[KZ], v[KZ];
#pragma unroll
        for (int i = 0; i < KZ; ++i) {
            o[i] = ElemOffset<8>::of(q.at(i)) >> 1;
            S[i] = lds_read4(o[i]);
        }
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t next = samples + 4u;
#pragma unroll
        for (int i = 0; i < KZ; ++i) {
            const float s = axy + dz2[column_order<KZ>(i)];
            v[i] = lds_read4(o[i] + (s >= S[i] ? next : samples));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < KZ; ++i) {
            const int r = column_order<KZ>(i);
            acc.blk[r] = acc.blk[r] + v[i];
        }
    }
};
// 16-bit rows: element (S, lo | hi << 16), the chain of CountRows::column with the sum in fp32 (fp16:
// the half is added by one mixed-precision FMA, h x 1 + sum; bf16: it lands in the high word, which
// is its fp32 value).
template <bool BF>
struct Half16Rows : RealRowsBase {
    static constexpr int kFormat = BF ? kBF16 : kF16;
    template <int KZ, int DEG>
    __device__ static __forceinline__ void pair(Acc<KZ>& acc, const ColumnQuotient<KZ, DEG>& q, float axy,
                                                const float (&dz2)[KZ], uint32_t) {
        uint2 e[KZ];
#pragma unroll
        for (int i = 0; i < KZ; ++i) e[i] = lds_read8(ElemOffset<8>::of(q.at(i)));
        __builtin_amdgcn_sched_barrier(0);
        float s = axy + dz2[column_order<KZ>(0)];
        uint32_t h;
        if constexpr (BF)
            asm("v_cmp_ge_f32_e32 vcc, %1, %2\n\ts_nop 1\n\t" SEL16_HIGH("%0", "%3")
                : "=v"(h) : "v"(s), "v"(e[0].x), "v"(e[0].y) : "vcc");
        else
            asm("v_cmp_ge_f32_e32 vcc, %1, %2\n\ts_nop 1\n\t" SEL16("%0", "%3")
                : "=v"(h) : "v"(s), "v"(e[0].x), "v"(e[0].y) : "vcc");
#pragma unroll
        for (int i = 1; i < KZ; ++i) {
            const int r = column_order<KZ>(i), prev = column_order<KZ>(i - 1);
            s = axy + dz2[r];
            uint32_t hn;
            if constexpr (BF)
                asm("v_cmp_ge_f32_e32 vcc, %2, %3\n\t"
                    "v_add_f32_e32 %0, %0, %5\n\t"
                    "s_nop 0\n\t" SEL16_HIGH("%1", "%4")
                    : "+&v"(acc.blk[prev]), "=v"(hn) : "v"(s), "v"(e[i].x), "v"(e[i].y), "v"(h) : "vcc");
            else
                asm("v_cmp_ge_f32_e32 vcc, %2, %3\n\t"
                    "v_fma_mix_f32 %0, %5, 1.0, %0 op_sel_hi:[1,0,0]\n\t"
                    "s_nop 0\n\t" SEL16("%1", "%4")
                    : "+&v"(acc.blk[prev]), "=v"(hn) : "v"(s), "v"(e[i].x), "v"(e[i].y), "v"(h) : "vcc");
            h = hn;
        }
        constexpr int last = column_order<KZ>(KZ - 1);
        if constexpr (BF) acc.blk[last] = acc.blk[last] + __uint_as_float(h);
        else acc.blk[last] = acc.blk[last] + (float)__builtin_bit_cast(_Float16, (unsigned short)h);
    }
};
// Complex rows, thresholds and samples apart (kC64Split): S is read first and the comparison picks
// the address of the one sample that is needed -- 12 LDS bytes an update at full bank spread,
// against 24 at a stride of 16 for elements that hold (re, im, S).
struct ComplexRows {
    static constexpr int kFormat = kC64Split;
    using part_t = ComplexSum;
    template <int KZ>
    struct Acc {
        RealAcc<KZ> re, im;
        __device__ __forceinline__ void end_pair(uint32_t kahan_block) {
            if (++re.n == kahan_block) {
                re.flush();
                im.flush();
            }
        }
        __device__ __forceinline__ void finish() {
            if (re.n) {
                re.flush();
                im.flush();
            }
        }
        __device__ __forceinline__ part_t part(int r) const { return {re.part(r), im.part(r)}; }
        __device__ __forceinline__ void store(const ConfocalArgs& a, size_t id, int r) const {
            static_cast<float2*>(a.out)[id] = make_float2(kahan_result(re.sum[r], re.comp[r]) * a.scale,
                                                          kahan_result(im.sum[r], im.comp[r]) * a.scale);
        }
    };
    // samples: LDS address of the sample of offset 0
    template <int KZ, int DEG>
    __device__ static __forceinline__ void pair(Acc<KZ>& acc, const ColumnQuotient<KZ, DEG>& q, float axy,
                                                const float (&dz2)[KZ], uint32_t samples) {
        uint32_t o[KZ];
        float S[KZ];
        uint2 v[KZ];
#pragma unroll
        for (int i = 0; i < KZ; ++i) {
            o[i] = ElemOffset<8>::of(q.at(i));
            S[i] = lds_read4(o[i] >> 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t next = samples + 8u;
#pragma unroll
        for (int i = 0; i < KZ; ++i) {
            const float s = axy + dz2[column_order<KZ>(i)];
            v[i] = lds_read8(o[i] + (s >= S[i] ? next : samples));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < KZ; ++i) {
            const int r = column_order<KZ>(i);
            acc.re.blk[r] = acc.re.blk[r] + __uint_as_float(v[i].x);
            acc.im.blk[r] = acc.im.blk[r] + __uint_as_float(v[i].y);
        }
    }
};

}  // namespace

// Pairs per part of a listed tile: the launch's work-groups spread over the listed tiles, at most
// 8 parts of at least 128 pairs.
__device__ __forceinline__ uint32_t list_part_pairs(uint32_t P, uint32_t count, uint32_t groups) {
    const uint32_t parts = max(1u, min(min(groups / max(count, 1u), 8u), P / 128u));
    return ((P + parts - 1u) / parts + 3u) / 4u * 4u;
}

// Work-group `block` of `blocks`: its tile's share of the pairs.  Returns the tile.
template <class Fz, int KZ, int DEG, bool TILES>
__device__ __forceinline__ uint32_t poly_tile(const LdsPolyArgs& a, uint32_t block, uint32_t blocks, char* smem) {
    constexpr uint32_t NW = 4, PS = NW;   // waves; pairs per stage (one per wave)
    using Off = ElemOffset<8>;
    using part_t = typename Fz::part_t;
    constexpr bool SPLIT = format_split(Fz::kFormat);
    constexpr uint32_t EB = Fz::kFormat == kF32Split ? 4u : 8u;   // bytes of an element (split: of its sample)
    // smem: [2][PS][seg] elements (split: thresholds first, then as many samples), then [2][PS] pair
    // records
    const uint32_t slot_bytes = a.seg * EB, lds0 = lds_offset(smem);
    const uint32_t s_bytes = SPLIT ? 2u * PS * a.seg * 4u : 0u;
    float4* const meta = reinterpret_cast<float4*>(smem + s_bytes + 2u * PS * slot_bytes);
    // ElemOffset's offset of the stage's first element; split: the threshold of offset o lies at o / 2,
    // its sample at EB o / 8 + samples
    const uint32_t origin = SPLIT ? 2u * lds0 : lds0, samples = lds0 + s_bytes - origin / 8u * EB;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const Grid& g = a.c.g;
    const uint32_t n0 = g.n[0], n1 = g.n[1], n2 = g.n[2], tiles = poly_tiles(g, KZ);
    // every tile of the grid, or those of a list whose length is on the device (then the launch is
    // fixed and its work-groups are shared out here)
    const uint32_t count = TILES ? __builtin_amdgcn_readfirstlane(*a.n_tiles) : tiles;
    const uint32_t part_pairs = TILES ? list_part_pairs(a.c.P, count, blocks) : a.part_pairs;
    const uint32_t part = count ? block / count : 0u, index = count ? block % count : 0u;
    if (TILES && (count == 0u || part * part_pairs >= a.c.P)) return 0u;
    const uint32_t tile = TILES ? __builtin_amdgcn_readfirstlane(a.tiles[index]) : xcd_remap(index, tiles);
    const uint32_t p0 = part * part_pairs, p1 = min(p0 + part_pairs, a.c.P);
    ColumnTile<KZ> t(g, tile, w, lane);
    if (TILES) t.idle = t.idle || __builtin_amdgcn_readfirstlane(a.fill[4u * tile + w]) < a.dense;
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
    const uint32_t row_bytes = a.c.ldh * (SPLIT ? 4u + EB : EB);
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
            // 2 elements of margin each way; the start even (split: a multiple of 4), so that a
            // 16-byte load never straddles a row end
            const int jl = ((int)__builtin_fmaf(__builtin_amdgcn_sqrtf(smin), a.c.inv2, pr.w) - 2) & (SPLIT ? ~3 : ~1);
            const int jh = (int)__builtin_fmaf(__builtin_amdgcn_sqrtf(smax), a.c.inv2, pr.w) + 2;
            mjl = jl;
            mcnt = min(jh + 2 - jl, (int)a.seg);
            mx = pr.x;
            my = pr.y;
            mw = pr.w + (float)(int)((((st & 1u) * PS + w) * a.seg) - (uint32_t)jl + (origin >> 3) + (uint32_t)Off::kBias);
        }
    };
    auto stage = [&](uint32_t b) {
        const uint32_t sl = b & 63u;
        if (sl == 0u) plan_windows(b);
        const uint32_t slot = (b & 1u) * PS + w;
        const int jl = __builtin_amdgcn_readlane(mjl, sl), cnt = __builtin_amdgcn_readlane(mcnt, sl);
        if (lane == sl) meta[slot] = make_float4(mx, my, mw, 0.0f);
        const char* row = static_cast<const char*>(a.c.H) + (size_t)(p0 + b * PS + w) * row_bytes;
        const uint32_t t_bytes = SPLIT ? a.c.ldh * 4u : 0u;
        if (SPLIT) {   // seg is a multiple of 256
            const __amdgpu_buffer_rsrc_t rt = make_rsrc(row, t_bytes);
            const uint32_t base = lds0 + slot * a.seg * 4u;
            for (int m = 0; m < cnt; m += 256) load_lds16(rt, base + (uint32_t)m * 4u, (jl + m) * 4 + (int)lane * 16);
        }
        const __amdgpu_buffer_rsrc_t rr = make_rsrc(row + t_bytes, row_bytes - t_bytes);
        constexpr int step = 1024 / (int)EB;
        const int vo = jl * (int)EB + (int)lane * 16;
        const uint32_t base = lds0 + s_bytes + slot * slot_bytes;
        for (int m = 0; m < cnt; m += step) load_lds16(rr, base + (uint32_t)m * EB, vo + m * (int)EB);
    };

    // (initialised as a whole: cleared in loops, the compiler keeps the sums as one vector and copies it
    // once a stage, 2 % of the time)
    typename Fz::template Acc<KZ> acc{};
    auto pair_step = [&](const float4 m) {
        const float dx = m.x - t.vx, dy = m.y - t.vy;
        const float axy = dx * dx + dy * dy;
        const ColumnQuotient<KZ, DEG> q(axy, u, u2, a.c.inv2, a.k1, a.k2, a.k3, m.z);
        Fz::template pair<KZ, DEG>(acc, q, axy, dz2, samples);
        acc.end_pair(a.c.kahan_block);
    };
    if (nstage) stage(0u);
    wait_loads();
    __syncthreads();
    for (uint32_t b = 0; b < nstage; ++b) {
        if (b + 1u < nstage) stage(b + 1u);
        const float4* mb = meta + (b & 1u) * PS;
        const uint32_t np = t.idle ? 0u : min(PS, p1 - p0 - b * PS);
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
    acc.finish();
    part_t* const sums = static_cast<part_t*>(a.parts);
    if (TILES) {   // [work-group = part x listed tiles + index][voxel of the column][lane]
        part_t* o = sums + (size_t)block * (256u * KZ) + threadIdx.x;
#pragma unroll
        for (int r = 0; r < KZ; ++r) o[256u * r] = acc.part(r);
    } else if (t.ix < n0 && t.iy < n1) {
        const size_t id = t.id(g);
        if (sums) {
            part_t* o = sums + (size_t)part * n0 * n1 * n2 + id;
#pragma unroll
            for (int r = 0; r < KZ; ++r) o[r] = acc.part(r);
        } else {
#pragma unroll
            for (int r = 0; r < KZ; ++r) acc.store(a.c, id + r, r);
        }
    }
    return tile;
}

// Count rows.
template <class Fz, int KZ, int DEG, bool TILES>
__global__ __launch_bounds__(256, 4) void confocal_lds_kernel_poly(LdsPolyArgs a) {
    extern __shared__ char smem[];
    if (!rows_wanted(a.c)) return;
    poly_tile<Fz, KZ, DEG, TILES>(a, blockIdx.x, gridDim.x, smem);
}
// The other rows.
template <class Fz, int KZ, int DEG>
__global__ __launch_bounds__(256, 4) void confocal_lds_kernel_column(LdsPolyArgs a) {
    extern __shared__ char smem[];
    if (!rows_wanted(a.c)) return;
    poly_tile<Fz, KZ, DEG, false>(a, blockIdx.x, gridDim.x, smem);
}

// Captures of many sizes: one work-group per item (capture, part x its tiles + tile).
template <class Fz, int KZ, int DEG>
__global__ __launch_bounds__(256, 4) void batch_lds_kernel_poly(BatchItems b, const LdsPolyArgs* __restrict__ caps) {
    extern __shared__ char smem[];
    const uint2 item = b.items[blockIdx.x];
    const uint32_t c = __builtin_amdgcn_readfirstlane(item.x), block = __builtin_amdgcn_readfirstlane(item.y);
    const LdsPolyArgs a = wave_uniform_load(caps + c);
    if (!rows_wanted(a.c)) return;
    poly_tile<Fz, KZ, DEG, false>(a, block, 0u, smem);
}

// The volume from the partial sums of its parts, in part order; a launch of its own, which costs less
// than having the last work-group of a tile add them up: the fences that this takes write back a
// whole L2 per work-group (1,961 pairs into 45 x 61 x 38: 0.20 ms against 0.08 with this kernel).
template <class T>
__device__ __forceinline__ T parts_at(const PartsSum& d, uint32_t parts, uint64_t i) {
    const T* const sums = static_cast<const T*>(d.sums) + i;
    T v = sums[0];
#pragma unroll 8
    for (uint32_t k = 1; k < parts; ++k) v += sums[(uint64_t)k * d.n];
    return v;
}
__device__ __forceinline__ void sum_parts(const PartsSum& d, uint32_t block, uint32_t blocks) {
    const bool counts = d.count_parts && __builtin_amdgcn_readfirstlane(*d.fmt_flag) == 0u;
    const uint32_t parts = counts ? d.count_parts : d.real_parts;
    if (parts <= 1u) return;   // written by the gather
    for (uint64_t i = (uint64_t)block * 256u + threadIdx.x; i < d.n; i += (uint64_t)blocks * 256u) {
        if (counts) static_cast<float*>(d.out)[i] = (float)parts_at<uint32_t>(d, parts, i);
        else if (!d.cplx) static_cast<float*>(d.out)[i] = (float)parts_at<double>(d, parts, i) * d.scale;
        else {
            const ComplexSum v = parts_at<ComplexSum>(d, parts, i);
            static_cast<float2*>(d.out)[i] = make_float2((float)v.re * d.scale, (float)v.im * d.scale);
        }
    }
}
__global__ __launch_bounds__(256) void sum_parts_kernel(PartsSum d) { sum_parts(d, blockIdx.x, gridDim.x); }
// Captures of many sizes, a row of work-groups each; the last of a row stamps its capture's completion.
__global__ __launch_bounds__(256) void batch_sum_parts_kernel(const PartsSum* __restrict__ d, uint32_t* remaining,
                                                              uint64_t* done) {
    const uint32_t c = blockIdx.y;
    const PartsSum s = wave_uniform_load(d + c);
    if (!s.out) return;
    sum_parts(s, blockIdx.x, gridDim.x);
    __syncthreads();
    if (threadIdx.x == 0 && atomicSub(&remaining[c], 1u) == 1u)
        atomicMax(reinterpret_cast<unsigned long long*>(&done[c]), (unsigned long long)wall_clock64());
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

// Marks the listed voxels: one bit per voxel (16 per column of a tile) and the number per quarter of a
// tile.  Lists follow the octree's blocks, so a wave's voxels share few quarters; the counters are
// updated once per (wave, quarter).
template <int KZ>
__global__ __launch_bounds__(256) void tile_mark_kernel(TileListArgs a, const uint32_t* __restrict__ voxels, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    TileVoxel t{0u, 0u, 0u};
    uint32_t q = 0xffffffffu;   // quarter
    if (i < n) {
        const uint32_t v = voxels[i];
        t = tile_voxel<KZ>(a.g, v & 1023u, (v >> 10) & 1023u, v >> 20);
        q = 4u * t.tile + (t.lane >> 6);
        const uint32_t col = t.tile * 256u + t.lane;
        atomicOr(&a.mask[col >> 1], 1u << (t.r + 16u * (col & 1u)));
    }
    bool left = i < n;
    while (__ballot(left) != 0ull) {
        const uint32_t first = (uint32_t)__builtin_ctzll(__ballot(left));
        const uint32_t quarter = __builtin_amdgcn_readlane(q, first);
        const bool mine = left && q == quarter;
        const uint64_t m = __ballot(mine);
        if ((threadIdx.x & 63u) == first) atomicAdd(&a.fill[quarter], (uint32_t)__builtin_popcountll(m));
        left = left && !mine;
    }
}
// Tiles with a quarter of at least `dense` listed voxels, in any order (each is computed by itself).
__global__ __launch_bounds__(256) void tile_pick_kernel(TileListArgs a, uint32_t tiles, uint32_t dense) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= tiles) return;
    const uint4 f = reinterpret_cast<const uint4*>(a.fill)[i];
    if (max(max(f.x, f.y), max(f.z, f.w)) >= dense) a.tiles[atomicAdd(&a.counts[0], 1u)] = i;
}
// The listed voxels of the other quarters, 64 neighbours of the list at a time.
template <int KZ>
__global__ __launch_bounds__(256) void tile_rest_kernel(TileListArgs a, const uint32_t* __restrict__ voxels, uint32_t n,
                                                        uint32_t dense) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63u;
    uint32_t v = 0;
    bool rest = false;
    if (i < n) {
        v = voxels[i];
        const TileVoxel t = tile_voxel<KZ>(a.g, v & 1023u, (v >> 10) & 1023u, v >> 20);
        rest = a.fill[4u * t.tile + (t.lane >> 6)] < dense;
    }
    const uint64_t m = __ballot(rest);
    uint32_t base = 0;
    if (lane == 0u && m) base = atomicAdd(&a.counts[1], (uint32_t)__builtin_popcountll(m));
    base = __builtin_amdgcn_readfirstlane(base);
    if (rest) a.rest[base + (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1ull))] = v;
}
// Volume values of the marked voxels of the listed tiles' well-filled quarters from their integer
// partial sums.
template <int KZ>
__global__ __launch_bounds__(256) void tile_store_kernel(TileListArgs a, LdsPolyArgs p, uint32_t groups) {
    const uint32_t count = a.counts[0];
    if (blockIdx.x >= count) return;
    const uint32_t part_pairs = list_part_pairs(p.c.P, count, groups), parts = (p.c.P + part_pairs - 1u) / part_pairs;
    const uint32_t tile = a.tiles[blockIdx.x], col = tile * 256u + threadIdx.x;
    const uint32_t bits = a.mask[col >> 1] >> (16u * (col & 1u)) & 0xffffu;
    if (!bits || a.fill[4u * tile + (threadIdx.x >> 6)] < p.dense) return;
    const uint32_t ntz = (a.g.n[2] + KZ - 1u) / KZ, nty = (a.g.n[1] + 15u) / 16u;
    const uint32_t tz = tile % ntz, ty = tile / ntz % nty, tx = tile / ntz / nty, w = threadIdx.x >> 6;
    const uint32_t ix = tx * 16u + (w & 1u) * 8u + (threadIdx.x & 7u), iy = ty * 16u + (w >> 1) * 8u + ((threadIdx.x >> 3) & 7u);
    float* out = static_cast<float*>(p.c.out) + ((size_t)ix * a.g.n[1] + iy) * a.g.n[2] + min(tz * KZ, a.g.n[2] - KZ);
    for (int r = 0; r < KZ; ++r)
        if (bits >> r & 1u) {
            uint32_t v = 0;
            for (uint32_t k = 0; k < parts; ++k)
                v += static_cast<const uint32_t*>(p.parts)[((size_t)k * count + blockIdx.x) * (256u * KZ) + 256u * r + threadIdx.x];
            out[r] = (float)v;
        }
}

// LDS of a work-group: two stages of 4 pairs and their records.
template <class Fz, class Kernel>
static hipError_t poly_lds(Kernel fn, uint32_t seg, size_t* bytes) {
    *bytes = 2u * 4u * ((size_t)seg * (Fz::kFormat == kC64Split ? 12u : 8u) + sizeof(float4));
    if (*bytes <= 64u * 1024u) return hipSuccess;
    return hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)*bytes);
}
template <class Fz, int KZ, int DEG, bool TILES>
static hipError_t poly_launch(const LdsPolyArgs& a, uint32_t groups, hipStream_t s) {
    const auto fn = [] {
        if constexpr (Fz::kFormat == kCount) return confocal_lds_kernel_poly<Fz, KZ, DEG, TILES>;
        else return confocal_lds_kernel_column<Fz, KZ, DEG>;
    }();
    size_t lds = 0;
    const hipError_t e = poly_lds<Fz>(fn, a.seg, &lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(fn, dim3(groups), dim3(256), lds, s, a);
    return hipGetLastError();
}
template <class Fz, bool TILES>
static hipError_t poly_launch_shape(const LdsPolyArgs& a, const LdsPolyShape& sh, uint32_t groups, hipStream_t s) {
    if constexpr (Fz::kFormat != kC64Split)   // two accumulators per voxel: 8 voxels per lane
        if (sh.kz == 16)
            return sh.deg == 2 ? poly_launch<Fz, 16, 2, TILES>(a, groups, s) : poly_launch<Fz, 16, 3, TILES>(a, groups, s);
    if (sh.kz != 8) return hipErrorInvalidValue;
    return sh.deg == 2 ? poly_launch<Fz, 8, 2, TILES>(a, groups, s) : poly_launch<Fz, 8, 3, TILES>(a, groups, s);
}
template <class Fz, int KZ, int DEG>
static hipError_t batch_poly_launch(const BatchItems& b, const LdsPolyArgs* caps, uint32_t seg, hipStream_t s) {
    const auto fn = batch_lds_kernel_poly<Fz, KZ, DEG>;
    size_t lds = 0;
    const hipError_t e = poly_lds<Fz>(fn, seg, &lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(fn, dim3(b.n), dim3(256), lds, s, b, caps);
    return hipGetLastError();
}
template <class Fz>
static hipError_t batch_poly_rows(const BatchItems& b, const LdsPolyArgs* caps, const LdsPolyShape& sh, hipStream_t s) {
    if constexpr (Fz::kFormat != kC64Split)
        if (sh.kz == 16)
            return sh.deg == 2 ? batch_poly_launch<Fz, 16, 2>(b, caps, sh.seg, s) : batch_poly_launch<Fz, 16, 3>(b, caps, sh.seg, s);
    if (sh.kz != 8) return hipErrorInvalidValue;
    return sh.deg == 2 ? batch_poly_launch<Fz, 8, 2>(b, caps, sh.seg, s) : batch_poly_launch<Fz, 8, 3>(b, caps, sh.seg, s);
}
hipError_t launch_batch_poly(const BatchItems& b, const LdsPolyArgs* caps, const LdsPolyShape& sh, int format,
                             hipStream_t s) {
    switch (format) {
        case kCount: return batch_poly_rows<CountRows>(b, caps, sh, s);
        case kF32Split: return batch_poly_rows<F32Rows>(b, caps, sh, s);
        case kF16: return batch_poly_rows<Half16Rows<false>>(b, caps, sh, s);
        case kBF16: return batch_poly_rows<Half16Rows<true>>(b, caps, sh, s);
        case kC64Split: return batch_poly_rows<ComplexRows>(b, caps, sh, s);
        default: return hipErrorInvalidValue;
    }
}
hipError_t launch_sum_parts(const PartsSum& d, hipStream_t s) {
    const uint32_t blocks = (uint32_t)std::max<uint64_t>(1u, std::min<uint64_t>((d.n + 255u) / 256u, 4096u));
    hipLaunchKernelGGL(sum_parts_kernel, dim3(blocks), dim3(256), 0, s, d);
    return hipGetLastError();
}
hipError_t launch_batch_sum_parts(const PartsSum* d, uint32_t n, uint32_t* remaining, uint64_t* done, hipStream_t s) {
    if (n > 65535u) return hipErrorInvalidValue;
    hipLaunchKernelGGL(batch_sum_parts_kernel, dim3(kBatchSumBlocks, n), dim3(256), 0, s, d, remaining, done);
    return hipGetLastError();
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
hipError_t launch_lds_poly(const LdsPolyArgs& a, const LdsPolyShape& sh, int format, uint32_t parts, hipStream_t s) {
    const uint32_t groups = (uint32_t)poly_tiles(a.c.g, sh.kz) * parts;
    switch (format) {
        case kCount: return poly_launch_shape<CountRows, false>(a, sh, groups, s);
        case kF32Split: return poly_launch_shape<F32Rows, false>(a, sh, groups, s);
        case kF16: return poly_launch_shape<Half16Rows<false>, false>(a, sh, groups, s);
        case kBF16: return poly_launch_shape<Half16Rows<true>, false>(a, sh, groups, s);
        case kC64Split: return poly_launch_shape<ComplexRows, false>(a, sh, groups, s);
        default: return hipErrorInvalidValue;
    }
}
uint32_t lds_poly_part_bytes(int format) { return format == kCount ? 4u : format == kC64Split ? 16u : 8u; }

// Parts of rows summed in compensated blocks hold whole blocks where those are short: the blocks, and
// so the error within them, are those of one part.
uint32_t part_unit(uint32_t kahan_block) {
    return kahan_block > 128u ? 4u : kahan_block % 4u == 0u ? kahan_block : kahan_block % 2u ? kahan_block * 4u : kahan_block * 2u;
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
                                   uint32_t dense, uint32_t groups, hipStream_t s) {
    a.fill = t.fill;
    a.dense = dense;
    a.tiles = t.tiles;
    a.n_tiles = t.counts;
    const hipError_t e = poly_launch_shape<CountRows, true>(a, sh, groups, s);
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
LdsPolyShape lds_poly_shape(const Grid& g, float inv2, float lz, double bound, double max_path, double budget, int format) {
    LdsPolyShape none;
    // column along z alone; coordinates whose squares and reciprocals stay normal floats
    if (g.inc[2] != 0.0f || g.inc[5] != 0.0f || g.inc[6] != 0.0f || g.inc[7] != 0.0f) return none;
    const double step = std::fabs((double)g.inc[8]), A = std::fabs((double)inv2);
    const double za = (double)lz - g.zero[2], zb = za - (double)g.inc[8] * (double)(g.n[2] - 1u);
    const double zmin = std::min(std::fabs(za), std::fabs(zb)) * (1.0 - 1e-5);
    if (!(za * zb > 0.0) || !(zmin > 1e-12) || !(max_path < 1e12) || !(step > 0.0)) return none;
    for (int kz : {16, 8}) {
        if (g.n[2] < (uint32_t)kz || (kz > 8 && format == kC64Split)) continue;
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
        // as confocal_lds_fits, with up to three more elements for the aligned start
        const double need = std::ceil(std::sqrt(d2) * A * (1.0 + 1e-6)) + 11.0;
        if (!(need <= (double)kPolySegMax)) continue;
        // Depth 16 spreads a pair's coefficients over more updates, depth 8 pads the last slab less:
        // per slice of z fp32 and bf16 rows take 5 to 6 % more time at depth 8, counts some 10 %
        // (4,096 pairs into 96^3, bf16: 0.79 ms at depth 16, 0.84 at 8; 9,216 pairs into
        // 128 x 120 x 100, fp32: 5.08 ms for 7 slabs of 16, 4.96 for 13 of 8).  The line at 10 %
        // padding is the counts'; for the rows that it serves (counts keep depth 16) the two sides
        // are level near 6 %, so up to 4 % are given away between 11 and 17 slabs of 8.
        const uint32_t pad16 = (g.n[2] + 15u) / 16u * 16u, pad8 = (g.n[2] + 7u) / 8u * 8u;
        if (kz == 16 && format != kCount && pad16 * 10u > pad8 * 11u) continue;
        LdsPolyShape sh;
        sh.kz = kz;
        sh.deg = deg;
        const uint32_t unit = format_split(format) ? 256u : 128u;
        sh.seg = ((uint32_t)need + unit - 1u) / unit * unit;
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
// Parts are of whole blocks of `unit` pairs.
uint32_t lds_poly_parts(const Grid& g, const LdsPolyShape& sh, uint32_t P, uint32_t sum_bytes, uint32_t unit,
                        uint32_t* part_pairs) {
    const uint64_t tiles = poly_tiles(g, sh.kz), vox = (uint64_t)g.n[0] * g.n[1] * g.n[2];
    uint64_t parts = std::max(std::min<uint64_t>((4096u + tiles - 1u) / tiles, P / 128u),
                              std::min<uint64_t>((1024u + tiles - 1u) / tiles, P / 32u));
    parts = std::max<uint64_t>(1u, std::min<uint64_t>(parts, (64ull << 20) / (sum_bytes * vox)));
    *part_pairs = (uint32_t)(((P + parts - 1u) / parts + unit - 1u) / unit * unit);
    return std::max(1u, (P + *part_pairs - 1u) / *part_pairs);
}

}  // namespace bpx
