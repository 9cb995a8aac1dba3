// generic.hip -- gfx950 kernels for the generic wire envelope's maintained
// F32 routes that the typed kernels do not already cover
// (crates/emel-kernels/src/any/generic.rs:1264-2055).
//
// Every route here is a sequential loop in the reference whose rounding
// depends on the order of its additions, so each kernel but k_gen_norm
// gives one lane the reference's whole loop for its unit of independent
// work, in the reference's order:
//   k_gen_rows      one lane per row: cumsum, soft_max_back and rms_norm_back
//                   of strided operands or narrow rows, and norm / rms_norm
//                   rows narrower than a wave (soft_max uses the typed strided
//                   path's exact sequential-sum kernel);
//   k_back_rows     soft_max_back and rms_norm_back of dense operands, wider
//                   rows: the sums as chains in order, the rest by whole
//                   workgroups;
//   k_gen_norm      a workgroup per row for norm and rms_norm rows of 64 or
//                   more columns that the typed row kernels cannot take
//                   (those run vectorisable rows with the generic arithmetic);
//                   both sum in f64 as a fixed-order tree: within rms_norm's
//                   1e-5 tolerance, the one route here not in the
//                   reference's order;
//   k_gen_ord       one lane per destination element: fill, arange, diag,
//                   diag_mask_inf/zero, concat, repeat_back (the source
//                   elements of one target summed in source-ordinal order);
//   k_l2_sum        one lane for the whole tensor (l2_norm's f32 sum), then
//                   k_l2_apply over every element;
//   k_count_*       an exact integer count (count_equal's f32 counter
//                   saturates at 2^24, which min() reproduces);
// Operands are addressed through their own extents and element strides, the
// reference's coordinates_for_index/byte_offset (generic.rs:896-933), walked
// incrementally along a row instead of re-decoded per element.
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "libm_replica.hpp"

namespace emel {
namespace {

constexpr int kRowBlock = 64; // one wave per workgroup spreads few rows over more CUs

// Ordinal -> element offset, advanced one ordinal at a time.
struct Walk {
    uint64_t c[4];
    int64_t off;

    __device__ __forceinline__ void init(const GView &v, uint64_t k)
    {
        off = 0;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            c[d] = k % v.ne[d];
            k /= v.ne[d];
            off += static_cast<int64_t>(c[d]) * v.st[d];
        }
    }

    __device__ __forceinline__ void next(const GView &v)
    {
        off += v.st[0];
        if (++c[0] < v.ne[0]) return;
        c[0] = 0;
        off += v.st[1] - static_cast<int64_t>(v.ne[0]) * v.st[0];
        if (++c[1] < v.ne[1]) return;
        c[1] = 0;
        off += v.st[2] - static_cast<int64_t>(v.ne[1]) * v.st[1];
        if (++c[2] < v.ne[2]) return;
        c[2] = 0;
        off += v.st[3] - static_cast<int64_t>(v.ne[2]) * v.st[2];
        ++c[3];
    }
};

__device__ __forceinline__ int64_t coords_offset(const GView &v, const uint64_t *c)
{
    int64_t off = 0;
#pragma unroll
    for (int d = 0; d < 4; ++d) off += static_cast<int64_t>(c[d]) * v.st[d];
    return off;
}

// ---- one lane per row -------------------------------------------------------------

template <GenRow OP>
__global__ __launch_bounds__(kRowBlock) void k_gen_rows(GenRowArgs a)
{
    const uint64_t r = static_cast<uint64_t>(blockIdx.x) * kRowBlock + threadIdx.x;
    if (r >= a.rows) return;
    const float *x = static_cast<const float *>(a.x.data);
    const float *g = static_cast<const float *>(a.g.data);
    float *y = static_cast<float *>(a.y.data);
    const uint64_t w = a.width;
    Walk x0, y0;
    x0.init(a.x, r * w);
    y0.init(a.y, r * w);

    if constexpr (OP == GenRow::Cumsum) { // generic.rs:1585-1609
        float sum = 0.0f;
        for (uint64_t c = 0; c < w; ++c) {
            sum += x[x0.off];
            y[y0.off] = sum;
            x0.next(a.x);
            y0.next(a.y);
        }
    } else if constexpr (OP == GenRow::Norm || OP == GenRow::RmsNorm) { // generic.rs:1988-2055
        Walk xi = x0;
        double sum = 0.0;
        for (uint64_t c = 0; c < w; ++c) {
            const float v = x[xi.off];
            sum += OP == GenRow::RmsNorm ? static_cast<double>(v * v) : static_cast<double>(v);
            xi.next(a.x);
        }
        const float mean = static_cast<float>(sum / static_cast<double>(w));
        double var = 0.0;
        if constexpr (OP == GenRow::Norm) {
            xi = x0;
            for (uint64_t c = 0; c < w; ++c) {
                const float centered = x[xi.off] - mean;
                var += static_cast<double>(centered * centered);
                xi.next(a.x);
            }
            var /= static_cast<double>(w);
        }
        const double base = OP == GenRow::RmsNorm ? static_cast<double>(mean) : var;
        const float scale = static_cast<float>(1.0 / __builtin_sqrt(base + static_cast<double>(a.eps)));
        xi = x0;
        Walk yi = y0;
        for (uint64_t c = 0; c < w; ++c) {
            const float v = x[xi.off];
            y[yi.off] = OP == GenRow::RmsNorm ? v * scale : (v - mean) * scale;
            xi.next(a.x);
            yi.next(a.y);
        }
    } else if constexpr (OP == GenRow::SoftMaxBack) { // generic.rs:1849-1881
        Walk g0;
        g0.init(a.g, r * w);
        Walk xi = x0, gi = g0;
        float dot = 0.0f;
        for (uint64_t c = 0; c < w; ++c) {
            dot = __builtin_fmaf(x[xi.off], g[gi.off], dot);
            xi.next(a.x);
            gi.next(a.g);
        }
        xi = x0;
        gi = g0;
        Walk yi = y0;
        for (uint64_t c = 0; c < w; ++c) {
            y[yi.off] = x[xi.off] * (g[gi.off] - dot);
            xi.next(a.x);
            gi.next(a.g);
            yi.next(a.y);
        }
    } else { // RmsNormBack, generic.rs:1883-1926
        Walk g0;
        g0.init(a.g, r * w);
        const double wd = static_cast<double>(w);
        Walk xi = x0;
        double sum = 0.0;
        for (uint64_t c = 0; c < w; ++c) {
            const float v = x[xi.off];
            sum += static_cast<double>(v * v);
            xi.next(a.x);
        }
        const double inv = 1.0 / __builtin_sqrt(sum / wd + static_cast<double>(a.eps));
        xi = x0;
        Walk gi = g0;
        double dot = 0.0;
        for (uint64_t c = 0; c < w; ++c) {
            dot += static_cast<double>(g[gi.off] * x[xi.off]);
            xi.next(a.x);
            gi.next(a.g);
        }
        xi = x0;
        gi = g0;
        Walk yi = y0;
        for (uint64_t c = 0; c < w; ++c) {
            const double xv = static_cast<double>(x[xi.off]);
            const double dy = static_cast<double>(g[gi.off]);
            y[yi.off] = static_cast<float>(dy * inv - xv * inv * inv * inv * dot / wd);
            xi.next(a.x);
            gi.next(a.g);
            yi.next(a.y);
        }
    }
}

// ---- soft_max_back and rms_norm_back over dense operands ---------------------------
// generic.rs:1849-1926: a row's sums are sequential (one f32 fma chain, or two
// f64 sums of f32 products), so their order cannot be split; what can be is
// everything around them.  A workgroup takes `group` whole rows, up to
// kBackTile elements (wider rows pass in tiles): all its threads load x and g
// once, 16 bytes a lane, keep them in registers for the result, and stage the
// chains' operands in LDS; then the chains run side by side:
//   soft_max_back  a lane per row, x and g from LDS, 7.5 cycles an element;
//   rms_norm_back  x*x and g*x rounded to f32 by all threads, then added by
//                  v_mfma_f64_4x4x4 against ones: four sequential f64
//                  additions of sixteen sums in 22 cycles (a lane that
//                  converted and added took 16 an element).  They are staged
//                  as doubles where the chain is what a launch waits for:
//                  widened by the chain, each step took 30 cycles.
// Bound by those chains for few wide rows (rms_norm_back, 512 rows of 4096:
// 24.0 us, 26.1 with floats staged; 2027 us with a lane per row walking global
// memory) and by memory for many (soft_max_back, 16384 rows of 512: 24 us,
// 4.2 TB/s; 192 us).
constexpr int kBackVec = 8;                             // float4 of x and of g per thread
constexpr uint32_t kBackTile = kBackVec * 4 * kBlock;   // elements per workgroup and pass
constexpr uint32_t kBackRows = 64;                      // rows per workgroup at most (32 for rms_norm_back)

struct BackArgs {
    const float *x, *g;
    float *y; // may be x or g
    uint64_t rows, width;
    uint32_t group; // rows per workgroup; 1 when width > kBackTile
    uint32_t ld;    // elements per staged row
    FastDiv by_width; // of the tile's element index (group > 1)
    float eps;
};

// VEC: 16-byte accesses; FOURS: a thread's four elements share a row; WIDE
// (RMS): the chains' operands are staged as doubles.
template <bool RMS, bool VEC, bool FOURS, bool WIDE>
__global__ __launch_bounds__(kBlock, 2) void k_back_rows(BackArgs a)
{
    extern __shared__ __attribute__((aligned(16))) float s_rows[];
    __shared__ double s_sum[kBackRows];
    __shared__ double s_inv[kBackRows];
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint64_t r0 = static_cast<uint64_t>(blockIdx.x) * a.group;
    const uint32_t rows = static_cast<uint32_t>(a.rows - r0 < a.group ? a.rows - r0 : a.group);
    const uint64_t first = r0 * a.width;
    const double wd = static_cast<double>(a.width);
    const uint64_t tiles = a.group > 1 ? 1 : (a.width + kBackTile - 1) / kBackTile;
    using Staged = typename std::conditional<WIDE, double, float>::type;
    using Staged4 = Staged __attribute__((ext_vector_type(4), aligned(16)));
    Staged *const s_p = reinterpret_cast<Staged *>(s_rows);
    Staged *const s_q = s_p + a.group * a.ld;

    float4 xv[kBackVec], gv[kBackVec];
    auto index = [&](int j) { return VEC ? (j * kBlock + tid) * 4 : j * kBlock * 4 + tid; };
    // element e of slot j: VEC takes four in a row, else every 256th
    auto elem = [&](int j, int e) { return VEC ? index(j) + e : index(j) + e * kBlock; };
    // Elements past the tile's n read zeros, and stores there are dropped.
    auto load = [&](uint64_t at, uint32_t n) {
        const BufRsrc xr = buffer_rsrc(a.x + at, n * 4), gr = buffer_rsrc(a.g + at, n * 4);
#pragma unroll
        for (int j = 0; j < kBackVec; ++j) {
            if constexpr (VEC) {
                xv[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(xr, index(j) * 4, 0, 0));
                gv[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(gr, index(j) * 4, 0, 0));
            } else {
                float xe[4], ge[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    xe[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, elem(j, e) * 4, 0, 0));
                    ge[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(gr, elem(j, e) * 4, 0, 0));
                }
                xv[j] = make_float4(xe[0], xe[1], xe[2], xe[3]);
                gv[j] = make_float4(ge[0], ge[1], ge[2], ge[3]);
            }
        }
    };
    auto place = [&](uint32_t i) { // the element's place in a staged array
        const uint32_t r = a.group > 1 ? a.by_width.div(i) : 0;
        return a.group > 1 ? r * a.ld + (i - r * static_cast<uint32_t>(a.width)) : i;
    };
    auto stage = [&](uint32_t n) {
#pragma unroll
        for (int j = 0; j < kBackVec; ++j) {
            float4 p = xv[j], q = gv[j];
            if constexpr (RMS) {
                q = make_float4(gv[j].x * xv[j].x, gv[j].y * xv[j].y, gv[j].z * xv[j].z, gv[j].w * xv[j].w);
                p = make_float4(xv[j].x * xv[j].x, xv[j].y * xv[j].y, xv[j].z * xv[j].z, xv[j].w * xv[j].w);
            }
            if constexpr (FOURS) {
                if (index(j) < n) {
                    const uint32_t o = place(index(j));
                    *reinterpret_cast<Staged4 *>(s_p + o) = Staged4{p.x, p.y, p.z, p.w};
                    *reinterpret_cast<Staged4 *>(s_q + o) = Staged4{q.x, q.y, q.z, q.w};
                }
            } else {
                const float pe[4] = {p.x, p.y, p.z, p.w}, qe[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t i = elem(j, e);
                    if (i < n) {
                        const uint32_t o = place(i);
                        s_p[o] = pe[e];
                        s_q[o] = qe[e];
                    }
                }
            }
        }
    };

    float dot = 0.0f;  // soft_max_back: lane r of wave 0 holds row r's
    double sums = 0.0; // rms_norm_back: the matrix result, below
    const uint32_t g4 = lane / 16;
    for (uint64_t t = 0; t < tiles; ++t) {
        const uint64_t left = static_cast<uint64_t>(rows) * a.width - t * kBackTile;
        const uint32_t n = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(left < kBackTile ? left : kBackTile));
        const uint32_t cols = a.group > 1 ? static_cast<uint32_t>(a.width) : n; // of a row in this tile
        load(first + t * kBackTile, n);
        stage(n);
        if constexpr (RMS) { // whole steps of four: -0 leaves a sum as it is
            const uint32_t pad = (4 - cols % 4) % 4;
            for (uint32_t i = tid; i < 2 * rows * pad; i += kBlock) {
                const uint32_t c = i / pad;
                s_p[(c < rows ? c : a.group + c - rows) * a.ld + cols + i % pad] = -0.0f;
            }
        }
        __syncthreads();
        if constexpr (RMS) {
            // Chain c < rows adds row c's squares, c >= rows row c - rows's
            // products; a wave runs sixteen.
            if (16 * wave < 2 * rows) {
                const uint32_t c = min(16 * wave + lane % 16, 2 * rows - 1);
                const Staged *s = s_p + (c < rows ? c : a.group + c - rows) * a.ld + g4;
                const uint32_t steps = (cols + 3) / 4;
                auto add = [&](Staged v) { sums = __builtin_amdgcn_mfma_f64_4x4x4f64(static_cast<double>(v), 1.0, sums, 0, 0, 0); };
                uint32_t k = 0;
                if (steps >= 8) { // the next eight are read while eight are added
                    Staged v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = s[4 * u];
#pragma unroll 2
                    for (k = 8; k + 8 <= steps; k += 8) {
                        Staged w[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) w[u] = s[4 * (k + u)];
#pragma unroll
                        for (int u = 0; u < 8; ++u) add(v[u]);
#pragma unroll
                        for (int u = 0; u < 8; ++u) v[u] = w[u];
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) add(v[u]);
                }
                for (; k < steps; ++k) add(s[4 * k]);
            }
        } else if (wave == 0 && lane < rows) {
            const float *p = s_rows + lane * a.ld, *q = s_rows + (a.group + lane) * a.ld;
            auto add = [&](float4 u, float4 v) {
                dot = __builtin_fmaf(u.x, v.x, dot);
                dot = __builtin_fmaf(u.y, v.y, dot);
                dot = __builtin_fmaf(u.z, v.z, dot);
                dot = __builtin_fmaf(u.w, v.w, dot);
            };
            auto p4 = [&](uint32_t i) { return *reinterpret_cast<const float4 *>(p + i); };
            auto q4 = [&](uint32_t i) { return *reinterpret_cast<const float4 *>(q + i); };
            uint32_t c = 0;
            if (cols >= 16) { // the next sixteen are read while sixteen are added
                float4 u[4], v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    u[i] = p4(4 * i);
                    v[i] = q4(4 * i);
                }
#pragma unroll 2
                for (c = 16; c + 16 <= cols; c += 16) {
                    float4 un[4], vn[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        un[i] = p4(c + 4 * i);
                        vn[i] = q4(c + 4 * i);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) add(u[i], v[i]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        u[i] = un[i];
                        v[i] = vn[i];
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) add(u[i], v[i]);
            }
            for (; c + 4 <= cols; c += 4) add(p4(c), q4(c));
            for (; c < cols; ++c) dot = __builtin_fmaf(p[c], q[c], dot);
        }
        if (t + 1 < tiles) __syncthreads(); // the next tile overwrites the staged one
    }
    if constexpr (RMS) {
        // result of chain 16 wave + 4 (lane / 4 % 4) + lane / 16 in each of four lanes
        const uint32_t c = 16 * wave + 4 * (lane / 4 % 4) + g4;
        if (lane % 4 == 0 && c < 2 * rows) s_sum[c] = sums;
        __syncthreads();
        if (tid < rows) s_inv[tid] = 1.0 / __builtin_sqrt(s_sum[tid] / wd + static_cast<double>(a.eps));
    } else if (wave == 0 && lane < rows) {
        s_sum[lane] = static_cast<double>(dot);
    }
    __syncthreads();

    for (uint64_t t = 0; t < tiles; ++t) {
        const uint64_t left = static_cast<uint64_t>(rows) * a.width - t * kBackTile;
        const uint32_t n = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(left < kBackTile ? left : kBackTile));
        const uint64_t at = first + t * kBackTile;
        const BufRsrc yr = buffer_rsrc(a.y + at, n * 4);
        if (tiles > 1) load(at, n);
#pragma unroll
        for (int j = 0; j < kBackVec; ++j) {
            const float xe[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w}, ge[4] = {gv[j].x, gv[j].y, gv[j].z, gv[j].w};
            float o[4];
            uint32_t r = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (a.group > 1 && (e == 0 || !FOURS)) r = min(a.by_width.div(elem(j, e)), rows - 1);
                if constexpr (RMS) {
                    const double xd = static_cast<double>(xe[e]), dy = static_cast<double>(ge[e]), inv = s_inv[r];
                    o[e] = static_cast<float>(dy * inv - xd * inv * inv * inv * s_sum[rows + r] / wd);
                } else {
                    o[e] = xe[e] * (ge[e] - static_cast<float>(s_sum[r]));
                }
            }
            if constexpr (VEC) {
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, make_float4(o[0], o[1], o[2], o[3])), yr,
                                                       index(j) * 4, 0, 0);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, o[e]), yr, elem(j, e) * 4, 0, 0);
            }
        }
    }
}

// ---- one lane per destination element ------------------------------------------

template <GenOrd OP>
__global__ __launch_bounds__(kBlock) void k_gen_ord(GenOrdArgs a, uint64_t count)
{
    const float *x = static_cast<const float *>(a.a.data);
    const float *xb = static_cast<const float *>(a.b.data);
    float *y = static_cast<float *>(a.y.data);
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t k = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; k < count; k += stride) {
        uint64_t c[4];
        uint64_t rem = k;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            c[d] = rem % a.y.ne[d];
            rem /= a.y.ne[d];
        }
        const int64_t oo = coords_offset(a.y, c);
        float v;
        if constexpr (OP == GenOrd::Fill) { // generic.rs:1736-1750
            v = a.p0;
        } else if constexpr (OP == GenOrd::Arange) { // generic.rs:1752-1770
            v = __builtin_fmaf(static_cast<float>(k), a.p1, a.p0);
        } else if constexpr (OP == GenOrd::Diag) { // generic.rs:1772-1793: dst (column, row)
            v = c[0] == c[1] ? x[static_cast<int64_t>(c[1]) * a.a.st[0]] : 0.0f;
        } else if constexpr (OP == GenOrd::DiagMaskInf || OP == GenOrd::DiagMaskZero) { // :1795-1820
            if (c[0] > c[1] + a.n_past)
                v = OP == GenOrd::DiagMaskInf ? -__builtin_inff() : 0.0f;
            else
                v = x[coords_offset(a.a, c)];
        } else if constexpr (OP == GenOrd::Concat) { // generic.rs:1703-1734
            const uint32_t ax = a.axis;
            if (c[ax] < a.a.ne[ax]) {
                v = x[coords_offset(a.a, c)];
            } else {
                c[ax] -= a.a.ne[ax];
                v = xb[coords_offset(a.b, c)];
            }
        } else { // RepeatBack, generic.rs:1667-1701
            // The source elements that map onto target t are t + m * T for
            // every multiple m; increasing source ordinal is lexicographic
            // (m3, m2, m1, m0).
            uint64_t q[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) q[d] = a.a.ne[d] / a.y.ne[d];
            float acc = 0.0f;
            for (uint64_t m3 = 0; m3 < q[3]; ++m3)
                for (uint64_t m2 = 0; m2 < q[2]; ++m2)
                    for (uint64_t m1 = 0; m1 < q[1]; ++m1) {
                        const int64_t base = static_cast<int64_t>(c[1] + m1 * a.y.ne[1]) * a.a.st[1] +
                                             static_cast<int64_t>(c[2] + m2 * a.y.ne[2]) * a.a.st[2] +
                                             static_cast<int64_t>(c[3] + m3 * a.y.ne[3]) * a.a.st[3];
                        for (uint64_t m0 = 0; m0 < q[0]; ++m0)
                            acc = acc + x[base + static_cast<int64_t>(c[0] + m0 * a.y.ne[0]) * a.a.st[0]];
                    }
            v = acc;
        }
        y[oo] = v;
    }
}

// ---- l2_norm: one sequential f32 sum, then a scale pass (generic.rs:1822-1847) ----

__global__ __launch_bounds__(64) void k_l2_sum(GView xv, uint64_t count, float *scale_out)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const float *x = static_cast<const float *>(xv.data);
    float sum = 0.0f;
    Walk w;
    w.init(xv, 0);
    for (uint64_t k = 0; k < count; ++k) {
        const float v = x[w.off];
        sum += v * v;
        w.next(xv);
    }
    scale_out[0] = 1.0f / __builtin_sqrtf(sum);
    scale_out[1] = sum;
}

__global__ __launch_bounds__(kBlock) void k_l2_apply(GView xv, GView yv, uint64_t count, const float *scale)
{
    const float *x = static_cast<const float *>(xv.data);
    float *y = static_cast<float *>(yv.data);
    const float s = scale[0];
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t k = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; k < count; k += stride) {
        Walk wx, wy;
        wx.init(xv, k);
        wy.init(yv, k);
        y[wy.off] = x[wx.off] * s;
    }
}

// ---- count_equal (generic.rs:1928-1946) -------------------------------------------

constexpr uint32_t kCountBlocks = 1024;

__global__ __launch_bounds__(kBlock) void k_count_partial(GView av, GView bv, uint64_t count,
                                                          unsigned long long *partial)
{
    __shared__ unsigned long long part[kBlock / kWave];
    const uint32_t *pa = static_cast<const uint32_t *>(av.data);
    const uint32_t *pb = static_cast<const uint32_t *>(bv.data);
    unsigned long long n = 0;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t k = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; k < count; k += stride) {
        Walk wa, wb;
        wa.init(av, k);
        wb.init(bv, k);
        n += pa[wa.off] == pb[wb.off] ? 1ull : 0ull;
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) n += __shfl_xor(n, off, kWave);
    if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int i = 0; i < kBlock / kWave; ++i) t += part[i];
        partial[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(kBlock) void k_count_final(const unsigned long long *partial, uint32_t n, float *dst)
{
    __shared__ unsigned long long part[kBlock / kWave];
    unsigned long long t = 0;
    for (uint32_t i = threadIdx.x; i < n; i += kBlock) t += partial[i];
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) t += __shfl_xor(t, off, kWave);
    if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long total = 0;
        for (int i = 0; i < kBlock / kWave; ++i) total += part[i];
        // The reference counts in f32: 2^24 + 1 rounds back to 2^24.
        dst[0] = static_cast<float>(total < (1ull << 24) ? total : (1ull << 24));
    }
}

uint32_t grid_for(uint64_t count, uint32_t block, uint64_t cap)
{
    uint64_t blocks = (count + block - 1) / block;
    if (blocks > cap) blocks = cap;
    if (blocks == 0) blocks = 1;
    return static_cast<uint32_t>(blocks);
}

} // namespace

// ---- norm and rms_norm: a workgroup per row ------------------------------------------
// generic.rs:1988-2055: per row of width = src0.ne[0] ordinals, s = sum of
// f64(v*v) (rms) or f64(v) (norm), mean = f32(s / width); norm adds the f64
// sum of f32(centered^2) divided by width; scale = f32(1 / sqrt(base + eps))
// in f64; y = v * scale or (v - mean) * scale in f32.  The f64 sums run as a
// fixed-order tree over the row's threads (parity within the 1e-5 relative
// tolerance of rms_norm, not bit for bit against the reference's sequential
// order); every f32 step is the reference's.  A generic row is one dim-0
// row of src0, so its elements sit at a row base plus column * st[0]; dst
// rows are addressed the same way when dst.ne[0] == width, else each
// element's ordinal is decoded through dst's own extents.
template <int BS>
__device__ __forceinline__ double block_sum_f64(double v, double *lds)
{
    v = wave_sum_dpp(v);
    if constexpr (BS == kWave) {
        return v;
    } else {
        const uint32_t w = threadIdx.x / kWave;
        __syncthreads(); // lds is reused by the next reduction
        if (threadIdx.x % kWave == 0) lds[w] = v;
        __syncthreads();
        double t = lds[0];
#pragma unroll
        for (int i = 1; i < BS / kWave; ++i) t += lds[i];
        return t;
    }
}

template <bool RMS, int BS>
__global__ __launch_bounds__(BS) void k_gen_norm(GenRowArgs a, bool dst_rows)
{
    __shared__ double lds[BS / kWave];
    const uint64_t r = blockIdx.x;
    const uint64_t w = a.width;
    const float *x = static_cast<const float *>(a.x.data);
    float *y = static_cast<float *>(a.y.data);
    Walk xr, yr;
    xr.init(a.x, r * w); // column 0 of the row
    const int64_t sx = a.x.st[0];
    if (dst_rows) yr.init(a.y, r * w);
    double sum = 0.0;
    for (uint64_t c = threadIdx.x; c < w; c += BS) {
        const float v = x[xr.off + static_cast<int64_t>(c) * sx];
        sum += RMS ? static_cast<double>(v * v) : static_cast<double>(v);
    }
    sum = block_sum_f64<BS>(sum, lds);
    const float mean = static_cast<float>(sum / static_cast<double>(w));
    double base = static_cast<double>(mean);
    if constexpr (!RMS) {
        double var = 0.0;
        for (uint64_t c = threadIdx.x; c < w; c += BS) {
            const float centered = x[xr.off + static_cast<int64_t>(c) * sx] - mean;
            var += static_cast<double>(centered * centered);
        }
        var = block_sum_f64<BS>(var, lds);
        base = var / static_cast<double>(w);
    }
    const float scale = static_cast<float>(1.0 / __builtin_sqrt(base + static_cast<double>(a.eps)));
    for (uint64_t c = threadIdx.x; c < w; c += BS) {
        const float v = x[xr.off + static_cast<int64_t>(c) * sx];
        const float o = RMS ? v * scale : (v - mean) * scale;
        int64_t yo;
        if (dst_rows) {
            yo = yr.off + static_cast<int64_t>(c) * a.y.st[0];
        } else {
            Walk e;
            e.init(a.y, r * w + c);
            yo = e.off;
        }
        y[yo] = o;
    }
}

Operand as_operand(const GView &v)
{
    return Operand{v.data, {v.ne[0], v.ne[1], v.ne[2], v.ne[3]}, {v.st[0], v.st[1], v.st[2], v.st[3]}};
}

// Vectorisable rows (dim 0 contiguous, 16-byte aligned, same shapes) run on
// the typed row kernels with the generic arithmetic (RowOp::GenRmsNorm /
// GenNorm: rows in registers, 128-bit accesses); other layouts on
// k_gen_norm.
template <bool RMS>
hipError_t launch_gen_norm(const GenRowArgs &a, hipStream_t s)
{
    RowArgs ra{};
    ra.op = RMS ? RowOp::GenRmsNorm : RowOp::GenNorm;
    ra.x = as_operand(a.x);
    ra.y = as_operand(a.y);
    ra.eps = a.eps;
    const hipError_t e = launch_rows(ra, s);
    if (e != hipErrorNotSupported) return e;
    if (a.rows > 0x7fffffffull) return hipErrorInvalidConfiguration;
    const bool dst_rows = a.y.ne[0] == a.width;
    const dim3 grid(static_cast<uint32_t>(a.rows));
    if (a.width <= 1024) k_gen_norm<RMS, kWave><<<grid, kWave, 0, s>>>(a, dst_rows);
    else k_gen_norm<RMS, kBlock><<<grid, kBlock, 0, s>>>(a, dst_rows);
    return hipGetLastError();
}

// Whether ordinal k of the view is element k of its memory.
bool dense(const GView &v)
{
    int64_t expect = 1;
    for (int d = 0; d < 4; ++d) {
        if (v.ne[d] > 1 && v.st[d] != expect) return false;
        expect *= static_cast<int64_t>(v.ne[d]);
    }
    return true;
}

// Rows per workgroup: as many as a tile holds, but at least 512 workgroups
// where there are as many rows, so that both of a CU's run; of odd widths a
// multiple of four, for 16-byte accesses (more rather than fewer, which would
// leave a few workgroups to a second round: 30001 rows of 17, soft_max_back
// 10.2 us by 56, 7.2 by 60).
template <bool RMS>
uint64_t back_group(const GenRowArgs &a)
{
    uint64_t most = a.width >= kBackTile ? 1 : kBackTile / a.width;
    if (most > kBackRows / (RMS ? 2 : 1)) most = kBackRows / (RMS ? 2 : 1);
    uint64_t group = (a.rows + 511) / 512;
    if (group > most) group = most;
    if (group >= 4 && a.width % 4 != 0) {
        group = (group + 3) / 4 * 4;
        if (group > most) group -= 4;
    }
    return group;
}

template <bool RMS>
bool back_vec(const GenRowArgs &a, uint64_t group) // every workgroup's first element is 16-byte aligned
{
    return group * a.width % 4 == 0 && (a.rows * a.width) % 4 == 0 &&
           ((reinterpret_cast<uintptr_t>(a.x.data) | reinterpret_cast<uintptr_t>(a.g.data) | reinterpret_cast<uintptr_t>(a.y.data)) & 15u) == 0;
}

// Dense operands of rows wide enough for a lane's 16-byte accesses and a
// chain's reads to pay for the staging; narrower rows are read well enough by
// a lane each.  us with lanes / workgroups:
//   soft_max_back  1000000 rows of 1 14 / 133, 60000 of 4 4.9 / 5.7, 10000 of
//                  4 4.1 / 3.9, 30000 of 8 6.4 / 4.1; odd widths and starts off
//                  16 bytes, where a lane's four elements span rows or are
//                  loaded one by one: 10000 of 9 5.3 / 6.6, 300 of 13 6.2 / 5.9,
//                  100000 of 13 15.7 / 19.5, 300001 of 13 72 / 48, 20000 of 15
//                  7.6 / 7.2;
//   rms_norm_back  1000000 of 1 16 / 401, 10000 of 4 4.9 / 6.7, 10000 of 8
//                  6.9 / 6.8, 100000 of 8 12 / 27, 100000 of 16 27.0 / 27.5; odd
//                  ones 10000 of 15 9.0 / 9.6, 10000 of 17 9.8 / 9.3, 60000 of 17
//                  15.6 / 30, 60000 of 23 26 / 30, 300001 of 17 169 / 132.
// And as long as the workgroups fit a launch's 2^32 work-items (rows of 16
// with 32 to a workgroup: 2^29 rows, 34 GB an operand; a lane per row takes
// 2^32).
template <bool RMS>
bool back_by_groups(const GenRowArgs &a)
{
    const uint64_t group = back_group<RMS>(a);
    if (!dense(a.x) || !dense(a.g) || !dense(a.y) || (a.rows + group - 1) / group > 0xffffffffull / kBlock) return false;
    if (a.width >= 24) return true;
    const bool fours = a.width % 4 == 0 && back_vec<RMS>(a, group);
    if (RMS) {
        if (fours) return a.width >= 16 || (a.width >= 8 && a.rows < 16384);
        if (a.width >= 16) return a.rows < 16384 || a.rows >= 131072;
        return a.width >= 8 && a.rows < 256;
    }
    if (fours) return a.width > 4 || a.rows < 32768;
    return a.width >= 14 || (a.width >= 8 && (a.rows < 512 || (a.width >= 11 && a.rows * a.width >= (1 << 21))));
}

template <bool RMS>
hipError_t launch_back(const GenRowArgs &a, hipStream_t s)
{
    BackArgs b{};
    b.x = static_cast<const float *>(a.x.data);
    b.g = static_cast<const float *>(a.g.data);
    b.y = static_cast<float *>(a.y.data);
    b.rows = a.rows;
    b.width = a.width;
    b.eps = a.eps;
    const uint64_t group = back_group<RMS>(a);
    b.group = static_cast<uint32_t>(group);
    const uint32_t cols = static_cast<uint32_t>(a.width < kBackTile ? a.width : kBackTile);
    b.ld = (cols + 63) / 64 * 64 + 4;
    b.by_width = FastDiv(cols);
    const uint64_t blocks = (a.rows + group - 1) / group;
    const bool vec = back_vec<RMS>(a, group);
    const uint32_t lds = 2 * b.group * b.ld * sizeof(float);
    auto go = [&](auto wide) {
        constexpr bool WIDE = decltype(wide)::value;
        const uint32_t bytes = WIDE ? 2 * lds : lds;
        const dim3 grid(static_cast<uint32_t>(blocks));
        if (vec && a.width % 4 == 0) k_back_rows<RMS, true, true, WIDE><<<grid, kBlock, bytes, s>>>(b);
        else if (vec) k_back_rows<RMS, true, false, WIDE><<<grid, kBlock, bytes, s>>>(b);
        else k_back_rows<RMS, false, false, WIDE><<<grid, kBlock, bytes, s>>>(b);
        return hipGetLastError();
    };
    // Staged as doubles where wide rows' chains have no other workgroup's
    // memory traffic beside them: one round of two workgroups per CU, each
    // with half of its 160 KB of LDS (or of one, with nearly all).  us with
    // floats / doubles: 512 rows of 4096 26.1 / 24.0, 300 of 2304 16.3 / 15.1,
    // 1500 of 1056 12.7 / 12.2, 16 of 512 6.35 / 6.15.  More workgroups lose
    // the others that floats leave room for, 700 of 4224 29.5 / 42.3, 2000 of
    // 4224 65.4 / 88.1, and short chains gain less than the staging costs,
    // 20000 of 128 12.1 / 14.7, 70000 of 64 23.6 / 25.9.
    if constexpr (RMS) {
        const uint32_t room = (blocks > 256 ? 78u : 156u) * 1024;
        if (a.width >= 512 && blocks <= 512 && 2 * lds <= room) return go(std::true_type{});
    }
    return go(std::false_type{});
}

// Rows narrower than a wave keep one lane per row (and the reference's
// sequential order).
constexpr uint64_t kNormRowMin = kWave;

hipError_t launch_generic_rows(const GenRowArgs &a, hipStream_t s)
{
    if (a.rows == 0) return hipSuccess;
    const uint64_t blocks = (a.rows + kRowBlock - 1) / kRowBlock;
    if (blocks > 0x7fffffffull) return hipErrorInvalidConfiguration;
    const dim3 grid(static_cast<uint32_t>(blocks));
    switch (a.op) {
    case GenRow::Cumsum: k_gen_rows<GenRow::Cumsum><<<grid, kRowBlock, 0, s>>>(a); break;
    case GenRow::SoftMax: { // generic.rs:1948-1986: the exact sequential-sum kernel of the typed strided path
        return launch_softmax_seq(as_operand(a.x), as_operand(a.y), s);
    }
    case GenRow::Norm:
        if (a.width >= kNormRowMin) return launch_gen_norm<false>(a, s);
        k_gen_rows<GenRow::Norm><<<grid, kRowBlock, 0, s>>>(a);
        break;
    case GenRow::RmsNorm:
        if (a.width >= kNormRowMin) return launch_gen_norm<true>(a, s);
        k_gen_rows<GenRow::RmsNorm><<<grid, kRowBlock, 0, s>>>(a);
        break;
    case GenRow::SoftMaxBack:
        if (back_by_groups<false>(a)) return launch_back<false>(a, s);
        k_gen_rows<GenRow::SoftMaxBack><<<grid, kRowBlock, 0, s>>>(a);
        break;
    case GenRow::RmsNormBack:
        if (back_by_groups<true>(a)) return launch_back<true>(a, s);
        k_gen_rows<GenRow::RmsNormBack><<<grid, kRowBlock, 0, s>>>(a);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_generic_ordinal(const GenOrdArgs &a, hipStream_t s)
{
    uint64_t count = 1;
    for (int d = 0; d < 4; ++d) count *= a.y.ne[d];
    const dim3 grid(grid_for(count, kBlock, 65536));
    switch (a.op) {
    case GenOrd::Fill: k_gen_ord<GenOrd::Fill><<<grid, kBlock, 0, s>>>(a, count); break;
    case GenOrd::Arange: k_gen_ord<GenOrd::Arange><<<grid, kBlock, 0, s>>>(a, count); break;
    case GenOrd::Diag: k_gen_ord<GenOrd::Diag><<<grid, kBlock, 0, s>>>(a, count); break;
    case GenOrd::DiagMaskInf: k_gen_ord<GenOrd::DiagMaskInf><<<grid, kBlock, 0, s>>>(a, count); break;
    case GenOrd::DiagMaskZero: k_gen_ord<GenOrd::DiagMaskZero><<<grid, kBlock, 0, s>>>(a, count); break;
    case GenOrd::Concat: k_gen_ord<GenOrd::Concat><<<grid, kBlock, 0, s>>>(a, count); break;
    case GenOrd::RepeatBack: k_gen_ord<GenOrd::RepeatBack><<<grid, kBlock, 0, s>>>(a, count); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

uint64_t generic_workspace_bytes(GenWork w)
{
    switch (w) {
    case GenWork::L2Norm: return 256;
    case GenWork::CountEqual: return kCountBlocks * sizeof(unsigned long long);
    }
    return 0;
}

hipError_t launch_generic_l2_norm(const GView &x, const GView &y, void *workspace, hipStream_t s)
{
    uint64_t count = 1;
    for (int d = 0; d < 4; ++d) count *= x.ne[d];
    float *scale = static_cast<float *>(workspace);
    k_l2_sum<<<1, 64, 0, s>>>(x, count, scale);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    k_l2_apply<<<grid_for(count, kBlock, 65536), kBlock, 0, s>>>(x, y, count, scale);
    return hipGetLastError();
}

hipError_t launch_generic_l2_sum(const GView &x, void *workspace, hipStream_t s)
{
    uint64_t count = 1;
    for (int d = 0; d < 4; ++d) count *= x.ne[d];
    k_l2_sum<<<1, 64, 0, s>>>(x, count, static_cast<float *>(workspace));
    return hipGetLastError();
}

hipError_t launch_generic_l2_apply(const GView &x, const GView &y, const void *workspace, hipStream_t s)
{
    uint64_t count = 1;
    for (int d = 0; d < 4; ++d) count *= x.ne[d];
    k_l2_apply<<<grid_for(count, kBlock, 65536), kBlock, 0, s>>>(x, y, count, static_cast<const float *>(workspace));
    return hipGetLastError();
}

hipError_t launch_generic_count_equal(const GView &a, const GView &b, float *dst, void *workspace, hipStream_t s)
{
    uint64_t count = 1;
    for (int d = 0; d < 4; ++d) count *= a.ne[d];
    auto *partial = static_cast<unsigned long long *>(workspace);
    const uint32_t blocks = grid_for(count, kBlock, kCountBlocks);
    k_count_partial<<<blocks, kBlock, 0, s>>>(a, b, count, partial);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    k_count_final<<<1, kBlock, 0, s>>>(partial, blocks, dst);
    return hipGetLastError();
}

} // namespace emel
