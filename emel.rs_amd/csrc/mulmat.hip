// mulmat.hip -- gfx950 kernels for the generic envelope's mul_mat (F32, F16)
// and mul_mat_argmax (crates/emel-kernels/src/any/generic.rs:1422-1515).
//
// The reference adds each output's products in the order of the inner
// dimension: one fused multiply-add per step in f32 (F32 operands), or an f64
// sum of f32 products (F16 operands; the product of two halves is exact in
// f32, so each step is one fused multiply-add in f64).  The matrix
// instructions v_mfma_f32_16x16x4_f32 and v_mfma_f64_16x16x4_f64 add their
// four products in that order, each with a single rounding, with denormals,
// so a chain of them over the inner dimension gives the sequential loop's
// bits (tests/test_gpu_generic.py compares them with the oracle).  Nothing is
// split along the inner dimension.
//
// Bound by those instructions where the outputs fill the chip (k = m = 4096,
// n = 512: F16 280 us, 61 TFLOP/s of the 73 that a large f64 product reaches;
// F32 154 us, 111 of 153) and by the latency of their chains where they do
// not (n = 1: 24 us, F32 25).  A lane per output that walked both operands in
// global memory took 32.1 ms for the first.
//
//   k_mm_tile   a workgroup per tile of the output, operands staged in LDS
//   k_mm_any    a lane per output, for short inner dimensions and for strides
//               that a tile's 32-bit offsets cannot span
//   k_mm_rows   a lane per row of lhs for one column, rows streamed through
//               LDS: mul_mat with n = 1 and mul_mat_argmax
//   k_mm_argmax_walk, k_mm_argmax_final
//               mul_mat_argmax for other layouts and short rows, and its merge
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "libm_replica.hpp"

namespace emel {
namespace {

typedef float acc4f __attribute__((ext_vector_type(4)));
typedef double acc4d __attribute__((ext_vector_type(4)));

// One product: y[i * y_si + j * y_sj] = sum over kk of p(i, kk) q(j, kk).
// j is the output's contiguous dimension in the reference's layouts, so the
// 16 lanes of a result row store 64 contiguous bytes.  Strides are in
// elements and not negative.
struct MmArgs {
    const void *p; // rows i: element (i, kk) at i * p_si + kk * p_sk
    const void *q; // element (j, kk) at j * q_sj + kk * q_sk
    float *y;
    int64_t p_si, p_sk, q_sj, q_sk, y_si, y_sj;
    uint32_t ni, nj;
    uint64_t k;
    uint32_t ti, tj; // tiles along i and j
};

// ---- tiles -----------------------------------------------------------------
// A 256-thread workgroup owns TI x TJ outputs.  Blocks of BK inner elements of
// its operand rows are staged in LDS, two buffers in turn with one barrier per
// block, and D blocks are in flight in registers: a tile's chain of matrix
// instructions runs at their latency, so few waves per SIMD have to cover the
// memory's latency themselves.
//
// An f32 or f64 matrix instruction occupies the SIMD's vector issue on this
// chip (33 cycles for f32 16x16x4, 65 for f64), and every vector instruction
// beside it adds its own 4 to 8 cycles.  So the loop holds as few as it can:
// loads are raw buffer loads from a base that advances in scalar registers
// (out-of-range lanes read zeros, so rows past the end need no clamp), and
// F16 is widened to f64 while it is staged, once per workgroup.
//
// F16's staged row holds BK doubles in 16-byte slots of two: slot (g, u) has
// the elements kk = 8 u + g and 8 u + 4 + g, so that lane group g = lane / 16
// of a matrix instruction feeds two instructions with one 128-bit read.  Eight
// lanes of such a read are served at a time, four of one group with rows 0-3
// (mod 8) and four of the next with rows 4-7; the slots' order and the rows'
// stride (kSlotG, kSlotU, kRow) put them in different banks.  F32 rows are
// staged as they are (p along kk, q along j) and read 4 bytes a lane.
//
// SMALL (F16, TI = TJ = 16): v_mfma_f64_4x4x4 takes 16 rows of q against 4
// rows of p at a third of the latency; each wave owns 4 rows of p.
//
// Past the end of the inner dimension p is padded with -0 and q with +0: each
// padded product is -0, which leaves every sum as it is, signed zeros
// included.
// Two waves per SIMD at least: with at most 256 registers a lane the matrix
// instructions accumulate in vector registers, without copies to and from the
// accumulation registers at the loop's ends.
template <bool F16, bool PVEC, bool QVEC, bool SMALL, int FI, int FJ, int WI, int WJ, int BK, int D>
__global__ __launch_bounds__(kBlock, 2) void k_mm_tile(MmArgs a)
{
    static_assert(D % 2 == 0, "the LDS buffers alternate with the register stages");
    constexpr int TI = SMALL ? 16 : 16 * FI * WI, TJ = SMALL ? 16 : 16 * FJ * WJ;
    constexpr int kES = F16 ? 2 : 4;
    constexpr int kChunk = 16 / kES;                    // elements per 128-bit load
    constexpr int kChunks = BK / kChunk;                // per row of a block
    // F16: slot (g, u) of a row is g * kSlotG + u * kSlotU, the row's stride 1
    // (or 2) slots past a multiple of 8.  SMALL reads four rows of p at a time,
    // so its p slots keep groups 4 apart (mod 8).
    constexpr bool kWide = kChunks >= 8;
    constexpr int kSlotG = kWide ? kChunks : 1, kSlotU = kWide ? 1 : 4;
    constexpr int kPSlotG = SMALL ? kChunks + 4 : kSlotG;
    constexpr int kRow = F16 ? (4 * kChunks + (kWide ? 1 : 2)) * 16 : BK * 4 + 16; // bytes per staged row
    constexpr int kPRow = SMALL ? (4 * kPSlotG + 1) * 16 : kRow;                    // and of p
    constexpr int kQRow = TJ + (TJ % 32 == 0 ? 16 : 0); // floats per staged row of F32's q (along j)
    constexpr int kBuf = TI * kPRow + (F16 ? TJ * kRow : BK * kQRow * 4);
    constexpr int kPLoads = TI * kChunks / kBlock;
    constexpr int kQLoads = F16 ? TJ * kChunks / kBlock : BK * TJ / 4 / kBlock;
    static_assert(TI * kChunks % kBlock == 0 && (F16 ? TJ * kChunks : BK * TJ / 4) % kBlock == 0, "whole rounds of loads");
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * kBuf];

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid % kWave;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    // Neighbouring workgroups share the operand of the dimension with more
    // tiles, the larger one.
    uint32_t bi, bj;
    if (a.ti <= a.tj) {
        bi = blockIdx.x % a.ti;
        bj = blockIdx.x / a.ti;
    } else {
        bj = blockIdx.x % a.tj;
        bi = blockIdx.x / a.tj;
    }
    const uint32_t i0 = bi * TI, j0 = bj * TJ;

    // The tile's first element of p and q, and the bytes from there to the end
    // of its last row's last element: nothing past them is read.
    const char *p0 = static_cast<const char *>(a.p) + static_cast<int64_t>(i0) * a.p_si * kES;
    const char *q0 = static_cast<const char *>(a.q) + static_cast<int64_t>(j0) * a.q_sj * kES;
    const int64_t ks = static_cast<int64_t>(a.k);
    const int64_t p_bytes = (static_cast<int64_t>(min(a.ni - i0, static_cast<uint32_t>(TI)) - 1) * a.p_si + (ks - 1) * a.p_sk + 1) * kES;
    const int64_t q_bytes = (static_cast<int64_t>(min(a.nj - j0, static_cast<uint32_t>(TJ)) - 1) * a.q_sj + (ks - 1) * a.q_sk + 1) * kES;
    auto block_rsrc = [&](const char *base, int64_t bytes, int64_t sk, uint64_t k0) {
        const int64_t at = static_cast<int64_t>(k0) * sk * kES;
        const int64_t left = bytes - at; // clamped to [0, 2^31 - 1], by its high words: scalar compares are 32 bits wide
        const int32_t high = static_cast<int32_t>(left >> 31);
        return buffer_rsrc(base + at, high < 0 ? 0u : high > 0 ? 0x7fffffffu : static_cast<uint32_t>(left));
    };
    // 16 bytes of an operand row: chunk `off` apart, element `sk` apart.
    auto load_chunk = [&](BufRsrc r, uint32_t off, uint32_t sk, bool vec) {
        if (vec) return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
        uint32_t e[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if constexpr (F16)
                e[c] = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(r, off + 4 * c, 0, 0)) |
                       (static_cast<uint32_t>(static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(r, off + 4 * c + 2, 0, 0)))
                        << 16);
            else
                e[c] = __builtin_amdgcn_raw_buffer_load_b32(r, off + c * sk, 0, 0);
        }
        return make_uint4(e[0], e[1], e[2], e[3]);
    };
    const uint32_t p_sib = static_cast<uint32_t>(a.p_si) * kES, p_skb = static_cast<uint32_t>(a.p_sk) * kES;
    const uint32_t q_sjb = static_cast<uint32_t>(a.q_sj) * kES, q_skb = static_cast<uint32_t>(a.q_sk) * kES;

    // Thread tid loads chunks tid, tid + 256, ... of the block.
    uint4 rp[D][kPLoads], rq[D][kQLoads];
    auto load = [&](int d, uint64_t k0) {
        const BufRsrc pr = block_rsrc(p0, p_bytes, a.p_sk, k0);
        const BufRsrc qr = block_rsrc(q0, q_bytes, a.q_sk, k0);
#pragma unroll
        for (int l = 0; l < kPLoads; ++l) {
            const uint32_t c = l * kBlock + tid;
            rp[d][l] = load_chunk(pr, c / kChunks * p_sib + c % kChunks * kChunk * p_skb, p_skb, PVEC);
        }
#pragma unroll
        for (int l = 0; l < kQLoads; ++l) {
            const uint32_t c = l * kBlock + tid;
            if constexpr (F16) {
                rq[d][l] = load_chunk(qr, c / kChunks * q_sjb + c % kChunks * kChunk * q_skb, q_skb, QVEC);
            } else if constexpr (QVEC) {
                rq[d][l] = load_chunk(qr, c / (TJ / 4) * q_skb + c % (TJ / 4) * 16, 4, true);
            } else { // consecutive lanes take consecutive columns
                uint32_t e[4];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t v = (4 * l + w) * kBlock + tid;
                    e[w] = __builtin_amdgcn_raw_buffer_load_b32(qr, v / TJ * q_skb + v % TJ * q_sjb, 0, 0);
                }
                rq[d][l] = make_uint4(e[0], e[1], e[2], e[3]);
            }
        }
    };
    // Elements of a chunk past the inner dimension's end: k is the chunk's
    // first.
    auto pad_chunk = [&](uint4 &w, uint64_t k, uint32_t pad) {
        uint32_t e[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if constexpr (F16) {
                e[c] = k + 2 * c >= a.k ? pad : k + 2 * c + 1 >= a.k ? (e[c] & 0xffffu) | (pad & 0xffff0000u) : e[c];
            } else {
                e[c] = k + c >= a.k ? pad : e[c];
            }
        }
        w = make_uint4(e[0], e[1], e[2], e[3]);
    };
    // Halves 4 t + g of chunk u, widened, to slot (g, u), place t.
    auto store_f16 = [&](unsigned char *row, uint32_t u, uint32_t slot_g, const uint4 &w) {
        double2 *o = reinterpret_cast<double2 *>(row) + u * kSlotU;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint32_t w0 = g < 2 ? w.x : w.y, w1 = g < 2 ? w.z : w.w;
            const uint16_t h0 = static_cast<uint16_t>(g % 2 ? w0 >> 16 : w0);
            const uint16_t h1 = static_cast<uint16_t>(g % 2 ? w1 >> 16 : w1);
            o[g * slot_g] = make_double2(hw_fp16_to_f32(h0), hw_fp16_to_f32(h1));
        }
    };
    auto store = [&](int d, uint64_t k0, unsigned char *buf, bool tail) {
#pragma unroll
        for (int l = 0; l < kPLoads; ++l) {
            const uint32_t c = l * kBlock + tid;
            if (tail) pad_chunk(rp[d][l], k0 + c % kChunks * kChunk, F16 ? 0x80008000u : 0x80000000u);
            unsigned char *row = buf + c / kChunks * kPRow;
            if constexpr (F16) store_f16(row, c % kChunks, kPSlotG, rp[d][l]);
            else *reinterpret_cast<uint4 *>(row + c % kChunks * 16) = rp[d][l];
        }
#pragma unroll
        for (int l = 0; l < kQLoads; ++l) {
            const uint32_t c = l * kBlock + tid;
            if constexpr (F16) {
                if (tail) pad_chunk(rq[d][l], k0 + c % kChunks * kChunk, 0u);
                store_f16(buf + TI * kPRow + c / kChunks * kRow, c % kChunks, kSlotG, rq[d][l]);
            } else {
                uint32_t *sq = reinterpret_cast<uint32_t *>(buf + TI * kPRow);
                if constexpr (QVEC) {
                    const uint32_t kk = c / (TJ / 4);
                    if (tail && k0 + kk >= a.k) rq[d][l] = make_uint4(0, 0, 0, 0);
                    *reinterpret_cast<uint4 *>(sq + kk * kQRow + c % (TJ / 4) * 4) = rq[d][l];
                } else {
                    const uint32_t e[4] = {rq[d][l].x, rq[d][l].y, rq[d][l].z, rq[d][l].w};
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const uint32_t v = (4 * l + w) * kBlock + tid;
                        sq[v / TJ * kQRow + v % TJ] = tail && k0 + v / TJ >= a.k ? 0u : e[w];
                    }
                }
            }
        }
    };

    using Acc = typename std::conditional<F16, acc4d, acc4f>::type;
    Acc acc[FI][FJ];
#pragma unroll
    for (int x = 0; x < FI; ++x)
#pragma unroll
        for (int z = 0; z < FJ; ++z) acc[x][z] = Acc{0, 0, 0, 0};
    double acc_small = 0.0;
    const uint32_t g = lane / 16, c16 = lane % 16;
    const uint32_t wi = wave % WI, wj = wave / WI;
    const bool multiplies = SMALL ? i0 + 4 * wave < a.ni : WI * WJ == kBlock / kWave || wave < WI * WJ;
    auto multiply = [&](const unsigned char *buf) {
        if constexpr (F16) {
            // Ahead of the other wave's staging: 5% of a whole 64x64 product.
            __builtin_amdgcn_s_setprio(2);
            const uint32_t prow = SMALL ? 4 * wave + lane % 4 : wi * FI * 16 + c16;
            const uint32_t qrow = SMALL ? c16 : wj * FJ * 16 + c16;
            const double2 *pb = reinterpret_cast<const double2 *>(buf + prow * kPRow) + g * kPSlotG;
            const double2 *qb = reinterpret_cast<const double2 *>(buf + TI * kPRow + qrow * kRow) + g * kSlotG;
#pragma unroll
            for (int u = 0; u < kChunks; ++u) {
                double2 fp[FI], fq[FJ];
#pragma unroll
                for (int x = 0; x < FI; ++x) fp[x] = pb[u * kSlotU + x * 16 * (kPRow / 16)];
#pragma unroll
                for (int z = 0; z < FJ; ++z) fq[z] = qb[u * kSlotU + z * 16 * (kRow / 16)];
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if constexpr (SMALL) {
                        acc_small = __builtin_amdgcn_mfma_f64_4x4x4f64(s ? fq[0].y : fq[0].x, s ? fp[0].y : fp[0].x,
                                                                       acc_small, 0, 0, 0);
                    } else {
#pragma unroll
                        for (int x = 0; x < FI; ++x)
#pragma unroll
                            for (int z = 0; z < FJ; ++z)
                                acc[x][z] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                    s ? fp[x].y : fp[x].x, s ? fq[z].y : fq[z].x, acc[x][z], 0, 0, 0);
                    }
                }
            }
            __builtin_amdgcn_s_setprio(0);
        } else {
            const float *pf = reinterpret_cast<const float *>(buf + (wi * FI * 16 + c16) * kRow) + g;
            const float *qf = reinterpret_cast<const float *>(buf + TI * kPRow) + g * kQRow + wj * FJ * 16 + c16;
            auto mac = [&](const float (&ep)[FI], const float (&eq)[FJ]) {
#pragma unroll
                for (int x = 0; x < FI; ++x)
#pragma unroll
                    for (int z = 0; z < FJ; ++z)
                        acc[x][z] = __builtin_amdgcn_mfma_f32_16x16x4f32(ep[x], eq[z], acc[x][z], 0, 0, 0);
            };
            auto read = [&](float (&ep)[FI], float (&eq)[FJ], int s) {
#pragma unroll
                for (int x = 0; x < FI; ++x) ep[x] = pf[x * 4 * kRow + s * 4];
#pragma unroll
                for (int z = 0; z < FJ; ++z) eq[z] = qf[s * 4 * kQRow + z * 16];
            };
            if constexpr (FI * FJ == 1) {
                // one chain: the next eight steps are read while eight are
                // multiplied (k = m = 4096, n = 16: 25 us against 34)
                constexpr int kStep = 8, kGroups = BK / 4 / kStep;
                float ep[2][kStep][FI], eq[2][kStep][FJ];
#pragma unroll
                for (int s = 0; s < kStep; ++s) read(ep[0][s], eq[0][s], s);
#pragma unroll
                for (int i = 0; i < kGroups; ++i) {
                    if (i + 1 < kGroups) {
#pragma unroll
                        for (int s = 0; s < kStep; ++s) read(ep[(i + 1) % 2][s], eq[(i + 1) % 2][s], (i + 1) * kStep + s);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int s = 0; s < kStep; ++s) mac(ep[i % 2][s], eq[i % 2][s]);
                }
            } else {
#pragma unroll 8
                for (int s = 0; s < BK / 4; ++s) {
                    float ep[FI], eq[FJ];
                    read(ep, eq, s);
                    mac(ep, eq);
                }
            }
        }
    };

    // Block b is multiplied from one buffer while the next is staged into the
    // other, between the same two barriers.  The loop has no exit inside and
    // every load in it is issued, so the later blocks' loads stay outstanding;
    // its last blocks, the one past the inner dimension's end among them, come
    // after it.
    const uint32_t nb = static_cast<uint32_t>((a.k + BK - 1) / BK);
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, d * BK);
    if (nb == 1) store(0, 0, lds, true);
    else store(0, 0, lds, false);
    load(0, D * BK);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    uint32_t b = 0;
    for (; b + D + 1 < nb; b += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            constexpr auto next = [](int x) { return (x + 1) % D; };
            if (multiplies) multiply(lds + (d % 2) * kBuf);
            store(next(d), 0, lds + ((d + 1) % 2) * kBuf, false);
            load(next(d), static_cast<uint64_t>(b + d + 1 + D) * BK);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0); // the next block's conversions would wait for its loads here
        }
    }
#pragma unroll
    for (int d = 0; d <= D; ++d) {
        if (b + d < nb) {
            if (multiplies) multiply(lds + (d % 2) * kBuf);
            if (b + d + 1 < nb) {
                store((d + 1) % D, static_cast<uint64_t>(b + d + 1) * BK, lds + ((d + 1) % 2) * kBuf, true);
                __syncthreads();
            }
        }
    }
    if (!multiplies) return;
    if constexpr (SMALL) { // lane: p row lane % 4, q row 4 (lane / 4 % 4) + g
        const uint32_t i = i0 + 4 * wave + lane % 4, j = j0 + 4 * (c16 / 4) + g;
        if (i < a.ni && j < a.nj)
            a.y[static_cast<int64_t>(i) * a.y_si + static_cast<int64_t>(j) * a.y_sj] = static_cast<float>(acc_small);
        return;
    }
    // Result register r of a lane: row 4 g + r (f32) or 4 r + g (f64), column
    // lane % 16.
#pragma unroll
    for (int x = 0; x < FI; ++x)
#pragma unroll
        for (int z = 0; z < FJ; ++z)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t i = i0 + (wi * FI + x) * 16 + (F16 ? 4 * r + g : 4 * g + r);
                const uint32_t j = j0 + (wj * FJ + z) * 16 + c16;
                if (i < a.ni && j < a.nj)
                    a.y[static_cast<int64_t>(i) * a.y_si + static_cast<int64_t>(j) * a.y_sj] =
                        static_cast<float>(acc[x][z][r]);
            }
}

template <bool F16, bool SMALL, int FI, int FJ, int WI, int WJ, int BK, int D>
void launch_tile(MmArgs a, bool pvec, bool qvec, hipStream_t s)
{
    constexpr uint32_t TI = SMALL ? 16 : 16 * FI * WI, TJ = SMALL ? 16 : 16 * FJ * WJ;
    a.ti = (a.ni + TI - 1) / TI;
    a.tj = (a.nj + TJ - 1) / TJ;
    const dim3 grid(a.ti * a.tj);
    if constexpr (F16) {
        if (pvec) k_mm_tile<true, true, true, SMALL, FI, FJ, WI, WJ, BK, D><<<grid, kBlock, 0, s>>>(a);
        else k_mm_tile<true, false, false, SMALL, FI, FJ, WI, WJ, BK, D><<<grid, kBlock, 0, s>>>(a);
    } else {
        if (pvec && qvec) k_mm_tile<false, true, true, SMALL, FI, FJ, WI, WJ, BK, D><<<grid, kBlock, 0, s>>>(a);
        else if (pvec) k_mm_tile<false, true, false, SMALL, FI, FJ, WI, WJ, BK, D><<<grid, kBlock, 0, s>>>(a);
        else k_mm_tile<false, false, false, SMALL, FI, FJ, WI, WJ, BK, D><<<grid, kBlock, 0, s>>>(a);
    }
}

template <bool F16>
__global__ __launch_bounds__(kBlock) void k_mm_any(MmArgs a)
{
    using T = typename std::conditional<F16, uint16_t, float>::type;
    const uint64_t total = static_cast<uint64_t>(a.ni) * a.nj;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t t = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; t < total; t += stride) {
        const int64_t i = static_cast<int64_t>(t / a.nj), j = static_cast<int64_t>(t % a.nj);
        const T *p = static_cast<const T *>(a.p) + i * a.p_si;
        const T *q = static_cast<const T *>(a.q) + j * a.q_sj;
        typename std::conditional<F16, double, float>::type v = 0;
        for (int64_t k = 0; k < static_cast<int64_t>(a.k); ++k) {
            if constexpr (F16)
                v += static_cast<double>(hw_fp16_to_f32(p[k * a.p_sk]) * hw_fp16_to_f32(q[k * a.q_sk]));
            else
                v = __builtin_fmaf(p[k * a.p_sk], q[k * a.q_sk], v);
        }
        a.y[i * a.y_si + j * a.y_sj] = static_cast<float>(v);
    }
}

// ---- rows ------------------------------------------------------------------
// One wave takes R rows of lhs against one vector, a lane per row and an fma
// per element in order.  A lane that walked its own row would touch a cache
// line per element and wave; here a tile of R x (2048 / R) floats (8 KB) is
// loaded in full lines, 128 bytes of a row or more at a time, two tiles ahead
// in registers, and turned in LDS (rows 16 bytes longer than a multiple of
// 128, so that neither side collides in banks).  The vector's elements are
// scalar loads.  Bound by memory where the rows fill the chip: the argmax over
// 151936 rows of 4096 takes 425 us, 5.9 TB/s (3.37 ms with a lane per row in
// global memory).
//
// mul_mat_argmax: the first row with the greatest dot.  A sequential scan from
// row 0 with a strict > keeps row 0 when its dot is NaN; otherwise the result
// is the lowest row holding the maximum of the non-NaN dots.  A candidate's
// key orders by value (-0 as +0), then by lower row; 0 is no candidate.
struct MmBest {
    uint64_t key;
    float v;
    uint32_t pad;
};

__device__ __forceinline__ uint64_t mm_key(float v, uint32_t row)
{
    if (v != v) return 0;
    const uint32_t b = __builtin_bit_cast(uint32_t, v + 0.0f);
    const uint32_t o = b & 0x80000000u ? ~b : b | 0x80000000u;
    return (static_cast<uint64_t>(o) << 32) | (0xffffffffu - row);
}

// The wave's greatest key, with its value, in lane 0's result.
__device__ __forceinline__ MmBest mm_wave_best(MmBest b)
{
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        const uint64_t k = __shfl_xor(b.key, off, kWave);
        const float v = __shfl_xor(b.v, off, kWave);
        if (k > b.key) {
            b.key = k;
            b.v = v;
        }
    }
    return b;
}

template <int R, bool ARGMAX>
__global__ __launch_bounds__(kWave) void k_mm_rows(const float *__restrict__ l, int64_t st, const float *__restrict__ h,
                                                   uint64_t k, uint32_t m, float *y, int64_t y_st, MmBest *partial,
                                                   float *row0)
{
    constexpr int D = 2, kTile = 2048 / R, kC = kTile / 4, kRow = kTile * 4 + 16;
    __shared__ __attribute__((aligned(16))) unsigned char lds[R * kRow];
    const uint32_t lane = threadIdx.x;
    const uint32_t nb = static_cast<uint32_t>((k + kTile - 1) / kTile);
    MmBest best{0, 0.0f, 0};
    for (uint32_t r0 = blockIdx.x * R; r0 < m; r0 += gridDim.x * R) { // m < 2^31
        const char *base = reinterpret_cast<const char *>(l + static_cast<int64_t>(r0) * st);
        const uint32_t rows = m - r0 < R ? m - r0 : R;
        const int64_t bytes = (static_cast<int64_t>(rows - 1) * st + static_cast<int64_t>(k)) * 4;
        float4 rv[D][8];
        auto load = [&](int d, uint32_t b) {
            const int64_t at = static_cast<int64_t>(b) * (kTile * 4);
            const int64_t left = bytes - at;
            const int32_t high = static_cast<int32_t>(left >> 31);
            const BufRsrc r = buffer_rsrc(base + at, high < 0 ? 0u : high > 0 ? 0x7fffffffu : static_cast<uint32_t>(left));
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t c = j * kWave + lane;
                rv[d][j] = ld_buf_nt(r, c / kC * (static_cast<uint32_t>(st) * 4) + c % kC * 16);
            }
        };
        auto store = [&](int d) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t c = j * kWave + lane;
                *reinterpret_cast<float4 *>(lds + c / kC * kRow + c % kC * 16) = rv[d][j];
            }
        };
        const float4 *mine = reinterpret_cast<const float4 *>(lds + lane % R * kRow);
        float v = 0.0f;
        auto add = [&](const float *hb, int c) {
            const float4 q = mine[c];
            v = __builtin_fmaf(q.x, hb[4 * c], v);
            v = __builtin_fmaf(q.y, hb[4 * c + 1], v);
            v = __builtin_fmaf(q.z, hb[4 * c + 2], v);
            v = __builtin_fmaf(q.w, hb[4 * c + 3], v);
        };
#pragma unroll
        for (int d = 0; d < D; ++d) load(d, d);
        uint32_t b = 0;
        for (; b + D < nb; b += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                store(d);
                load(d, b + d + D);
                __syncthreads();
                const float *hb = h + static_cast<uint64_t>(b + d) * kTile;
#pragma unroll
                for (int c = 0; c < kC; ++c) add(hb, c);
                __syncthreads();
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (b + d < nb) {
                store(d);
                __syncthreads();
                const uint64_t k0 = static_cast<uint64_t>(b + d) * kTile;
                const int n = static_cast<int>(min<uint64_t>(kTile, k - k0) / 4);
                for (int c = 0; c < n; ++c) add(h + k0, c);
                __syncthreads();
            }
        }
        const uint32_t row = r0 + lane;
        if (lane < rows) {
            if constexpr (ARGMAX) {
                if (row == 0) row0[0] = v;
                const uint64_t key = mm_key(v, row);
                if (key > best.key) best = MmBest{key, v, 0};
            } else {
                y[static_cast<int64_t>(row) * y_st] = v;
            }
        }
    }
    if constexpr (ARGMAX) {
        best = mm_wave_best(best);
        if (lane == 0) partial[blockIdx.x] = best;
    }
}

// Other layouts and short rows: each lane walks its own row.
__global__ __launch_bounds__(kBlock) void k_mm_argmax_walk(GenMatArgs a, MmBest *partial, float *row0)
{
    const float *l = static_cast<const float *>(a.lhs.data);
    const float *r = static_cast<const float *>(a.rhs.data);
    MmBest best{0, 0.0f, 0};
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t row = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; row < a.m; row += stride) {
        const float *lp = l + static_cast<int64_t>(row) * a.lhs.st[1];
        float v = 0.0f;
        for (uint64_t i = 0; i < a.k; ++i)
            v = __builtin_fmaf(lp[static_cast<int64_t>(i) * a.lhs.st[0]], r[static_cast<int64_t>(i) * a.rhs.st[0]], v);
        if (row == 0) row0[0] = v;
        const uint64_t key = mm_key(v, static_cast<uint32_t>(row));
        if (key > best.key) best = MmBest{key, v, 0};
    }
    best = mm_wave_best(best);
    if (threadIdx.x % kWave == 0) partial[blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave] = best;
}

constexpr int kFinalBlock = 1024;

__global__ __launch_bounds__(kFinalBlock) void k_mm_argmax_final(const MmBest *partial, uint32_t n, const float *row0,
                                                                 float *dst, int32_t *index_out)
{
    __shared__ MmBest part[kFinalBlock / kWave];
    MmBest best{0, 0.0f, 0};
    for (uint32_t i = threadIdx.x; i < n; i += kFinalBlock) {
        const MmBest o = partial[i];
        if (o.key > best.key) best = o;
    }
    best = mm_wave_best(best);
    if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kFinalBlock / kWave; ++i)
            if (part[i].key > best.key) best = part[i];
        const float v0 = row0[0];
        if (v0 != v0 || best.key == 0) {
            dst[0] = v0;
            index_out[0] = 0;
        } else {
            dst[0] = best.v;
            index_out[0] = static_cast<int32_t>(0xffffffffu - static_cast<uint32_t>(best.key));
        }
    }
}

constexpr uint32_t kMmPartials = 8192; // partial results of one argmax at most

bool rows_vectorisable(const GView &lhs, uint64_t k, const void *h, int64_t h_st)
{
    // Whole aligned chunks of a row, 64 rows within a buffer's 32-bit offsets.
    // Rows of four leave a tile of LDS nearly empty: m = 16777216 takes
    // 166 us here and 107 with a lane walking each row, the argmax 153 and 74
    // (rows of eight: 186 and 275, 174 and 294).
    return lhs.st[0] == 1 && lhs.st[1] % 4 == 0 && lhs.st[1] < (int64_t{1} << 22) && k % 4 == 0 && k >= 8 && h_st == 1 &&
           (reinterpret_cast<uintptr_t>(lhs.data) & 15u) == 0 && (reinterpret_cast<uintptr_t>(h) & 3u) == 0;
}

template <bool ARGMAX>
uint32_t launch_rows_dot(const GenMatArgs &a, MmBest *partial, float *row0, hipStream_t s)
{
    const float *l = static_cast<const float *>(a.lhs.data), *h = static_cast<const float *>(a.rhs.data);
    float *y = static_cast<float *>(a.y.data);
    const uint32_t m = static_cast<uint32_t>(a.m);
    auto go = [&](auto r) {
        constexpr int R = decltype(r)::value;
        const uint32_t blocks = static_cast<uint32_t>(std::min<uint64_t>((a.m + R - 1) / R, kMmPartials));
        k_mm_rows<R, ARGMAX><<<blocks, kWave, 0, s>>>(l, a.lhs.st[1], h, a.k, m, y, a.y.st[1], partial, row0);
        return blocks;
    };
    // about 2048 waves or more: 8 per CU, with 16 KB of loads each, cover the
    // memory's latency (60000 rows of 2048: 84 us, 5.8 TB/s)
    if (a.m >= 64 * 2048) return go(std::integral_constant<int, 64>{});
    if (a.m >= 32 * 2048) return go(std::integral_constant<int, 32>{});
    return go(std::integral_constant<int, 16>{});
}

uint64_t tiles(uint64_t ni, uint64_t nj, uint64_t t) { return ((ni + t - 1) / t) * ((nj + t - 1) / t); }

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

} // namespace

namespace {

// Which tile.  A chain of matrix instructions runs at their latency, so the
// outputs are spread over the SIMDs before tiles grow: 16x16 up to 512 of
// them (k = m = 4096, n = 32, F16: 38 us against 54 with 32x32 and 165 with
// 64x64; F32 30, 32, 87) and where one dimension has at most 16 (n = 16: 26,
// 54, 165 us), 32x32 above (n = 64: 54 us against 67 and 164), and 64x64,
// which loads and widens least per product, where its tiles fill nine tenths
// of their last round of the chip's 256 CUs (n = 512: F16 278 us against 350
// with 32x32 and 500 with 16x16, F32 158, 205, 300; n = 256: F16 164, 170,
// 250; but k = 704, m = 10533, n = 283 fills 0.81 and takes 102 against 97).
//
// Where one dimension has at most 32, a 64x64 tile is half padding or more,
// and its tiles fill their rounds on the other dimension alone.  There 32x32
// is faster while both operands are read along their lines: k = 4096 and
// m = 65536, us with 16x16 / 32x32 / 64x64, F16 n = 1 207 / 339 / 555, n = 17
// 498 / 336 / 555, k = 4095 n = 16 501 / 421 / 643; F32 n = 4 207 / 242 / 307,
// n = 32 382 / 238 / 302.  16x16 only for whole chunks of halves: F32's
// swings between 0.6 and 1.3 of 64x64 with the narrow side and the length.
// Short inner dimensions do not pay for the smaller tiles' more blocks (k = 32,
// m = 32000, n = 4, F16: 9.0 / 6.0 / 5.2), and a transposed operand is
// gathered, so that the larger tile uses more of each line (k = 4096,
// m = 65536, n = 1: 682 / 614 / 379).
//
// A tile also costs its launch of blocks however short the inner dimension is,
// so up to 32 elements a lane per output may be faster (us with lanes / with
// the tiles above: k = 1, m = 16777216, n = 1 37 / 1530, F16 38 / 2450;
// k = 1, m = n = 1 1.8 / 3.6; k = 4, m = 1048576, n = 4 16 / 65; k = 8,
// m = n = 8192 281 / 104).  Both are estimated, in us, from 15000 products timed
// at k = 1 to 4096 and 1 to 16777216 outputs: the lanes' steps one after the
// other and their loads, dearer where neighbouring outputs' elements are k
// apart; and each tile's share of the chip.  One row or column of outputs whose
// lanes read contiguous elements is a stream of the matrix, which a tile reads
// in short pieces, up to longer dimensions (m = 1048576, n = 1, lhs along m:
// k = 64 66 / 163, 512 634 / 868; lhs along k, m = 1, n = 1048576: k = 64
// 67 / 95, 256 322 / 300; 151936 outputs, lhs along m, k = 256 82 / 65).
template <bool F16>
bool lanes_are_faster(const MmArgs &a, int edge, bool pvec)
{
    const double k = static_cast<double>(a.k), nj = static_cast<double>(a.nj), outputs = a.ni * nj;
    const bool stream = (a.nj == 1 && a.p_si == 1) || (a.ni == 1 && a.q_sj == 1);
    if (stream && outputs >= (1 << 19) && a.k <= (pvec ? 128 : 512)) return true;
    if (a.k > 32) return false;
    double apart = 0.0; // a wave takes nj columns of 64 / nj rows: rows and columns it reads, per lane
    if (a.p_si != 1 && nj < 64) apart += 1 / nj;
    if (a.q_sj != 1) apart += std::min(nj, 64.0) / 64;
    const double lanes = 1.9 + 0.11 * k + outputs * 1e-6 * (1.3 + 0.6 * k + apart * (a.k < 8 ? 0.25 : 1.6) * k);
    // a launch, and a tile of 16x16, 32x32, 64x64: operands read in 16 bytes, or one by one
    constexpr double cost[2][4] = {{F16 ? 2.6 : 2.9, F16 ? 0.0034 : 0.0026, F16 ? 0.0039 : 0.0029, F16 ? 0.0064 : 0.0043},
                                   {F16 ? 4.2 : 3.8, F16 ? 0.0083 : 0.0063, F16 ? 0.0057 : 0.005, F16 ? 0.01 : 0.008}};
    const double *c = cost[!(pvec && (F16 || a.q_sj == 1))];
    return lanes < c[0] + c[edge == 16 ? 1 : edge == 32 ? 2 : 3] * static_cast<double>(tiles(a.ni, a.nj, edge));
}

template <bool F16>
void launch_mm(const MmArgs &a, bool pvec, bool qvec, hipStream_t s)
{
    const uint64_t t64 = tiles(a.ni, a.nj, 64), round = 256;
    const uint32_t narrow = std::min(a.ni, a.nj);
    const bool lines = a.p_sk == 1 && (F16 || a.q_sj == 1); // k along p, j along q (F16's q: k)
    int edge = narrow > 16 && tiles(a.ni, a.nj, 16) > 512 ? 32 : 16;
    if (10 * t64 >= 9 * ((t64 + round - 1) / round * round)) {
        edge = 64;
        if (narrow <= 32 && lines && a.k >= (F16 ? 64 : 256)) edge = F16 && narrow <= 16 && pvec && a.k >= 256 ? 16 : 32;
    }
    // and past the spans of the tiles' 32-bit offsets: the largest tile's rows and block, in bytes
    constexpr int64_t es = F16 ? 2 : 4, span = 0x7fffffff / es;
    const bool far = a.p_si > span / 256 || a.p_sk > span / 256 || a.q_sj > span / 256 || a.q_sk > span / 256;
    if (far || lanes_are_faster<F16>(a, edge, pvec)) {
        const uint64_t blocks = (static_cast<uint64_t>(a.ni) * a.nj + kBlock - 1) / kBlock;
        k_mm_any<F16><<<static_cast<uint32_t>(std::min(blocks, uint64_t{65536})), kBlock, 0, s>>>(a);
        return;
    }
    if (edge == 64) launch_tile<F16, false, 2, 2, 2, 2, 32, 4>(a, pvec, qvec, s);
    else if (edge == 32) launch_tile<F16, false, 1, 1, 2, 2, 64, 2>(a, pvec, qvec, s);
    else launch_tile<F16, F16, 1, 1, 1, 1, 128, 4>(a, pvec, qvec, s);
}

} // namespace

hipError_t launch_generic_mul_mat(const GenMatArgs &g, hipStream_t s)
{
    MmArgs a{};
    a.k = g.k;
    uint64_t ni, nj;
    bool pvec, qvec;
    // One column: the rows' waves need to fill the chip (k = 4096, us with rows
    // / with tiles: m = 4096 52 / 24, 11008 93 / 39, 14000 82 / 57, 16384 57 / 61,
    // 24000 68 / 85, 32000 93 / 109).
    if (!g.f16 && g.n == 1 && g.m >= 16384 && g.m <= 0x7fffffffull && rows_vectorisable(g.lhs, g.k, g.rhs.data, g.rhs.st[1])) {
        launch_rows_dot<false>(g, nullptr, nullptr, s);
        return hipGetLastError();
    }
    if (g.f16) { // dst [m, n] is contiguous along lhs' rows
        a.p = g.rhs.data;
        a.q = g.lhs.data;
        a.p_si = a.q_sj = static_cast<int64_t>(g.k);
        a.p_sk = a.q_sk = 1;
        a.y_si = g.y.st[1];
        a.y_sj = g.y.st[0];
        ni = g.n;
        nj = g.m;
        pvec = qvec = g.k % 8 == 0 && aligned16(a.p) && aligned16(a.q);
    } else { // dst [n, m] is contiguous along rhs' columns
        a.p = g.lhs.data;
        a.q = g.rhs.data;
        a.p_si = g.lhs.st[1];
        a.p_sk = g.lhs.st[0];
        a.q_sj = g.rhs.st[0];
        a.q_sk = g.rhs.st[1];
        a.y_si = g.y.st[1];
        a.y_sj = g.y.st[0];
        ni = g.m;
        nj = g.n;
        pvec = a.p_sk == 1 && a.p_si % 4 == 0 && g.k % 4 == 0 && aligned16(a.p);
        qvec = a.q_sj == 1 && a.q_sk % 4 == 0 && nj % 4 == 0 && aligned16(a.q);
    }
    // One launch takes fewer than 2^32 work-items, 2^24 tiles: larger products
    // run in slabs of at most 2^23 of the smallest tiles.
    const uint64_t slab_i = std::min(ni, uint64_t{1} << 26);
    const uint64_t slab_j = (uint64_t{1} << 23) / ((slab_i + 15) / 16) * 16;
    const uint64_t es = g.f16 ? 2 : 4;
    for (uint64_t i = 0; i < ni; i += slab_i)
        for (uint64_t j = 0; j < nj; j += slab_j) {
            MmArgs b = a;
            b.p = static_cast<const char *>(a.p) + i * es * static_cast<uint64_t>(a.p_si);
            b.q = static_cast<const char *>(a.q) + j * es * static_cast<uint64_t>(a.q_sj);
            b.y = static_cast<float *>(g.y.data) + static_cast<int64_t>(i) * a.y_si + static_cast<int64_t>(j) * a.y_sj;
            b.ni = static_cast<uint32_t>(ni - i < slab_i ? ni - i : slab_i);
            b.nj = static_cast<uint32_t>(nj - j < slab_j ? nj - j : slab_j);
            if (g.f16) launch_mm<true>(b, pvec, qvec, s);
            else launch_mm<false>(b, pvec, qvec, s);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    return hipSuccess;
}

uint64_t mul_mat_argmax_workspace_bytes() { return 256 + kMmPartials * sizeof(MmBest); }

hipError_t launch_generic_mul_mat_argmax(const GenMatArgs &a, hipStream_t s)
{
    char *ws = static_cast<char *>(a.workspace);
    float *row0 = reinterpret_cast<float *>(ws);
    MmBest *partial = reinterpret_cast<MmBest *>(ws + 256);
    uint32_t n;
    // Short rows' lanes leave fewer partial results to the merge: us by rows /
    // by lanes for rows of 8, m = 8192 5.2 / 5.8, 24000 6.5 / 5.6, 65536
    // 6.9 / 6.1, 262144 8.6 / 10.2; of 12, 7.1 / 6.0 at 65536; of 16, 6.6 / 6.6
    // at 24000.
    const bool few = a.k < 16 && a.m >= 12000 && a.m < (1 << 17);
    if (!few && rows_vectorisable(a.lhs, a.k, a.rhs.data, a.rhs.st[0])) {
        n = launch_rows_dot<true>(a, partial, row0, s);
    } else {
        const uint32_t blocks = static_cast<uint32_t>(std::min<uint64_t>((a.m + kBlock - 1) / kBlock, kMmPartials / (kBlock / kWave)));
        k_mm_argmax_walk<<<blocks, kBlock, 0, s>>>(a, partial, row0);
        n = blocks * (kBlock / kWave);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    k_mm_argmax_final<<<1, kFinalBlock, 0, s>>>(partial, n, row0, static_cast<float *>(a.y.data), a.index_out);
    return hipGetLastError();
}

} // namespace emel
