// Batched GEMM on 16-bit matrix cores with operands staged through registers
// (gfx950): float16 operands, and float32 operands as three bfloat16 terms.
// Same contract and tile walk as gemm_dl_kernel (pe_gemm_dl.h).
//
// Why registers: a slab's global loads are plain 16-byte loads, which need no
// more than element alignment, so rows of any pitch and any base address take
// full-width loads (gemm_dl_kernel needs whole aligned vectors; the element
// loads it left those operands to ran eight loads where this runs one); and
// what a slab holds can be converted on its way to LDS.
//
// float32: each element x is split into x0 + x1 + x2, x0 the bfloat16 nearest
// to x, x1 the one nearest to x - x0, x2 = x - x0 - x1, which 8 bits hold: the
// split is exact, |x1| <= 2^-8 |x|, |x2| <= 2^-17 |x|.  A product x y is summed
// as x0 y0 (one accumulator) and x0 y1 + x1 y0 + x1 y1 + x0 y2 + x2 y0 + x1 y2
// + x2 y1 (another), products exact, sums float32; x2 y2, below 2^-33 |x y|, is
// left out.  A sum with a single non-zero product is that product rounded once
// but for the low accumulator's own roundings, 2^-28 of it (4 million normal
// pairs emulated: largest error 5.99e-8, 5.96e-8 rounded once, 0.1 % of values
// differ; without x1 y2 and x2 y1, up to 2^-24.1 |x y|, 1.0e-7 and 4 %).  Eight
// v_mfma_f32_32x32x16_bf16 take the place of eight v_mfma_f32_32x32x2_f32 of
// twice the length: twice the rate.  The large terms' sums round once per 16 k
// instead of once per 2 k, so longer sums are nearer to 64 bits than float32
// MFMAs' (relative error at K = 192 / 777 / 4096: 7.8e-8 / 1.6e-7 / 4.0e-7
// against 2.5e-7 / 5.0e-7 / 1.2e-6).
//
// Both operands are scaled by 2^24 first, so that every float32, subnormal ones
// too, splits into normal bfloat16 terms, and the sums by 2^-48 afterwards: terms
// of products down to 2^-149 stay normal as well.  Scaled sums of 2^127 and above
// (2^79 unscaled), inf and NaN among them, as elements of 2^104 and above become,
// mark the tile, and a marked tile is computed again on float32 MFMAs.  (Without
// the scale, elements below 2^-103 had to mark it: scores under a decay of 0.95
// a position times values, 4096 x 4096 x 128, 81.7 us, now 39.7; float32 MFMAs
// 45.9.)
//
// Two LDS stages and two register sets per block: during a slab's MFMAs the
// next slab is converted and stored to the other stage (float32: a third of a
// pair's split after each MFMA, so that both units work at once) and the loads
// of two more are in flight; one barrier per slab.  K's odd end goes into the
// first slab and a tile that would pass rows ending inside a vector starts
// earlier, so that the loop's loads are all whole vectors.  LDS layouts and
// fragment reads of the L_MN operands are DlOperand's for float16, one plane
// per term; L_K rows are swizzled for the same reads.
//
// Measured on one MI355X: float16 2001 x 1537 x 3003 207 -> 47 us (cold 208 ->
// 43), 3001 x 5003 x 3011 944 -> 185; float32 4096^3 943 -> 822 us (167
// TFLOP/s), 16 x 1000 x 777 x 1536 cold 277 -> 245, 2001 x 1537 x 3003 259 ->
// 156; with six products (x1 y2 and x2 y1 left out) 733, 217 and 140.  float32
// counters at 4096^3, of that form: matrix cores 63 % busy at 1.56 GHz, where
// the float32 kernel runs 89 % at 2.2: the part is at its power limit, and the
// conversion's vector work costs clock.  Tried on it: the compiler's own
// schedule 770 us, no low accumulators (64 registers fewer, no gain, errors as
// float32's), three blocks per CU (spills), no check of small elements 723.
#pragma once

#include "pe_gemm_dl.h"

#include <type_traits>

namespace pe {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

template <typename E>
struct RsVec;
template <>
struct RsVec<F32> {
    static constexpr int V = 4, PLANES = 3;  // elements per load, 16-bit terms
    typedef float type __attribute__((ext_vector_type(4)));
    typedef float utype __attribute__((ext_vector_type(4), aligned(4)));
};
template <>
struct RsVec<F16> {
    static constexpr int V = 8, PLANES = 1;
    typedef _Float16 type __attribute__((ext_vector_type(8)));
    typedef _Float16 utype __attribute__((ext_vector_type(8), aligned(2)));
};

// Factor of both float32 operands before the split: the last bit of any
// float32, 2^-149 at the least, becomes 2^-125 or more, so that no term is a
// subnormal bfloat16.
constexpr float kRsScale = 0x1p24f;

// Two floats rounded to nearest even, a in the low half.
__device__ __forceinline__ uint32_t rs_pack(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const f32x2 x = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2));
}
// Two floats split into three bfloat16 pairs (the remainders are exact).
__device__ __forceinline__ void rs_split2(float a, float b, uint32_t (&t)[3]) {
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        t[p] = rs_pack(a, b);
        if (p < 2) {
            a = a - __builtin_bit_cast(float, t[p] << 16);
            b = b - __builtin_bit_cast(float, t[p] & 0xffff0000u);
        }
    }
}

// One operand's share of a slab of BK k: ROWS rows (m or n).  (The loads are
// host functions too: a test runs them against the ends of an operand.)
template <typename E, int ROWS, int LAYOUT, int BK>
struct RsOperand {
    using R = RsVec<E>;
    using T = typename E::T;
    using X = typename R::type;
    static constexpr int V = R::V, PLANES = R::PLANES;
    static constexpr int NV = ROWS * BK / V / kGemmThreads;  // vectors per thread
    static constexpr int PLANE = ROWS * BK;                  // elements of one term
    static constexpr int ELEMS = PLANE * PLANES;
    static constexpr int VPR = LAYOUT == L_K ? BK / V : ROWS / V;  // vectors along the contiguous axis
    static constexpr int STEP = kGemmThreads / VPR;          // rows (L_K) or k (L_MN) between a thread's vectors
    static_assert(NV >= 1 && kGemmThreads % VPR == 0, "whole vectors per thread");
    static constexpr int FLD = ROWS + 4;                     // float32 pass: LDS pitch of a k row

    __host__ __device__ __forceinline__ static void pos(int tid, int v, int& r, int& k) {
        const int a = tid / VPR + v * STEP, c = (tid % VPR) * V;
        r = LAYOUT == L_K ? a : c;
        k = LAYOUT == L_K ? c : a;
    }
    // Byte offsets, from the slab's first element, of a thread's vectors in a
    // slab whose every k is in range.  Rows past the operand repeat its last
    // row (L_K) or last vector (L_MN): they feed outputs that are never
    // stored.
    __host__ __device__ __forceinline__ static void offsets(int64_t rs, int64_t ks, int rows_left, int tid,
                                                            uint32_t (&o)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            int r, k;
            pos(tid, v, r, k);
            r = LAYOUT == L_K ? min(r, rows_left - 1) : max(0, min(r, rows_left - V));
            o[v] = uint32_t((int64_t(r) * rs + int64_t(k) * ks) * E::kBytes);
        }
    }
    // L_MN rows that end inside a vector: the tile that would pass them
    // starts `back` rows earlier, so that it ends with them (tiles of
    // operands shorter than a tile keep their place and take load_part).
    __host__ __device__ __forceinline__ static int back(int rows_left, int first_row) {
        return LAYOUT == L_MN && rows_left < ROWS && rows_left % V != 0 && first_row > 0 ? ROWS - rows_left : 0;
    }
    // Whether offsets() serves a tile: no vector straddles the last row.
    __host__ __device__ __forceinline__ static bool whole(int rows_left) {
        return LAYOUT == L_K || rows_left >= ROWS || rows_left % V == 0;
    }
    __host__ __device__ __forceinline__ static X vload(const T* p) {
        return *reinterpret_cast<const typename R::utype*>(p);
    }

    __host__ __device__ __forceinline__ static X load_one(const T* base, uint32_t o) {
        return vload(reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + o));
    }
    __host__ __device__ __forceinline__ static void load_full(const T* base, const uint32_t (&o)[NV], X (&x)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; ++v) x[v] = load_one(base, o[v]);
    }
    // x moved down by d elements, zeros shifted in (d >= V: all zero).
    __host__ __device__ __forceinline__ static void shift(X& x, int d) {
        u32x4 w = __builtin_bit_cast(u32x4, x);
        constexpr int E4 = V / 4;  // elements per dword
        if (d >= V) w = u32x4{0, 0, 0, 0};
        if (d & (2 * E4)) w = u32x4{w[2], w[3], 0, 0};
        if (d & E4) w = u32x4{w[1], w[2], w[3], 0};
        if constexpr (E4 == 2) {
            if (d & 1)
                w = u32x4{(w[0] >> 16) | (w[1] << 16), (w[1] >> 16) | (w[2] << 16), (w[2] >> 16) | (w[3] << 16),
                          w[3] >> 16};
        }
        x = __builtin_bit_cast(X, w);
    }
    // Elements n and up of x zeroed (0 <= n).
    __host__ __device__ __forceinline__ static void keep(X& x, int n) {
#pragma unroll
        for (int j = 0; j < V; ++j) x[j] = j < n ? x[j] : T(0);
    }
    // Any slab of k_left k that has `before` k of the operand before it.  A
    // vector that would pass the end of its slab (L_K) or rows (L_MN) is
    // loaded so that it ends there and moved into place; where less than a
    // vector lies before that end (a slab of fewer than V k at the operand's
    // first k) it starts at the operand's first k, and what it holds past the
    // slab is cleared.  k past the end is zero, rows past it are in-bounds
    // values (or zeros) that feed outputs which are never stored.  Every load
    // lies within V elements that the operand has along its contiguous axis.
    __host__ __device__ __forceinline__ static void load_part(const T* base, int64_t rs, int64_t ks, int rows_left,
                                                              int k_left, int before, int tid, X (&x)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            int r, k;
            pos(tid, v, r, k);
            if constexpr (LAYOUT == L_K) {
                const int k1 = max(min(k, k_left - V), -before);
                x[v] = vload(base + int64_t(min(r, rows_left - 1)) * rs + k1);
                shift(x[v], k - k1);
                if (k_left + before < V) keep(x[v], k_left - k);
            } else {
                const int r1 = min(r, rows_left - V);
                x[v] = vload(base + int64_t(min(k, k_left - 1)) * ks + r1);
                shift(x[v], k < k_left ? r - r1 : V);
            }
        }
    }

    // Element offset of (r, k) in a plane.  L_K: rows of 16 or 32 k, 16-byte groups
    // XORed so that the lanes of one ds_read_b128 phase (lanes 0-3, 12-15,
    // 20-23, 24-27 and 4-11, 16-19, 28-31 of each half wave, as bank-conflict
    // counts show) fall in distinct banks.  L_MN: 16-byte group g of k row k at
    // g ^ (KSWZ (k % 4)); with 16 groups a row (128 rows) 4 keeps the 32 lanes
    // of a ds_read_b64_tr_b16 phase (two groups of 16 rows, four k) in distinct
    // banks, where DlOperand's 2, which 64-row tiles keep, puts both groups of
    // rows on the same ones: float32 16 x 1000 x 777 x 1536, 1.5 -> 0 conflict
    // cycles per LDS instruction, 222.3 -> 219.0 us, float16 2001 x 1537 x 3003
    // 43.6 -> 43.3.
    static constexpr int KSWZ = ROWS == 128 ? 4 : 2;
    __device__ __forceinline__ static int at(int r, int k) {
        if constexpr (LAYOUT == L_MN) return k * ROWS + (((r >> 3) ^ (KSWZ * (k & 3))) << 3) + (r & 7);
        else if constexpr (BK == 16) return r * 16 + (((k >> 3) ^ ((r >> 3) & 1)) << 3) + (k & 7);
        else return (k >> 5) * ROWS * 32 + r * 32 + ((((k & 31) >> 3) ^ ((r >> 2) & 3)) << 3) + (k & 7);
    }
    using L = DlOperand<F16, ROWS, L_MN, true>;
    // Per-lane part of a fragment's address, and the fragment of block i
    // (rows 32 i .. 32 i + 31 of the wave, which starts at wrow0), MFMA step
    // st: 8 k of one row per lane.
    __device__ __forceinline__ static typename L::LaneOff lane_off(int lane, int wrow0) {
        if constexpr (LAYOUT == L_MN && KSWZ == 4) {
            // As DlOperand's, o[i] for fragment block i of a 64-row wave.
            const int G = lane >> 4, j = (lane & 15) >> 2, q = lane & 3;
            typename L::LaneOff x;
#pragma unroll
            for (int i = 0; i < 2; ++i) x.o[i] = at(wrow0 + 32 * i + 16 * (G & 1) + 4 * q, 8 * (G >> 1) + j);
            return x;
        } else if constexpr (LAYOUT == L_MN) {
            return L::lane_off(lane, wrow0);
        } else {
            typename L::LaneOff x;
#pragma unroll
            for (int st = 0; st < 2; ++st) x.o[st] = at(wrow0 + (lane & 31), (16 * st + 8 * (lane >> 5)) % BK);
            return x;
        }
    }
    __device__ __forceinline__ static f16x8 frag(const _Float16* plane, const typename L::LaneOff& lo, int wrow0, int i,
                                                 int st) {
        if constexpr (LAYOUT == L_MN) {
            f16x8 v[2];
            if constexpr (KSWZ == 4) L::frag(plane, {{lo.o[i], lo.o[i]}}, 0, 0, st, v);
            else L::frag(plane, lo, wrow0, i, st, v);
            return v[st % 2];
        } else {
            return *reinterpret_cast<const f16x8*>(plane + (st / 2) * ROWS * 32 + lo.o[st % 2] + i * 32 * (BK == 16 ? 16 : 32));
        }
    }
    // The three terms of a thread's vector v (elements 0, 1 and 2, 3).
    __device__ __forceinline__ static void store_terms(_Float16* lds, int tid, int v, const uint32_t (&tt)[2][3]) {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        int r, k;
        pos(tid, v, r, k);
        _Float16* p = lds + at(r, k);
#pragma unroll
        for (int e = 0; e < 3; ++e) *reinterpret_cast<u32x2*>(p + e * PLANE) = u32x2{tt[0][e], tt[1][e]};
    }
    // The thread's vectors into LDS; float32: scaled and split.
    __device__ __forceinline__ static void store(_Float16* lds, int tid, const X (&x)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            int r, k;
            pos(tid, v, r, k);
            if constexpr (E::kBytes == 2) {
                *reinterpret_cast<X*>(lds + at(r, k)) = x[v];
            } else {
                uint32_t tt[2][3];
                rs_split2(x[v][0] * kRsScale, x[v][1] * kRsScale, tt[0]);
                rs_split2(x[v][2] * kRsScale, x[v][3] * kRsScale, tt[1]);
                store_terms(lds, tid, v, tt);
            }
        }
    }
    // float32 pass: k-major float32, [BK][FLD].
    __device__ __forceinline__ static void store_f32(float* lds, int tid, const X (&x)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            int r, k;
            pos(tid, v, r, k);
            if constexpr (LAYOUT == L_MN) {
                f32x4 y;
#pragma unroll
                for (int j = 0; j < 4; ++j) y[j] = float(x[v][j]);
                *reinterpret_cast<f32x4*>(lds + k * FLD + r) = y;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) lds[(k + j) * FLD + r] = float(x[v][j]);
            }
        }
    }
};

// dl_store_tile's masked form for a window: rows r0 <= row < r1 and columns
// c0 <= col < c1, relative to the lane's first element.
template <int NTM, int FM, int FN>
__device__ __forceinline__ void rs_store_window(const float* wbase, uint32_t lane_off, uint32_t cms4, uint32_t cns4,
                                                int r0, int r1, int c0, int c1, const f32x16 (&acc)[FM][FN]) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            if (32 * j < c0 || 32 * j >= c1) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 32 * i + 8 * (r / 4) + r % 4;
                if (row < r0 || row >= r1) continue;
                const uint32_t off = lane_off + uint32_t(row) * cms4 + uint32_t(32 * j) * cns4;
                if constexpr (NTM == 1)
                    asm volatile("global_store_dword %0, %1, %2 nt" : : "v"(off), "v"(acc[i][j][r]), "s"(wbase));
                else
                    asm volatile("global_store_dword %0, %1, %2" : : "v"(off), "v"(acc[i][j][r]), "s"(wbase));
            }
        }
}

// Waits for this wave's LDS operations (not for its global loads) and meets
// the block.
__device__ __forceinline__ void rs_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <typename E, int BM, int BN, int BK, int AL, int BL, int MINB>
__global__ __launch_bounds__(kGemmThreads, MINB) void gemm_rs_kernel(GemmArgs g) {
    using T = typename E::T;
    using OA = RsOperand<E, BM, AL, BK>;
    using OB = RsOperand<E, BN, BL, BK>;
    constexpr bool kF32 = E::kBytes == 4;
    constexpr int PLANES = OA::PLANES, STEPS = BK / 16;
    constexpr int WM = BM / 2, WN = BN / 2;
    constexpr int FM = WM / 32, FN = WN / 32;
    constexpr int STAGE = OA::ELEMS + OB::ELEMS;
    static_assert(!kF32 || STAGE * 4 >= BK * (OA::FLD + OB::FLD) * 4, "the float32 pass fits the two stages");
    __shared__ __attribute__((aligned(16))) _Float16 lds[2 * STAGE];
    __shared__ int redo;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const uint32_t tiles_all = g.tiles_per_batch * g.nbatch_total;
    const auto loa = OA::lane_off(lane, wm * WM);
    const auto lob = OB::lane_off(lane, wn * WN);

    TileWalk walk(g.total_blocks);
    for (uint32_t bid = walk.next; bid < walk.end; bid += walk.step) {
        const uint32_t split = bid / tiles_all;
        uint32_t t = bid - split * tiles_all;
        const uint32_t batch = t / g.tiles_per_batch;
        t -= batch * g.tiles_per_batch;
        const int tm = int(t / uint32_t(g.tiles_n));
        const int tn = int(t - uint32_t(tm) * uint32_t(g.tiles_n));
        int64_t a_off = 0, b_off = 0, c_off = 0;
        uint32_t rem = batch;
        for (int d = g.nbatch - 1; d >= 0; --d) {
            uint32_t q, r;
            g.batch_div[d].divmod(rem, q, r);
            a_off += int64_t(r) * g.a_bs[d];
            b_off += int64_t(r) * g.b_bs[d];
            c_off += int64_t(r) * g.c_bs[d];
            rem = q;
        }
        const int backm = OA::back(g.M - tm * BM, tm), backn = OB::back(g.N - tn * BN, tn);
        const int m0 = tm * BM - backm, n0 = tn * BN - backn;
        const int kb = int(split) * g.k_per_split;
        const int k_len = min(g.K, kb + g.k_per_split) - kb;
        const int nslabs = (k_len + BK - 1) / BK;
        const int rows_a = g.M - m0, rows_b = g.N - n0;
        const T* const A = static_cast<const T*>(g.a) + a_off + int64_t(m0) * g.a_ms + int64_t(kb) * g.a_ks;
        const T* const B = static_cast<const T*>(g.b) + b_off + int64_t(n0) * g.b_ns + int64_t(kb) * g.b_ks;
        uint32_t offa[OA::NV], offb[OB::NV];
        OA::offsets(g.a_ms, g.a_ks, rows_a, tid, offa);
        OB::offsets(g.b_ns, g.b_ks, rows_b, tid, offb);
        // The steady loop's loads need every vector in range; K's odd end goes
        // into slab 0, so that the other slabs are whole.
        const bool steady = g.off32 && OA::whole(rows_a) && OB::whole(rows_b);
        const int first = k_len - (nslabs - 1) * BK;

        // Two register sets: slab s + 1 and s + 2 while the MFMAs read slab s.
        typename OA::X xa[2][OA::NV];
        typename OB::X xb[2][OB::NV];
        auto load_part = [&](int k0, int kn) {  // k0 .. k0 + kn - 1 into set 0
            OA::load_part(A + int64_t(k0) * g.a_ks, g.a_ms, g.a_ks, rows_a, kn, kb + k0, tid, xa[0]);
            OB::load_part(B + int64_t(k0) * g.b_ks, g.b_ns, g.b_ks, rows_b, kn, kb + k0, tid, xb[0]);
        };

        f32x16 acc[FM][FN], lo[kF32 ? FM : 1][kF32 ? FN : 1];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[i][j][r] = 0.0f;
                    if constexpr (kF32) lo[i][j][r] = 0.0f;
                }

        // The MFMAs of the slab in stage p.
        auto multiply = [&](int p) {
            const _Float16* const sa = lds + p * STAGE;
            const _Float16* const sb = sa + OA::ELEMS;
#pragma unroll
            for (int st = 0; st < STEPS; ++st) {
                f16x8 fa[PLANES][FM], fb[PLANES][FN];
#pragma unroll
                for (int p = 0; p < PLANES; ++p) {
#pragma unroll
                    for (int i = 0; i < FM; ++i) fa[p][i] = OA::frag(sa + p * OA::PLANE, loa, wm * WM, i, st);
#pragma unroll
                    for (int j = 0; j < FN; ++j) fb[p][j] = OB::frag(sb + p * OB::PLANE, lob, wn * WN, j, st);
                }
                if constexpr (kF32) {
                    auto mm = [&](int p, int q, f32x16 (&c)[FM][FN]) {
#pragma unroll
                        for (int i = 0; i < FM; ++i)
#pragma unroll
                            for (int j = 0; j < FN; ++j)
                                c[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                                    __builtin_bit_cast(bf16x8, fa[p][i]), __builtin_bit_cast(bf16x8, fb[q][j]), c[i][j],
                                    0, 0, 0);
                    };
                    mm(0, 0, acc);
                    mm(0, 1, lo);
                    mm(1, 0, lo);
                    mm(1, 1, lo);
                    mm(0, 2, lo);
                    mm(2, 0, lo);
                    mm(1, 2, lo);
                    mm(2, 1, lo);
                } else {
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[0][i], fb[0][j], acc[i][j], 0, 0, 0);
                }
            }
        };
        using P0 = std::integral_constant<int, 0>;
        using P1 = std::integral_constant<int, 1>;
        int s = 0;
        // First element of the last slab whose loads were issued; the steps
        // are opaque so that they stay in scalar registers (a kernel argument
        // loaded again inside the loop makes every LDS wait a full one).
        int64_t ska = BK * g.a_ks, skb = BK * g.b_ks;
        asm volatile("" : "+s"(ska), "+s"(skb));
        const T* na = A + int64_t(first) * g.a_ks;
        const T* nb = B + int64_t(first) * g.b_ks;
        // Steady state, slab s of parity p: its MFMAs, slab s + 1 to the other
        // stage, the loads of slab s + 3.  float32: the conversion of slab s + 1 runs between the
        // MFMAs of slab s, a third of a pair's split (four or five vector
        // instructions) after each of the first 24, so that the matrix core and the vector
        // unit work at the same time whatever the other waves of the SIMD do;
        // the compiler alone runs the two one after the other.
        auto fast = [&](auto p, auto q) {
            constexpr int P = decltype(p)::value, Q = decltype(q)::value;
            rs_barrier();  // slab s is in its stage; the other stage is free
            if (++s + 2 < nslabs) {  // else the last slab's again, unused
                na += ska;
                nb += skb;
            }
            if constexpr (!kF32) {
                multiply(P);
                OA::store(lds + Q * STAGE, tid, xa[Q]);
                OB::store(lds + Q * STAGE + OA::ELEMS, tid, xb[Q]);
                OA::load_full(na, offa, xa[Q]);
                OB::load_full(nb, offb, xb[Q]);
            } else {
                const _Float16* const sa = lds + P * STAGE;
                const _Float16* const sb = sa + OA::ELEMS;
                f16x8 fa[STEPS][PLANES][FM], fb[STEPS][PLANES][FN];
#pragma unroll
                for (int st = 0; st < STEPS; ++st)
#pragma unroll
                    for (int e = 0; e < PLANES; ++e) {
#pragma unroll
                        for (int i = 0; i < FM; ++i) fa[st][e][i] = OA::frag(sa + e * OA::PLANE, loa, wm * WM, i, st);
#pragma unroll
                        for (int j = 0; j < FN; ++j) fb[st][e][j] = OB::frag(sb + e * OB::PLANE, lob, wn * WN, j, st);
                    }
                __builtin_amdgcn_sched_barrier(0);
                constexpr int NVEC = OA::NV + OB::NV, PIECES = NVEC * 6, SLOTS = 8 * FM * FN * STEPS;
                constexpr int PER = (PIECES + SLOTS - 1) / SLOTS;
                constexpr int PI[8] = {0, 0, 1, 1, 0, 2, 1, 2}, QI[8] = {0, 1, 0, 1, 2, 0, 2, 1};
                float ra = 0.0f, rb = 0.0f;
                uint32_t tt[2][3];
#pragma unroll
                for (int slot = 0; slot < SLOTS; ++slot) {
                    const int st = slot / (8 * FM * FN), pr = slot / (FM * FN) % 8, i = slot / FN % FM, j = slot % FN;
                    f32x16& c = pr == 0 ? acc[i][j] : lo[i][j];
                    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[st][PI[pr]][i]),
                                                                __builtin_bit_cast(bf16x8, fb[st][QI[pr]][j]), c, 0, 0, 0);
#pragma unroll
                    for (int u = 0; u < PER; ++u) {
                        const int idx = slot * PER + u;
                        if (idx >= PIECES) continue;
                        const int v = idx / 6, half = idx / 3 % 2, ph = idx % 3;
                        if (ph == 0) {
                            ra = v < OA::NV ? xa[Q][v < OA::NV ? v : 0][2 * half] : xb[Q][v < OA::NV ? 0 : v - OA::NV][2 * half];
                            rb = v < OA::NV ? xa[Q][v < OA::NV ? v : 0][2 * half + 1]
                                            : xb[Q][v < OA::NV ? 0 : v - OA::NV][2 * half + 1];
                            ra = ra * kRsScale;
                            rb = rb * kRsScale;
                        } else {
                            ra = ra - __builtin_bit_cast(float, tt[half][ph - 1] << 16);
                            rb = rb - __builtin_bit_cast(float, tt[half][ph - 1] & 0xffff0000u);
                        }
                        tt[half][ph] = rs_pack(ra, rb);
                        if (half == 1 && ph == 2) {
                            if (v < OA::NV) {
                                OA::store_terms(lds + Q * STAGE, tid, v, tt);
                                xa[Q][v < OA::NV ? v : 0] = OA::load_one(na, offa[v < OA::NV ? v : 0]);
                            } else {
                                const int w = v < OA::NV ? 0 : v - OA::NV;
                                OB::store_terms(lds + Q * STAGE + OA::ELEMS, tid, w, tt);
                                xb[Q][w] = OB::load_one(nb, offb[w]);
                            }
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        load_part(0, first);
        rs_barrier();  // the last tile's reads are done
        if (kF32 && tid == 0) redo = 0;
        if (steady && nslabs > 1) {
            OA::load_full(na, offa, xa[1]);
            OB::load_full(nb, offb, xb[1]);
        }
        OA::store(lds, tid, xa[0]);
        OB::store(lds + OA::ELEMS, tid, xb[0]);
        if (steady) {
            if (nslabs > 2) {
                na += ska;
                nb += skb;
                OA::load_full(na, offa, xa[0]);
                OB::load_full(nb, offb, xb[0]);
            }
            while (s + 2 < nslabs) {
                fast(P0{}, P1{});
                fast(P1{}, P0{});
            }
#pragma unroll
            for (int v = 0; v < OA::NV; ++v) xa[0][v] = xa[1][v];
#pragma unroll
            for (int v = 0; v < OB::NV; ++v) xb[0][v] = xb[1][v];
        } else if (nslabs > 1) {
            load_part(first, BK);
        }
        // The last one or two slabs; all of them, one stage and one slab of
        // loads ahead, where the steady loop does not serve (rows that end
        // inside a vector of an operand shorter than a tile, or strides
        // beyond the 32-bit offsets).
        for (;;) {
            rs_barrier();
            multiply(0);
            if (++s >= nslabs) break;
            rs_barrier();
            OA::store(lds, tid, xa[0]);
            OB::store(lds + OA::ELEMS, tid, xb[0]);
            if (!steady && s + 1 < nslabs) load_part(first + s * BK, BK);
        }

        if constexpr (kF32) {
            // The largest scaled sum against 2^127.
            uint32_t top = 0;
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        acc[i][j][r] = acc[i][j][r] + lo[i][j][r];
                        top = max(top, __builtin_bit_cast(uint32_t, float(acc[i][j][r])) << 1);
                        acc[i][j][r] = acc[i][j][r] * (1.0f / (kRsScale * kRsScale));
                    }
            if (top >= (254u << 24)) redo = 1;
            rs_barrier();
            if (redo) {
                // The tile again, on float32 MFMAs.
                float* const fa32 = reinterpret_cast<float*>(lds);
                float* const fb32 = fa32 + BK * OA::FLD;
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
                for (s = 0; s < nslabs; ++s) {
                    load_part(s == 0 ? 0 : first + (s - 1) * BK, s == 0 ? first : BK);
                    rs_barrier();
                    OA::store_f32(fa32, tid, xa[0]);
                    OB::store_f32(fb32, tid, xb[0]);
                    rs_barrier();
                    for (int kk = 0; kk < BK; kk += 2) {
                        const int kr = kk + (lane >> 5);
                        float fa[FM], fb[FN];
#pragma unroll
                        for (int i = 0; i < FM; ++i) fa[i] = fa32[kr * OA::FLD + wm * WM + i * 32 + (lane & 31)];
#pragma unroll
                        for (int j = 0; j < FN; ++j) fb[j] = fb32[kr * OB::FLD + wn * WN + j * 32 + (lane & 31)];
#pragma unroll
                        for (int i = 0; i < FM; ++i)
#pragma unroll
                            for (int j = 0; j < FN; ++j)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
                    }
                }
            }
        }

        // Epilogue, as gemm_dl_kernel's.
        float* __restrict__ C;
        int64_t cms, cns;
        if (g.nsplit > 1) {
            C = g.partial + ((int64_t(split) * g.nbatch_total + batch) * g.M) * int64_t(g.N);
            cms = g.N;
            cns = 1;
        } else {
            C = g.c + c_off;
            cms = g.c_ms;
            cns = g.c_ns;
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7");
        const int wm0 = m0 + wm * WM, wn0 = n0 + wn * WN;
        const float* wbase = dl_uniform_base(C + int64_t(wm0) * cms + int64_t(wn0) * cns);
        uint32_t cms4 = uint32_t(cms) * 4u, cns4 = uint32_t(cns) * 4u, ln = uint32_t(lane);
        int rrem = g.M - wm0, crem = g.N - wn0;
        asm volatile("" : "+s"(cms4), "+s"(cns4), "+v"(ln), "+s"(rrem), "+s"(crem));
        const uint32_t lofs = (ln >> 5) * 4u * cms4 + (ln & 31u) * cns4;
        const int ntm = g.store_nt;  // store flavour (nt_mode)
        if (rows_a >= BM && rows_b >= BN && backm == 0 && backn == 0) {
            if (ntm == 2) dl_store_tile<2, false>(wbase, lofs, cms4, cns4, 0, 0, acc);
            else if (ntm != 0) dl_store_tile<1, false>(wbase, lofs, cms4, cns4, 0, 0, acc);
            else dl_store_tile<0, false>(wbase, lofs, cms4, cns4, 0, 0, acc);
        } else {
            // Rows and columns of this tile's own share, relative to the lane's first.
            const int lr = 4 * int(ln >> 5), lc = int(ln & 31u);
            const int r0 = backm - wm * WM - lr, c0 = backn - wn * WN - lc;
            if (ntm != 0) rs_store_window<1>(wbase, lofs, cms4, cns4, r0, rrem - lr, c0, crem - lc, acc);
            else rs_store_window<0>(wbase, lofs, cms4, cns4, r0, rrem - lr, c0, crem - lc, acc);
        }
    }
}

}  // namespace pe
