// Matrix-vector contractions (a GEMM whose M or N is 1) on gfx950: matvec and
// vecmat, dot products, batched rows against rows, and the scores and values
// of one decoded token against a key / value cache.
//
//   out[b, n] = sum_k W[b, n, k] * x[b, k]        (fixed order, no less exact than the tiles)
//
// What bounds these is reading W once; the MFMA GEMMs leave 63 of 64 rows of
// a tile idle and walk K in slabs with a barrier each.  Two kernels, by the
// axis along which W is contiguous:
//
//   gemv_row_kernel  (k contiguous): LPR lanes share a row, 16 bytes each,
//     and every lane holds R rows (U vectors of one row for rows longer than
//     64 vectors), so R x U loads are in flight and one x vector serves R
//     rows.  The R sums of the LPR lanes are reduced together: log2(R)
//     halving exchanges, each lane keeping half the rows it held, then plain
//     butterflies, R - 1 + log2(LPR / R) exchanges instead of R log2(LPR).
//   gemv_col_kernel  (n contiguous): a thread owns 16 bytes of columns and
//     every KR-th k of its block's range, U loads in flight; the KR partial
//     sums meet in LDS and are added in order.
//
// Few outputs and a long K: K is split over blocks and the partials are summed
// in split order or by a wave for each output, in 64 bits.  Rows may start at
// any element (16-byte loads at element alignment where the strides are not
// whole vectors); the last K % V elements of a row are read one by one and
// rows past the end are clamped in bounds and never stored.
//
// Sums: a lane or thread adds at most K / LPR or K / KR products in float32,
// and what could round more often than the matrix cores (they round a block of
// products once) is added in 64 bits: short rows and columns, the sums of
// float16 lanes and of a column's threads, the partials.  Over 340 shapes, K =
// 8 to 2^22, the relative error against 64 bits is 0.01 to 0.93 of the tiles'
// (sums all in 32 bits but for the float16 lanes': up to 1.14).
//
// Measured on one MI355X (W rotated over 1 GiB), GEMM kernels before -> now:
// f32 8192 x 4096 matvec 46.5 -> 22.1 us (6.1 TB/s; a copy reaches 6.5), the
// f16 scores and values of 512 heads x 2048 positions x 128 together 152 -> 87
// us.  W in the Infinity Cache (the same call again): f32 4096^2 ij,j->i 27.9 ->
// 10.0 us, i,ij->j 28.9 -> 18.7.  Against the first shapes: W through ordinary
// loads 24-31 and 50 + 55 us; four rows per lane for long rows (x
// shared) 30 us, two 23.6; U = 2 or 8 24.4; eight k in flight per thread for the
// columns 49, sixteen 60 us (four: 46); 64-bit lane sums exchanged through LDS
// instead of DPP 66 us for the scores (46), pairwise sums within a lane's vector
// 55-58, all products in 64 bits 51.6 for the scores, 54 for the values.
#include "pe_gemv.h"

#include <algorithm>
#include <type_traits>

namespace pe {

namespace {

constexpr int kThreads = 256;

template <typename E>
struct Vec16;
template <>
struct Vec16<F32> {
    static constexpr int V = 4;
    typedef float type __attribute__((ext_vector_type(4)));
    typedef float utype __attribute__((ext_vector_type(4), aligned(4)));
};
template <>
struct Vec16<F16> {
    static constexpr int V = 8;
    typedef _Float16 type __attribute__((ext_vector_type(8)));
    typedef _Float16 utype __attribute__((ext_vector_type(8), aligned(2)));
};

template <typename E, bool UNAL>
__device__ __forceinline__ typename Vec16<E>::type ld16(const typename E::T* p) {
    if constexpr (UNAL) return *reinterpret_cast<const typename Vec16<E>::utype*>(p);
    else return *reinterpret_cast<const typename Vec16<E>::type*>(p);
}

// W is read once: non-temporal loads.
template <typename E, bool UNAL>
__device__ __forceinline__ typename Vec16<E>::type ldw(const typename E::T* p) {
    if constexpr (UNAL) return __builtin_nontemporal_load(reinterpret_cast<const typename Vec16<E>::utype*>(p));
    else return __builtin_nontemporal_load(reinterpret_cast<const typename Vec16<E>::type*>(p));
}

// Sum of four products as two sums of two: for float16 the first product
// of each is exact, so a chain of four roundings at the size of the running sum
// becomes two at a pair's, one at the four's and one at the sum's.
template <typename E>
__device__ __forceinline__ float dot4(const typename E::T (&w)[4], const typename E::T (&x)[4]) {
    const float lo = __builtin_fmaf(E::to_f32(w[1]), E::to_f32(x[1]), E::to_f32(w[0]) * E::to_f32(x[0]));
    const float hi = __builtin_fmaf(E::to_f32(w[3]), E::to_f32(x[3]), E::to_f32(w[2]) * E::to_f32(x[2]));
    return lo + hi;
}

// acc + w x, one rounding (in 64 bits float16's product is exact in 32).
template <typename E, typename A>
__device__ __forceinline__ A mad(typename E::T w, typename E::T x, A acc) {
    if constexpr (sizeof(A) == 8 && E::kBytes == 4) return __builtin_fma(double(w), double(x), acc);
    else if constexpr (sizeof(A) == 8) return acc + A(E::to_f32(w) * E::to_f32(x));
    else return __builtin_fmaf(E::to_f32(w), E::to_f32(x), acc);
}

// acc + sum of w[e] * x[e] in element order.
template <typename E, typename A>
__device__ __forceinline__ A dot16(typename Vec16<E>::type w, typename Vec16<E>::type x, A acc) {
#pragma unroll
    for (int e = 0; e < Vec16<E>::V; ++e) acc = mad<E, A>(w[e], x[e], acc);
    return acc;
}

// Type in which the row kernel's lanes' partial sums meet: float16 operands in
// 64 bits, one rounding for all of them.  The matrix cores round a block of
// products once, which chains and meets in 32 bits do not reach (relative error
// over K = 64: tiles 5.7e-8, 32 bits 6.6e-8, this 5.2e-8; the times are the
// same).
template <typename E>
struct Meet {
    using T = float;
};
template <>
struct Meet<F16> {
    using T = double;
};

// Lane l ^ m's value (m a power of two, known when unrolled): within rows of 16
// lanes by DPP moves, which need no LDS round trip each.
__device__ __forceinline__ int xor_lane(int v, int m) {
    if (m == 1) return __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xf, 0xf, false);       // quad_perm 1,0,3,2
    if (m == 2) return __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xf, 0xf, false);       // quad_perm 2,3,0,1
    if (m == 4) {
        v = __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false);                 // half-row mirror: ^ 7
        return __builtin_amdgcn_update_dpp(v, v, 0x1B, 0xf, 0xf, false);               // quad_perm 3,2,1,0: ^ 3
    }
    if (m == 8) return __builtin_amdgcn_update_dpp(v, v, 0x128, 0xf, 0xf, false);      // row_ror 8
    return __shfl_xor(v, m);
}
__device__ __forceinline__ float xor_lane(float v, int m) {
    return __int_as_float(xor_lane(__float_as_int(v), m));
}
__device__ __forceinline__ double xor_lane(double v, int m) {
    return __hiloint2double(xor_lane(__double2hiint(v), m), xor_lane(__double2loint(v), m));
}

// Offsets of batch `b` in W, x and the output.
__device__ __forceinline__ void batch_offsets(const GemvArgs& g, uint32_t b, int64_t& w, int64_t& x, int64_t& o) {
    w = x = o = 0;
    for (int d = g.nbatch - 1; d >= 0; --d) {
        uint32_t q, r;
        g.batch_div[d].divmod(b, q, r);
        w += int64_t(r) * g.w_bs[d];
        x += int64_t(r) * g.x_bs[d];
        o += int64_t(r) * g.o_bs[d];
        b = q;
    }
}

// XROW: a tile's rows are consecutive (batch, n) pairs with an x of their own
// (few rows per batch); else a tile lies in one batch and shares x.
template <typename E, int LPR, int R, int U, bool XROW, bool UNAL>
__global__ __launch_bounds__(kThreads) void gemv_row_kernel(GemvArgs g) {
    using T = typename E::T;
    using X = typename Vec16<E>::type;
    constexpr int V = Vec16<E>::V;
    constexpr int G = 64 / LPR;      // rows side by side in a wave
    constexpr int TR = G * R;        // rows of a wave
    const int lane = threadIdx.x & 63, l = lane % LPR, grp = lane / LPR;
    const uint32_t wave = threadIdx.x >> 6;

    uint32_t batch = 0, row0;
    uint32_t nrows;
    if constexpr (XROW) {
        row0 = (blockIdx.x * 4 + wave) * TR;
        nrows = g.rows;
    } else {
        batch = blockIdx.x / g.tiles;
        row0 = ((blockIdx.x - batch * g.tiles) * 4 + wave) * TR;
        nrows = uint32_t(g.N);
    }
    if (row0 >= nrows) return;

    const int kb = int(blockIdx.y) * g.k_per_split;
    const int klen = k_range(g.K, kb, g.k_per_split);
    const T* wp[R];
    const T* xp[XROW ? R : 1];
    int64_t oo = 0;
    if constexpr (!XROW) {
        int64_t wo, xo;
        batch_offsets(g, batch, wo, xo, oo);
        xp[0] = static_cast<const T*>(g.x) + xo + kb;
        const T* w0 = static_cast<const T*>(g.w) + wo + kb;
#pragma unroll
        for (int i = 0; i < R; ++i) wp[i] = w0 + int64_t(min(row0 + i * G + grp, nrows - 1)) * g.w_ns;
    } else {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const uint32_t r = min(row0 + i * G + grp, nrows - 1);
            uint32_t b, n;
            g.n_div.divmod(r, b, n);
            int64_t wo, xo, o;
            batch_offsets(g, b, wo, xo, o);
            wp[i] = static_cast<const T*>(g.w) + wo + int64_t(n) * g.w_ns + kb;
            xp[i] = static_cast<const T*>(g.x) + xo + kb;
        }
    }

    // float16 rows of up to eight vectors: all in 64 bits (K = 32: 4.4e-8
    // through the tiles, 5.3e-8 with a 32-bit chain; K = 33 4.9e-8 and 5.3e-8).
    using A = std::conditional_t<(LPR <= 8), typename Meet<E>::T, float>;
    A acc[R][U];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int u = 0; u < U; ++u) acc[i][u] = 0;

    const int nv = klen / V;
    int v0 = 0;
    for (; v0 + LPR * U <= nv; v0 += LPR * U) {
        X w[R][U], x[XROW ? R : 1][U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = (v0 + u * LPR + l) * V;
#pragma unroll
            for (int i = 0; i < R; ++i) w[i][u] = ldw<E, UNAL>(wp[i] + k);
#pragma unroll
            for (int i = 0; i < (XROW ? R : 1); ++i) x[i][u] = ld16<E, UNAL>(xp[i] + k);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < R; ++i) acc[i][u] = dot16<E, A>(w[i][u], x[XROW ? i : 0][u], acc[i][u]);
    }
    for (; v0 < nv; v0 += LPR) {
        if (v0 + l < nv) {
            const int k = (v0 + l) * V;
            X w[R], x[XROW ? R : 1];
#pragma unroll
            for (int i = 0; i < R; ++i) w[i] = ldw<E, UNAL>(wp[i] + k);
#pragma unroll
            for (int i = 0; i < (XROW ? R : 1); ++i) x[i] = ld16<E, UNAL>(xp[i] + k);
#pragma unroll
            for (int i = 0; i < R; ++i) acc[i][0] = dot16<E, A>(w[i], x[XROW ? i : 0], acc[i][0]);
        }
    }
    for (int t = l; t < klen - nv * V; t += LPR) {
        const int k = nv * V + t;
#pragma unroll
        for (int i = 0; i < R; ++i)
            acc[i][0] = mad<E, A>(wp[i][k], xp[XROW ? i : 0][k], acc[i][0]);
    }

    using M = typename Meet<E>::T;
    M s[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        s[i] = acc[i][0];
#pragma unroll
        for (int u = 1; u < U; ++u) s[i] = s[i] + acc[i][u];
    }
    // Halving exchanges: after the one over lane bit m, a lane holds the rows
    // whose index has bit m's place set as its own lane index has.
    int held = 0;  // index of the row that s[0] is, of this group's R
    int m = LPR / 2;
#pragma unroll
    for (int half = R / 2; half >= 1 && m >= 1; half /= 2, m /= 2) {
        const bool up = (l & m) != 0;
#pragma unroll
        for (int i = 0; i < half; ++i) {
            const M keep = up ? s[i + half] : s[i];
            const M send = up ? s[i] : s[i + half];
            s[i] = keep + xor_lane(send, m);
        }
        held += up ? half : 0;
    }
    static_assert(R <= LPR, "a lane is left with one row");
#pragma unroll
    for (; m >= 1; m /= 2) s[0] = s[0] + xor_lane(s[0], m);
    // LPR / R lanes hold the same row: the first stores.
    if (l % (LPR / R) != 0) return;
    const uint32_t r = row0 + uint32_t(held) * G + grp;
    if (r >= nrows) return;
    if (g.nsplit > 1) {
        g.partial[int64_t(blockIdx.y) * g.rows + (XROW ? r : batch * uint32_t(g.N) + r)] = float(s[0]);
    } else if constexpr (XROW) {
        uint32_t b, n;
        g.n_div.divmod(r, b, n);
        int64_t wo, xo, o;
        batch_offsets(g, b, wo, xo, o);
        g.out[o + int64_t(n) * g.o_ns] = float(s[0]);
    } else {
        g.out[oo + int64_t(r) * g.o_ns] = float(s[0]);
    }
}

// CL column lanes (16 bytes of columns each) x KR = 256 / CL rows of k.
template <typename E, int CL, int U, bool UNAL>
__global__ __launch_bounds__(kThreads) void gemv_col_kernel(GemvArgs g) {
    using T = typename E::T;
    using X = typename Vec16<E>::type;
    constexpr int V = Vec16<E>::V;
    constexpr int KR = kThreads / CL;
    __shared__ double red[KR * CL * V];
    const int col = threadIdx.x % CL, kr = threadIdx.x / CL;
    const uint32_t batch = blockIdx.x / g.tiles;
    const int tile = int(blockIdx.x - batch * g.tiles);
    int64_t wo, xo, oo;
    batch_offsets(g, batch, wo, xo, oo);
    // The last vector of a row starts at N - V: its columns that another
    // vector owns too are summed twice and stored once.
    const int n_own = (tile * CL + col) * V;
    const int n0 = min(n_own, g.N - V);
    // (unsigned: k may step past an end just below 2^31)
    const uint32_t kb = blockIdx.y * uint32_t(g.k_per_split);
    const uint32_t ke = kb + uint32_t(k_range(g.K, int32_t(kb), g.k_per_split));
    const T* w = static_cast<const T*>(g.w) + wo + n0;
    const T* x = static_cast<const T*>(g.x) + xo;

    double tot[V];
#pragma unroll
    for (int e = 0; e < V; ++e) tot[e] = 0.0;
    uint32_t k = kb + kr;
    // U k at a time, in float32 or in 64 bits.
    auto walk = [&](auto zero) {
        using A = decltype(zero);
        A acc[V];
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] = zero;
        for (; k + (U - 1) * KR < ke; k += U * KR) {
            X wv[U];
            T xv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                wv[u] = ldw<E, UNAL>(w + int64_t(k + u * KR) * g.w_ks);
                xv[u] = x[int64_t(k + u * KR) * g.x_ks];
            }
            if constexpr (V == 8 && U == 4 && sizeof(A) == 4) {
#pragma unroll
                for (int e = 0; e < V; ++e) acc[e] = acc[e] + dot4<E>({wv[0][e], wv[1][e], wv[2][e], wv[3][e]}, xv);
            } else {
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int e = 0; e < V; ++e) acc[e] = mad<E, A>(wv[u][e], xv[u], acc[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < V; ++e) tot[e] = acc[e];
    };
    // 64 bits for a thread's last k, for all of a short K's (float16: sixteen a
    // thread) and where the thread rows' sums meet: in 32 bits, K = 8 to 64
    // came out up to 1.14 times as far from 64 bits as through the tiles.
    if (E::kBytes == 2 && ke - kb <= 16 * KR) walk(0.0);
    else walk(0.0f);
    for (; k < ke; k += KR) {
        const X wv = ldw<E, UNAL>(w + int64_t(k) * g.w_ks);
        const T xv = x[int64_t(k) * g.x_ks];
#pragma unroll
        for (int e = 0; e < V; ++e) tot[e] = mad<E, double>(wv[e], xv, tot[e]);
    }
    float* out = g.nsplit > 1 ? g.partial + int64_t(blockIdx.y) * g.rows + int64_t(batch) * g.N : g.out + oo;
    const int64_t o_ns = g.nsplit > 1 ? 1 : g.o_ns;
    // [kr][e][col]: each store and read is a run of CL lanes.
#pragma unroll
    for (int e = 0; e < V; ++e) red[(kr * V + e) * CL + col] = tot[e];
    __syncthreads();
    for (int i = threadIdx.x; i < CL * V; i += kThreads) {
        const int c = i % CL, e = i / CL;
        double s = red[e * CL + c];
#pragma unroll
        for (int r = 1; r < KR; ++r) s = s + red[(r * V + e) * CL + c];
        const int own = (tile * CL + c) * V;
        const int n = min(own, g.N - V) + e;
        if (own < g.N && n >= own) out[int64_t(n) * o_ns] = float(s);
    }
}

// out[row] = sum of the row's nsplit partials in 64 bits.  WAVE: one wave per
// row, lane l adding splits l, l + 64, ... in order, then a butterfly (many
// splits of few rows, where one thread per output would wait for its loads in
// turn); else a thread per row, in split order.
template <bool WAVE>
__global__ __launch_bounds__(kThreads) void gemv_reduce_kernel(GemvArgs g) {
    const uint32_t row = WAVE ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x * kThreads + threadIdx.x;
    if (row >= g.rows) return;
    const int lane = WAVE ? threadIdx.x & 63 : 0;
    double s = 0.0;
    if constexpr (WAVE) {
        for (int i = lane; i < g.nsplit; i += 64) s = s + double(g.partial[int64_t(i) * g.rows + row]);
#pragma unroll
        for (int m = 32; m >= 1; m /= 2) s = s + __shfl_xor(s, m);
    } else {
        constexpr int U = 8;
        for (int i = 0; i < g.nsplit; i += U) {
            float x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) x[u] = g.partial[int64_t(min(i + u, g.nsplit - 1)) * g.rows + row];
#pragma unroll
            for (int u = 0; u < U; ++u) s = s + (i + u < g.nsplit ? double(x[u]) : 0.0);
        }
    }
    if (lane == 0) {
        uint32_t b, n;
        g.n_div.divmod(row, b, n);
        int64_t wo, xo, o;
        batch_offsets(g, b, wo, xo, o);
        g.out[o + int64_t(n) * g.o_ns] = float(s);
    }
}

using RowFn = void (*)(GemvArgs);

template <typename E, int LPR, int R, int U>
RowFn row_fn(bool xrow, bool unal) {
    if (xrow) return unal ? &gemv_row_kernel<E, LPR, R, U, true, true> : &gemv_row_kernel<E, LPR, R, U, true, false>;
    return unal ? &gemv_row_kernel<E, LPR, R, U, false, true> : &gemv_row_kernel<E, LPR, R, U, false, false>;
}

template <typename E>
RowFn row_pick(int lpr, bool xrow, bool unal) {
    switch (lpr) {
        case 4: return row_fn<E, 4, 4, 1>(xrow, unal);
        case 8: return row_fn<E, 8, 8, 1>(xrow, unal);
        case 16: return row_fn<E, 16, 8, 1>(xrow, unal);
        case 32: return row_fn<E, 32, 8, 1>(xrow, unal);
        default: return row_fn<E, 64, 1, 4>(xrow, unal);
    }
}

template <typename E>
RowFn col_pick(int cl, bool unal) {
    switch (cl) {
        case 4: return unal ? &gemv_col_kernel<E, 4, 4, true> : &gemv_col_kernel<E, 4, 4, false>;
        case 8: return unal ? &gemv_col_kernel<E, 8, 4, true> : &gemv_col_kernel<E, 8, 4, false>;
        case 16: return unal ? &gemv_col_kernel<E, 16, 4, true> : &gemv_col_kernel<E, 16, 4, false>;
        case 32: return unal ? &gemv_col_kernel<E, 32, 4, true> : &gemv_col_kernel<E, 32, 4, false>;
        default: return unal ? &gemv_col_kernel<E, 64, 4, true> : &gemv_col_kernel<E, 64, 4, false>;
    }
}

int pow2_at_least(int64_t n, int lo, int hi) {
    int p = lo;
    while (p < hi && p < n) p *= 2;
    return p;
}

}  // namespace

// The kernel, its lane split and the K split for a GEMM descriptor whose M or
// N is 1; kind 0 = not a matrix-vector product that these kernels take.
// Nothing here depends on the operands' addresses, so the workspace size
// holds for any of them.
//
// Splits: enough for two waves per SIMD (rows) or two blocks per CU (columns),
// each at least eight loads a lane (rows) or eight k a thread (columns) long.
// Twice or four times as many cost more in partials than they hide (8192^2
// f32 vecmat 50.2 us at two blocks per CU, 55 and 58 at four and eight).
GemvPlan gemv_plan(const pe_gemm_desc& d, int64_t nb) {
    GemvPlan p{};
    if (d.tile != 0 || d.split_k != 0 || (d.M != 1 && d.N != 1)) return p;
    const int V = d.dtype == PE_F32 ? 4 : 8;
    // The vector is the operand with a single row; of two, A.
    const bool a_vec = d.M == 1;
    p.a_vec = a_vec;
    p.N = a_vec ? d.N : d.M;
    const int64_t w_ns = p.N == 1 ? 0 : (a_vec ? d.b_ns : d.a_ms);
    const int64_t w_ks = a_vec ? d.b_ks : d.a_ks;
    const int64_t x_ks = a_vec ? d.a_ks : d.b_ks;
    const int64_t rows = nb * p.N;
    if (d.K < V || rows == 0 || rows >= (int64_t(1) << 31)) return p;
    const int64_t cus = cu_count();
    if (w_ks == 1 && x_ks == 1) {
        p.kind = 1;
        p.lpr = pow2_at_least(ceil_div(d.K, V), 4, 64);
        // Tiles of rows that share an x; few rows per batch: one x each.
        const int r = p.lpr == 64 ? 1 : p.lpr == 4 ? 4 : 8;
        const int tr = 64 / p.lpr * r;
        p.xrow = p.N < tr;
        const int64_t waves = p.xrow ? ceil_div(rows, tr) : nb * ceil_div(p.N, tr);
        int64_t split = std::min<int64_t>(ceil_div(8 * cus, waves), d.K / (8 * 64 * V));
        p.split = int(std::max<int64_t>(1, std::min<int64_t>(split, 1024)));
        if (p.lpr < 64) p.split = 1;
        p.tiles = uint32_t(p.xrow ? ceil_div(rows, 4 * tr) : ceil_div(p.N, 4 * tr));
        p.blocks = p.xrow ? p.tiles : nb * int64_t(p.tiles);
        p.kps = int(ceil_div(ceil_div(d.K, p.split), 64 * V) * 64 * V);
    } else if (w_ns == 1 && p.N >= V) {
        p.kind = 2;
        p.lpr = pow2_at_least(ceil_div(p.N, V), 4, 64);
        p.tiles = uint32_t(ceil_div(p.N, int64_t(p.lpr) * V));
        p.blocks = nb * int64_t(p.tiles);
        const int kr = kThreads / p.lpr;
        int64_t split = std::min<int64_t>(ceil_div(2 * cus, p.blocks), d.K / std::max(64, 8 * kr));
        p.split = int(std::max<int64_t>(1, std::min<int64_t>(split, 64)));
        p.kps = int(ceil_div(ceil_div(d.K, p.split), kr) * kr);
    } else {
        return p;
    }
    if (p.split == 1) p.kps = int(d.K);
    p.split = int(ceil_div(d.K, p.kps));
    if (p.blocks > kMaxBlocks) p.kind = 0;  // (the tile kernels walk a smaller grid)
    p.ws_bytes = p.split > 1 ? int64_t(p.split) * rows * 4 : 0;
    return p;
}

hipError_t launch_gemv(const pe_gemm_desc& d, const GemvPlan& p, int64_t nb, const void* a, const void* b, float* c,
                       void* ws, hipStream_t s) {
    GemvArgs g{};
    g.w = p.a_vec ? b : a;
    g.x = p.a_vec ? a : b;
    g.out = c;
    g.partial = static_cast<float*>(ws);
    g.N = int32_t(p.N);
    g.K = int32_t(d.K);
    g.rows = uint32_t(nb * p.N);
    g.tiles = p.tiles;
    g.nsplit = p.split;
    g.k_per_split = p.kps;
    g.w_ns = p.N == 1 ? 0 : (p.a_vec ? d.b_ns : d.a_ms);
    g.w_ks = p.a_vec ? d.b_ks : d.a_ks;
    g.x_ks = p.a_vec ? d.a_ks : d.b_ks;
    g.o_ns = p.N == 1 ? 0 : (p.a_vec ? d.c_ns : d.c_ms);
    g.n_div.init(uint32_t(p.N));
    g.nbatch = d.nbatch;
    const int V = d.dtype == PE_F32 ? 4 : 8;
    bool al = aligned(g.w, 16) && (p.kind == 1 ? g.w_ns : g.w_ks) % V == 0;
    if (p.kind == 1) al = al && aligned(g.x, 16);
    else al = al && p.N % V == 0;
    for (int i = 0; i < d.nbatch; ++i) {
        g.batch_div[i].init(uint32_t(d.batch_shape[i]));
        g.w_bs[i] = p.a_vec ? d.b_bstride[i] : d.a_bstride[i];
        g.x_bs[i] = p.a_vec ? d.a_bstride[i] : d.b_bstride[i];
        g.o_bs[i] = d.c_bstride[i];
        al = al && g.w_bs[i] % V == 0 && (p.kind == 2 || g.x_bs[i] % V == 0);
    }
    const RowFn fn = p.kind == 1 ? (d.dtype == PE_F32 ? row_pick<F32>(p.lpr, p.xrow, !al)
                                                      : row_pick<F16>(p.lpr, p.xrow, !al))
                                 : (d.dtype == PE_F32 ? col_pick<F32>(p.lpr, !al) : col_pick<F16>(p.lpr, !al));
    void* args[] = {&g};
    hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(fn), dim3(uint32_t(p.blocks), uint32_t(p.split)),
                                   dim3(kThreads), args, 0, s);
    if (e != hipSuccess || p.split == 1) return e;
    const bool wave = p.split > kWaveReduceSplits;
    return hipLaunchKernel(wave ? reinterpret_cast<const void*>(&gemv_reduce_kernel<true>)
                                : reinterpret_cast<const void*>(&gemv_reduce_kernel<false>),
                           dim3(uint32_t(ceil_div(g.rows, wave ? 4 : kThreads))), dim3(kThreads), args, 0, s);
}

}  // namespace pe
