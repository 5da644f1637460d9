// The register-staged GEMM's operand loads (RsOperand in pe_gemm_rs.h), run on
// the CPU over operands that end, and then begin, at an inaccessible page:
// every load lies in the operand, or this program dies, and delivers its
// elements, with zeros past K.  Tiles, splits and slabs as gemm_rs_kernel has
// them.
#include "pe_gemm_rs.h"

#include <sys/mman.h>
#include <unistd.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>

using namespace pe;

static float value(int64_t r, int64_t k, int64_t K) { return float((r * K + k) % 2039 + 1); }

template <typename E, int ROWS, int L, int BK>
static long run(int64_t rows, int64_t K, int64_t kps) {
    using O = RsOperand<E, ROWS, L, BK>;
    using T = typename E::T;
    constexpr int V = O::V;
    const int64_t rs = L == L_K ? K : 1, ks = L == L_K ? 1 : rows;
    const int64_t page = sysconf(_SC_PAGESIZE), bytes = rows * K * int64_t(sizeof(T));
    const int64_t body = (bytes + page - 1) / page * page;
    char* map = static_cast<char*>(mmap(nullptr, body + 2 * page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    if (map == MAP_FAILED || mprotect(map, page, PROT_NONE) || mprotect(map + page + body, page, PROT_NONE)) exit(3);
    long bad = 0;
    for (int at_end = 0; at_end < 2; ++at_end) {
        T* const op = reinterpret_cast<T*>(map + page + (at_end ? body - bytes : 0));
        for (int64_t r = 0; r < rows; ++r)
            for (int64_t k = 0; k < K; ++k) op[r * rs + k * ks] = T(value(r, k, K));
        for (int tm = 0; tm * ROWS < rows; ++tm) {
            const int back = O::back(int(rows) - tm * ROWS, tm), m0 = tm * ROWS - back, left = int(rows) - m0;
            for (int64_t kb = 0; kb < K; kb += kps) {
                const int klen = int(K - kb < kps ? K - kb : kps), nslabs = (klen + BK - 1) / BK;
                const int first = klen - (nslabs - 1) * BK;
                const T* const A = op + m0 * rs + kb * ks;
                for (int s = 0; s < nslabs; ++s) {
                    const int k0 = s == 0 ? 0 : first + (s - 1) * BK, kn = s == 0 ? first : BK;
                    for (int tid = 0; tid < kGemmThreads; ++tid) {
                        typename O::X x[O::NV];
                        if (s > 0 && O::whole(left)) {
                            uint32_t o[O::NV];
                            O::offsets(rs, ks, left, tid, o);
                            O::load_full(A + k0 * ks, o, x);
                        } else {
                            O::load_part(A + k0 * ks, rs, ks, left, kn, int(kb) + k0, tid, x);
                        }
                        for (int v = 0; v < O::NV; ++v) {
                            int r, k;
                            O::pos(tid, v, r, k);
                            for (int j = 0; j < V; ++j) {
                                const int rr = L == L_K ? r : r + j, kk = L == L_K ? k + j : k;
                                if (rr >= left) continue;  // feeds outputs that are never stored
                                const float want = kk < kn ? value(m0 + rr, kb + k0 + kk, K) : 0.0f;
                                bad += float(x[v][j]) != want;
                            }
                        }
                    }
                }
            }
        }
    }
    munmap(map, body + 2 * page);
    return bad;
}

int main(int argc, char** argv) {
    if (argc != 6) return 2;
    const int v = atoi(argv[1]), tile = atoi(argv[2]);
    const bool lk = !strcmp(argv[3], "k");
    const int64_t rows = atoll(argv[4]), K = atoll(argv[5]);
    long bad = 0;
    for (int64_t kps : {K, int64_t(64), int64_t(96), int64_t(160)}) {
        if (v == 4) bad += lk ? run<F32, 128, L_K, 16>(rows, K, kps) : run<F32, 128, L_MN, 16>(rows, K, kps);
        else if (tile == 128) bad += lk ? run<F16, 128, L_K, 64>(rows, K, kps) : run<F16, 128, L_MN, 64>(rows, K, kps);
        else bad += lk ? run<F16, 64, L_K, 32>(rows, K, kps) : run<F16, 64, L_MN, 32>(rows, K, kps);
    }
    if (bad) printf("%ld wrong elements\n", bad);
    return bad != 0;
}
