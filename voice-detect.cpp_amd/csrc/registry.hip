// registry.hip - speaker identification against an enrolled registry on gfx950.
//
// Scores S = Q R^T for B query embeddings against N enrolled ones (D dims,
// f32), then keeps the k best rows per query.  Every product of two f32
// values is exact in f64 (24 + 24 significant bits) and the D products are
// summed in f64: the arithmetic of the reference's verify, whose distance is
// 1 - sum(ea * eb) accumulated in double (src/model.cpp:65-78), so a query's
// score for a row equals 1 - verify's distance for that pair up to the order
// of the f64 sum.  Ranking: highest score first, equal scores by the lower row
// index, so the result is deterministic.
//
// registry_score_kernel: the scores on f64 MFMA (v_mfma_f64_16x16x4) from rows
// and queries loaded straight to registers; the scores of a workgroup's chunk
// of rows are staged in LDS and the best k rows per query picked there, one
// candidate list per query and chunk (in no particular order for k > 16).
// registry_merge_kernel: one workgroup per query picks the best k of its
// candidates.
#include <cfloat>

#include "common.hpp"
#include "vdk.h"

namespace vdk {
namespace {

constexpr int kMaxK = 64;
// Rows per workgroup of the score kernel, i.e. per candidate list: 256, or 64
// up to 16384 rows, where 256 would leave most CUs idle (1 x 3000 x 256, k = 5:
// 12 workgroups against 47).  A caller's workspace sized for lists of 256 rows
// is enough: the lists are then 256 rows long.
constexpr int kRows = 256, kRowsSmall = 64, kSmallN = 16384;

typedef double double4v __attribute__((ext_vector_type(4)));

// (s, i) ranks before (t, j): higher score, then lower index
__device__ __forceinline__ bool ranks_before(double s, int i, double t, int j) {
    return s > t || (s == t && i < j);
}

// Best (score, index) over `width` lanes (xor butterfly; width divides 64).
template <int WIDTH>
__device__ __forceinline__ void lane_best(double& s, int& i) {
#pragma unroll
    for (int off = WIDTH / 2; off > 0; off >>= 1) {
        const double os = __shfl_xor(s, off, WIDTH);
        const int oi = __shfl_xor(i, off, WIDTH);
        if (ranks_before(os, oi, s, i)) { s = os; i = oi; }
    }
}

// A pick of the best k out of many, used by both kernels below.  The values
// are dealt out to G >= k groups; the k-th best of the groups' maxima ranks at
// or after the k-th best value, so every value of the answer ranks at or
// before it ("the bar"), and few others do (k = 10 of 256 with 16 groups: 16).
// Those few are listed and each one's rank among them counted.  Groups are
// strided over the rows, so runs of equal scores (rows of zeros, duplicates)
// raise the bar to their k-th row instead of listing them all.

// A wave scores 16 * RT rows x 16 * QT queries, the workgroup 16 * NW * RT
// rows.  Lane l = 16 g + c feeds row / query c of each 16-wide block:
// one 16-byte load covers its 4 values of a 16-dim step (dims 4 g .. 4 g + 3,
// converted to f64 at use; the products are exact), of which MFMA j takes
// value j, so a score is summed over the dims in the order (step, j, g)
// whatever the launch's shape.  Loads go straight to registers, P steps ahead:
// a step's QT + RT loads feed 4 * QT * RT MFMAs of 64 cycles, so neither LDS
// nor L1 bandwidth matters and f64 MFMA is the bound (64 x 100000 x 192:
// 37 us at the 67 TFLOP/s that MFMAs alone reach; this kernel 79 us at k = 10,
// of which the pick is 12; the f64 FMA kernel it replaces 171 us, bound by its
// LDS reads, conversions and its k rounds of arg-max exchanges).
template <int NW, int QT, int RT, int P, int G>
__global__ __launch_bounds__(NW * 64) void registry_score_kernel(const float* __restrict__ q, int B,
                                                             const float* __restrict__ reg, int N, int D, int k,
                                                             double* __restrict__ cand_s, int* __restrict__ cand_i) {
    constexpr int NQ = 16 * QT, NR = 16 * NW * RT, LD = NR + 8;   // + 64 bytes: neighbouring queries on other banks
    constexpr int TPQ = NW * 64 / NQ, RPT = NR / TPQ, GPT = G / TPQ;   // threads per query, rows / groups per thread
    static_assert(TPQ <= 64 && GPT >= 1 && GPT <= RPT && RPT % GPT == 0 && NR <= 256, "selection shape");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    double* const sc = reinterpret_cast<double*>(smem);                        // [NQ][LD] scores
    uint8_t* const list = smem + sizeof(double) * NQ * LD;                     // [NQ][NR] rows past the bar
    int* const count = reinterpret_cast<int*>(list + NQ * NR);                 // [NQ]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
    const int q0 = blockIdx.y * NQ, b0 = blockIdx.x * NR, n0 = b0 + wave * 16 * RT;

    double4v acc[RT][QT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < QT; ++t) acc[r][t] = double4v{0.0, 0.0, 0.0, 0.0};

    if (n0 < N) {   // (wave-uniform)
        // rows and queries past the end read the last one; they are masked below
        const float *rp[RT], *qp[QT];
#pragma unroll
        for (int r = 0; r < RT; ++r) rp[r] = reg + (size_t)min(n0 + 16 * r + c, N - 1) * D + 4 * g;
#pragma unroll
        for (int t = 0; t < QT; ++t) qp[t] = q + (size_t)min(q0 + 16 * t + c, B - 1) * D + 4 * g;
        const int ns = (D + 15) >> 4;
        const float4v zero{0.0f, 0.0f, 0.0f, 0.0f};
        float4v rv[2][P][RT], qv[2][P][QT];
        auto load = [&](int buf, int s0) {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int d = (s0 + p) * 16;
                const bool on = d + 4 * g < D;   // D % 4 == 0
#pragma unroll
                for (int r = 0; r < RT; ++r)
                    rv[buf][p][r] = on ? *reinterpret_cast<const float4v*>(rp[r] + d) : zero;
#pragma unroll
                for (int t = 0; t < QT; ++t)
                    qv[buf][p][t] = on ? *reinterpret_cast<const float4v*>(qp[t] + d) : zero;
            }
        };
        auto compute = [&](int buf) {
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    double b[QT];
#pragma unroll
                    for (int t = 0; t < QT; ++t) b[t] = (double)qv[buf][p][t][j];
#pragma unroll
                    for (int r = 0; r < RT; ++r) {
                        const double a = (double)rv[buf][p][r][j];
#pragma unroll
                        for (int t = 0; t < QT; ++t)
                            acc[r][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b[t], acc[r][t], 0, 0, 0);
                    }
                }
        };
        load(0, 0);
#pragma unroll 1
        for (int s = 0; s < ns; s += 2 * P) {
            load(1, s + P);   // past the end: zeros, not loads
            compute(0);
            load(0, s + 2 * P);
            compute(1);
        }
    }

    // accumulator i of lane (g, c) is row 4 i + g of its block, query c; scores
    // that are not finite are never picked
    const double kNone = -__builtin_inf();
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = (wave * RT + r) * 16 + 4 * i + g;
                const double v = acc[r][t][i];
                sc[(16 * t + c) * LD + row] = b0 + row < N && v >= -DBL_MAX && v <= DBL_MAX ? v : kNone;
            }
    if (tid < NQ) count[tid] = 0;
    __syncthreads();

    const int qi = tid / TPQ, t = tid - qi * TPQ;   // (a query's threads are neighbours in one wave)
    const double* const sq = sc + qi * LD;
    // the maxima of this thread's groups (row t + TPQ * j is in group j % GPT), lower rows first
    double gs[GPT];
    int gr[GPT];
#pragma unroll
    for (int u = 0; u < GPT; ++u) { gs[u] = kNone; gr[u] = INT_MAX; }
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const double v = sq[t + TPQ * j];
        if (v > gs[j % GPT]) { gs[j % GPT] = v; gr[j % GPT] = t + TPQ * j; }
    }
    // the bar: the k-th best maximum (nothing is barred while fewer than k groups hold a score)
    int rank[GPT];
#pragma unroll
    for (int u = 0; u < GPT; ++u) rank[u] = 0;
#pragma unroll 4
    for (int o = 0; o < TPQ; ++o)
#pragma unroll
        for (int w = 0; w < GPT; ++w) {
            const double os = __shfl(gs[w], o, TPQ);
            const int orow = __shfl(gr[w], o, TPQ);
#pragma unroll
            for (int u = 0; u < GPT; ++u) rank[u] += ranks_before(os, orow, gs[u], gr[u]) ? 1 : 0;
        }
    double bar = kNone;
    int bar_row = INT_MAX;
#pragma unroll
    for (int u = 0; u < GPT; ++u)
        if (rank[u] == k - 1) { bar = gs[u]; bar_row = gr[u]; }
#pragma unroll
    for (int off = TPQ / 2; off > 0; off >>= 1) {
        const double os = __shfl_xor(bar, off, TPQ);
        const int orow = __shfl_xor(bar_row, off, TPQ);
        if (os > bar) { bar = os; bar_row = orow; }
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int row = t + TPQ * j;
        const double v = sq[row];
        if (v > bar || (v == bar && row <= bar_row && v > kNone)) list[qi * NR + atomicAdd(&count[qi], 1)] = (uint8_t)row;
    }
    __syncthreads();
    if (q0 + qi >= B) return;
    const int n = count[qi];
    const uint8_t* const lq = list + qi * NR;
    const size_t o = ((size_t)(q0 + qi) * gridDim.x + blockIdx.x) * k;
    if (G > 16 && n > k) {
        // many past the bar (k = 64 of 256: 166): a score that exactly k exceed, by
        // bisection between the bar and the best (n * n / TPQ comparisons to
        // rank them all took 750 us at 64 x 100000, k = 64)
        double lo = bar, hi = kNone;
#pragma unroll
        for (int u = 0; u < GPT; ++u) hi = fmax(hi, gs[u]);
#pragma unroll
        for (int off = TPQ / 2; off > 0; off >>= 1) hi = fmax(hi, __shfl_xor(hi, off, TPQ));
        int found = -1;
        for (int it = 0; it < 48; ++it) {
            const double mid = 0.5 * lo + 0.5 * hi;
            int above = 0;
#pragma unroll
            for (int j = 0; j < RPT; ++j) above += sq[t + TPQ * j] > mid ? 1 : 0;
#pragma unroll
            for (int off = TPQ / 2; off > 0; off >>= 1) above += __shfl_xor(above, off, TPQ);
            found = above == k ? 1 : found;
            if (found < 0 && above > k) lo = mid;
            if (found < 0 && above < k) hi = mid;
            if (found > 0) lo = hi = mid;   // (stays)
            if (__all(found > 0)) break;
        }
        if (found > 0) {   // (the same for a query's threads)
            int at = 0;
#pragma unroll
            for (int j = 0; j < RPT; ++j) at += sq[t + TPQ * j] > hi ? 1 : 0;
            int before = at;   // exclusive prefix over the query's threads
#pragma unroll
            for (int off = 1; off < TPQ; off <<= 1) {
                const int x = __shfl_up(before, off, TPQ);
                before += t >= off ? x : 0;
            }
            size_t w = o + before - at;
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const double v = sq[t + TPQ * j];
                if (v > hi) {
                    cand_s[w] = v;
                    cand_i[w++] = b0 + t + TPQ * j;
                }
            }
            return;
        }
    }
    for (int e = t; e < n; e += TPQ) {
        const int row = lq[e];
        const double v = sq[row];
        int r = 0;
#pragma unroll 4
        for (int m = 0; m < n; ++m) {
            const int orow = lq[m];
            r += ranks_before(sq[orow], orow, v, row) ? 1 : 0;
        }
        if (r < k) {
            cand_s[o + r] = v;
            cand_i[o + r] = b0 + row;
        }
    }
    for (int r = n + t; r < k; r += TPQ) {   // the chunk has fewer than k rows left
        cand_s[o + r] = -DBL_MAX;
        cand_i[o + r] = INT_MAX;
    }
}

// One workgroup of NT threads per query picks the best k of its n <= NT * M
// candidates (M = 0: any number, re-read) by the bar of 64 groups; should more
// than kMergeList pass the bar, by k rounds of a workgroup arg-max.  Bound by its
// latencies (one round trip to memory, then ~1000 instructions in a row): 64
// queries x 391 lists of 10 take 10 us, 21.8 with the rounds alone.
constexpr int kMergeList = 2048;
template <int NT, int M>
__global__ __launch_bounds__(NT) void registry_merge_kernel(const double* __restrict__ cand_s,
                                                            const int* __restrict__ cand_i, int n, int k,
                                                            int* __restrict__ out_i, float* __restrict__ out_s) {
    constexpr int NW = NT / 64;
    __shared__ double gs[NW][64], ls[kMergeList], bar_s;
    __shared__ int gi[NW][64], li[kMergeList], bar_i, count;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const double* const cs = cand_s + (size_t)blockIdx.x * n;
    const int* const ci = cand_i + (size_t)blockIdx.x * n;
    out_i += (size_t)blockIdx.x * k;
    out_s += (size_t)blockIdx.x * k;
    // the thread's candidates: M in registers, or (M = 0) re-read on each pass
    double v[M ? M : 1];
    int id[M ? M : 1];
    if constexpr (M > 0) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int e = tid + m * NT;
            v[m] = e < n ? cs[e] : -DBL_MAX;
            id[m] = e < n ? ci[e] : INT_MAX;
        }
    }
    auto each = [&](auto f) {
        if constexpr (M > 0) {
#pragma unroll
            for (int m = 0; m < M; ++m) f(v[m], id[m]);
        } else {
#pragma unroll 4
            for (int e = tid; e < n; e += NT) f(cs[e], ci[e]);
        }
    };
    if (tid == 0) count = 0;
    double s = -DBL_MAX;
    int i = INT_MAX;
    each([&](double x, int xi) {
        if (ranks_before(x, xi, s, i)) { s = x; i = xi; }
    });
    gs[wave][lane] = s;
    gi[wave][lane] = i;
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int w = 1; w < NW; ++w)
            if (ranks_before(gs[w][lane], gi[w][lane], s, i)) { s = gs[w][lane]; i = gi[w][lane]; }
        int rank = 0;
#pragma unroll 8
        for (int o = 0; o < 64; ++o) {
            const double os = __shfl(s, o);
            const int oi = __shfl(i, o);
            // empty groups (INT_MAX) are told apart by their lanes
            rank += ranks_before(os, oi, s, i) || (i == INT_MAX && oi == INT_MAX && o < lane) ? 1 : 0;
        }
        if (rank == k - 1) { bar_s = s; bar_i = i; }   // (i == INT_MAX: nothing is barred)
    }
    __syncthreads();
    const double bs = bar_s;
    const int bi = bar_i;
    each([&](double x, int xi) {
        if (xi != INT_MAX && !ranks_before(bs, bi, x, xi)) {
            const int at = atomicAdd(&count, 1);
            if (at < kMergeList) { ls[at] = x; li[at] = xi; }
        }
    });
    __syncthreads();
    const int nl = count;
    if (nl <= kMergeList) {
        for (int e = tid; e < nl; e += NT) {
            int r = 0;
#pragma unroll 4
            for (int m = 0; m < nl; ++m) r += ranks_before(ls[m], li[m], ls[e], li[e]) ? 1 : 0;
            if (r < k) {
                out_i[r] = li[e];
                out_s[r] = (float)ls[e];
            }
        }
        for (int r = nl + tid; r < k; r += NT) {   // fewer than k finite scores
            out_i[r] = INT_MAX;
            out_s[r] = (float)-DBL_MAX;
        }
        return;
    }
    double last_s = DBL_MAX;
    int last_i = -1;
    for (int r = 0; r < k; ++r) {
        double b = -DBL_MAX;
        int j = INT_MAX;
        each([&](double x, int xi) {
            if (xi != INT_MAX && ranks_before(last_s, last_i, x, xi) && ranks_before(x, xi, b, j)) {
                b = x;
                j = xi;
            }
        });
        lane_best<64>(b, j);
        __syncthreads();   // the previous round's maxima are read
        if (lane == 0) { gs[wave][0] = b; gi[wave][0] = j; }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NW; ++w)
            if (ranks_before(gs[w][0], gi[w][0], b, j)) { b = gs[w][0]; j = gi[w][0]; }
        if (tid == 0) {
            out_i[r] = j;
            out_s[r] = (float)b;
        }
        last_s = b;
        last_i = j;
    }
}

size_t workspace_bytes(int B, int N, int k, int rows) {
    const size_t lists = (size_t)(N + rows - 1) / rows;
    return (size_t)B * lists * k * (sizeof(double) + sizeof(int)) + 256;
}

template <int NW, int QT, int RT, int P, int G>
void launch_score(const float* q, int B, const float* reg, int N, int D, int k, double* cand_s, int* cand_i,
                  hipStream_t s) {
    constexpr int NQ = 16 * QT, NR = 16 * NW * RT;
    constexpr int lds = sizeof(double) * NQ * (NR + 8) + NQ * NR + sizeof(int) * NQ;
    if (lds > 64 * 1024)
        VDK_HIP(hipFuncSetAttribute((const void*)registry_score_kernel<NW, QT, RT, P, G>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    hipLaunchKernelGGL((registry_score_kernel<NW, QT, RT, P, G>), dim3(cdiv(N, NR), cdiv(B, NQ)),
                       dim3(NW * 64), lds, s, q, B,
                       reg, N, D, k, cand_s, cand_i);
    VDK_HIP(hipGetLastError());
}

template <int NW, int QT, int RT, int P>
void launch_score_k(const float* q, int B, const float* reg, int N, int D, int k, double* cand_s, int* cand_i,
                    hipStream_t s) {
    if (k <= 16) launch_score<NW, QT, RT, P, 16>(q, B, reg, N, D, k, cand_s, cand_i, s);
    else launch_score<NW, QT, RT, P, 64>(q, B, reg, N, D, k, cand_s, cand_i, s);
}

}  // namespace
}  // namespace vdk

using namespace vdk;

extern "C" size_t vdk_registry_topk_workspace_size(int B, int N, int k) {
    if (B <= 0 || N <= 0 || k <= 0) return 0;
    return workspace_bytes(B, N, k, N <= kSmallN ? kRowsSmall : kRows);
}

extern "C" int vdk_registry_topk(const float* d_queries, int B, const float* d_registry, int N, int D, int k,
                                 void* d_work, size_t work_bytes, int* d_idx, float* d_score, void* stream) {
    return guarded([&] {
        require(d_queries && d_registry && d_work && d_idx && d_score, "registry_topk: NULL device pointer");
        require(B > 0 && N > 0 && D > 0, "registry_topk: empty queries or registry");
        require(D % 4 == 0 && (reinterpret_cast<uintptr_t>(d_queries) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(d_registry) & 15) == 0,
                "registry_topk: D must be a multiple of 4 and the embeddings 16-byte aligned");
        require(k >= 1 && k <= kMaxK, "registry_topk: k must be in 1..64");
        require(k <= N, "registry_topk: k exceeds the registry size");
        require((size_t)N * D < (1ull << 31) && (size_t)B * D < (1ull << 31), "registry_topk: registry too large");
        require(work_bytes >= workspace_bytes(B, N, k, kRows), "registry_topk: workspace too small");
        const bool small = N <= kSmallN && work_bytes >= workspace_bytes(B, N, k, kRowsSmall);
        const int rows = small ? kRowsSmall : kRows, lists = (N + rows - 1) / rows;
        double* cand_s = static_cast<double*>(d_work);
        int* cand_i = reinterpret_cast<int*>(cand_s + (size_t)B * lists * k);
        hipStream_t s = static_cast<hipStream_t>(stream);
        // up to 16 queries one block of them per wave, two above (64 x 100000 x 192,
        // k = 10, us: 8 waves of 2 x 2 blocks 79, 4 waves of 4 x 2 92, of 4 x 4
        // 93; 1 query: 4 waves of 4 x 1 28)
        if (small) {
            if (B <= 16) launch_score_k<4, 1, 1, 4>(d_queries, B, d_registry, N, D, k, cand_s, cand_i, s);
            else launch_score_k<4, 2, 1, 2>(d_queries, B, d_registry, N, D, k, cand_s, cand_i, s);
        } else {
            if (B <= 16) launch_score_k<4, 1, 4, 2>(d_queries, B, d_registry, N, D, k, cand_s, cand_i, s);
            else launch_score_k<8, 2, 2, 1>(d_queries, B, d_registry, N, D, k, cand_s, cand_i, s);
        }
        const int n = lists * k;
        if (n <= 256 * 2)
            hipLaunchKernelGGL((registry_merge_kernel<256, 2>), dim3(B), dim3(256), 0, s, cand_s, cand_i, n, k, d_idx,
                               d_score);
        else if (n <= 1024 * 4)
            hipLaunchKernelGGL((registry_merge_kernel<1024, 4>), dim3(B), dim3(1024), 0, s, cand_s, cand_i, n, k,
                               d_idx, d_score);
        else if (n <= 1024 * 16)
            hipLaunchKernelGGL((registry_merge_kernel<1024, 16>), dim3(B), dim3(1024), 0, s, cand_s, cand_i, n, k,
                               d_idx, d_score);
        else
            hipLaunchKernelGGL((registry_merge_kernel<1024, 0>), dim3(B), dim3(1024), 0, s, cand_s, cand_i, n, k, d_idx,
                               d_score);
        VDK_HIP(hipGetLastError());
    });
}
