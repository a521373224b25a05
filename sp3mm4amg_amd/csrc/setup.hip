// setup.hip -- the step before the Galerkin product in an aggregation AMG
// setup, on the GPU: the transpose R = P^T and the smoothed-aggregation
// prolongator P = (I - omega D^-1 A) P0 (P0 = the 0/1 aggregation matrix).
// The reference receives P and R from its caller; these kernels let a whole
// hierarchy be built level after level without leaving HBM.
#include <algorithm>
#include <atomic>
#include <cstdlib>

#include "device_common.hpp"
#include "jacobi_plan.hpp"
#include "kernels.hpp"

namespace sp3mm {

// lanes per row for row-parallel kernels: a power of two near the average row
// length / SP3MM_SPMV_ROW_DIV (default 4), at most a wavefront
static int lanes_for(int64_t M, int64_t nnz)
{
    static const double div = [] {
        const char *e = getenv("SP3MM_SPMV_ROW_DIV");
        const double v = e ? atof(e) : 4.0;
        return v >= 1.0 && v <= 64.0 ? v : 4.0;
    }();
    const double avg = M ? (double)nnz / (double)M / div : 1.0;
    int L = 1;
    while (L < 64 && L < avg) L *= 2;
    return L;
}

#define SP3MM_BY_LANES(K, ...)                                                                   \
    switch (L) {                                                                                 \
    case 1: hipLaunchKernelGGL(K<1>, __VA_ARGS__); break;                                        \
    case 2: hipLaunchKernelGGL(K<2>, __VA_ARGS__); break;                                        \
    case 4: hipLaunchKernelGGL(K<4>, __VA_ARGS__); break;                                        \
    case 8: hipLaunchKernelGGL(K<8>, __VA_ARGS__); break;                                        \
    case 16: hipLaunchKernelGGL(K<16>, __VA_ARGS__); break;                                      \
    case 32: hipLaunchKernelGGL(K<32>, __VA_ARGS__); break;                                      \
    default: hipLaunchKernelGGL(K<64>, __VA_ARGS__); break;                                      \
    }

// ---------------------------------------------------------------------------
// transpose: per-column counts, scan (the caller), scatter, per-row sort
// ---------------------------------------------------------------------------
__global__ void k_col_count(const int32_t *__restrict__ col, int64_t nnz, int32_t *__restrict__ cnt)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nnz; e += stride) atomicAdd(cnt + col[e], 1);
}

// L lanes per row of A: its entries go to the rows of A^T named by their
// columns, at the next free position of that row (order fixed afterwards);
// with tsrc, each entry's index in A goes along (the transpose's permutation)
template <typename VT, int L>
__global__ void __launch_bounds__(256) k_transpose_scatter(const int64_t *__restrict__ rp,
                                                            const int32_t *__restrict__ col,
                                                            const VT *__restrict__ val, int64_t M,
                                                            const int64_t *__restrict__ trp,
                                                            int32_t *__restrict__ cursor, int32_t *__restrict__ tcol,
                                                            VT *__restrict__ tval, int32_t *__restrict__ tsrc)
{
    const int sub = threadIdx.x & (L - 1);
    const int64_t stride = (int64_t)gridDim.x * (blockDim.x / L);
    for (int64_t r = (int64_t)blockIdx.x * (blockDim.x / L) + threadIdx.x / L; r < M; r += stride) {
        for (int64_t e = rp[r] + sub; e < rp[r + 1]; e += L) {
            const int c = col[e];
            const int64_t pos = trp[c] + atomicAdd(cursor + c, 1);
            tcol[pos] = (int32_t)r;
            tval[pos] = val[e];
            if (tsrc) tsrc[pos] = (int32_t)e;
        }
    }
}

// one wavefront per row of A^T: rank sort of its (distinct) column indices;
// isrc/osrc (optional) move with the values.
// Rows of kSortBitsFrom entries or more whose columns lie within kSortSpan of
// each other set a bit per column in LDS; a column's rank is the bits below it,
// from the counts before each word.  Other rows compare every pair: keys of up
// to kSortLds entries staged in LDS, more from global memory.  Comparing costs
// n^2 / 64 steps a row, the bits n / 64 and span / 2048 (892 rows of 255 entries,
// the third level of an 81x66x71 hierarchy: 80 us and 7; 6,600 rows of 70: 15
// and 7; rows of 31 take 24 us per 48,000 by comparing).
constexpr int kSortLds = 1024;
constexpr int kSortBitsFrom = 48;
constexpr int kSortSpan = kSortLds / 2 * 32;  // half the row's LDS for bits, half for counts

template <typename VT>
__global__ void __launch_bounds__(256) k_sort_rows(const int64_t *__restrict__ rp, int64_t M,
                                                    const int32_t *__restrict__ icol, const VT *__restrict__ ival,
                                                    const int32_t *__restrict__ isrc, int32_t *__restrict__ ocol,
                                                    VT *__restrict__ oval, int32_t *__restrict__ osrc)
{
    __shared__ int keys[4][kSortLds];
    const int w = threadIdx.x / kWave;
    const int l = lane();
    int *kw = keys[w];
    for (int64_t r = (int64_t)blockIdx.x * 4 + w; r < M; r += (int64_t)gridDim.x * 4) {
        const int64_t b = rp[r];
        const int n = (int)(rp[r + 1] - b);
        if (n >= kSortBitsFrom) {
            int lo = INT32_MAX, hi = 0;
            for (int j = l; j < n; j += kWave) {
                const int k = icol[b + j];
                lo = min(lo, k);
                hi = max(hi, k);
            }
            for (int o = 32; o > 0; o >>= 1) {
                lo = min(lo, __shfl_xor(lo, o));
                hi = max(hi, __shfl_xor(hi, o));
            }
            if (hi - lo < kSortSpan) {
                unsigned *bits = reinterpret_cast<unsigned *>(kw);
                int *before = kw + kSortLds / 2;
                const int words = (hi - lo) / 32 + 1, per = (words + kWave - 1) / kWave;
                for (int i = l; i < words; i += kWave) bits[i] = 0u;
                wave_sync();
                for (int j = l; j < n; j += kWave) {
                    const int d = icol[b + j] - lo;
                    atomicOr(bits + (d >> 5), 1u << (d & 31));
                }
                wave_sync();
                const int w0 = min(l * per, words), w1 = min(w0 + per, words);
                int own = 0;
                for (int i = w0; i < w1; i++) own += __popc(bits[i]);
                int run = own;
                for (int o = 1; o < kWave; o <<= 1) {
                    const int y = __shfl_up(run, o);
                    if (l >= o) run += y;
                }
                run -= own;
                for (int i = w0; i < w1; i++) {
                    before[i] = run;
                    run += __popc(bits[i]);
                }
                wave_sync();
                for (int j = l; j < n; j += kWave) {
                    const int k = icol[b + j], d = k - lo;
                    const int rank = before[d >> 5] + __popc(bits[d >> 5] & ((1u << (d & 31)) - 1u));
                    ocol[b + rank] = k;
                    oval[b + rank] = ival[b + j];
                    if (osrc) osrc[b + rank] = isrc[b + j];
                }
                wave_sync();
                continue;
            }
        }
        const bool staged = n <= kSortLds;
        if (staged)
            for (int j = l; j < n; j += kWave) kw[j] = icol[b + j];
        wave_sync();
        const int *src = staged ? kw : icol + b;
        for (int j = l; j < n; j += kWave) {
            const int k = src[j];
            int rank = 0;
            for (int i = 0; i < n; i++) rank += src[i] < k;
            ocol[b + rank] = k;
            oval[b + rank] = ival[b + j];
            if (osrc) osrc[b + rank] = isrc[b + j];
        }
        wave_sync();
    }
}

// out[j] = src[perm[j]]: the values of a transpose whose pattern is known
template <typename VT>
__global__ void __launch_bounds__(256) k_gather_vals(const VT *__restrict__ src, const int32_t *__restrict__ perm,
                                                      int64_t n, VT *__restrict__ out)
{
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x)
        out[j] = src[perm[j]];
}

// ---------------------------------------------------------------------------
// S = I - omega D^-1 A on the pattern of A (a missing diagonal is inserted)
// ---------------------------------------------------------------------------
// d_i = a_ii (mode 0) or |a_ii| + 1 (mode 1).  L lanes per row; row r's
// diagonal value, whether it is stored and how many of its columns are
// smaller, summed over the lanes.
template <int L>
__device__ __forceinline__ void sa_row_scan(const int32_t *__restrict__ col, const double *__restrict__ val,
                                            int64_t b, int64_t e1, int64_t r, int sub, double &d, int &nless,
                                            int &has)
{
    d = 0.0;
    nless = 0;
    has = 0;
    for (int64_t e = b + sub; e < e1; e += L) {
        const int c = col[e];
        if (c == r) {
            if (val) d = val[e];
            has = 1;
        }
        nless += c < r;
    }
    for (int o = L / 2; o > 0; o >>= 1) {
        d += __shfl_xor(d, o, L);
        nless += __shfl_xor(nless, o, L);
        has |= __shfl_xor(has, o, L);
    }
}

// count pass: row lengths of S
template <int L>
__global__ void __launch_bounds__(256) k_sa_count(const int64_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                   int64_t M, int32_t *__restrict__ len)
{
    const int sub = threadIdx.x & (L - 1);
    const int64_t stride = (int64_t)gridDim.x * (blockDim.x / L);
    for (int64_t r = (int64_t)blockIdx.x * (blockDim.x / L) + threadIdx.x / L; r < M; r += stride) {
        double d;
        int nless, has;
        sa_row_scan<L>(col, nullptr, rp[r], rp[r + 1], r, sub, d, nless, has);
        if (sub == 0) len[r] = (int32_t)(rp[r + 1] - rp[r]) + (has ? 0 : 1);
    }
}

// fill pass: S's columns and values at the offsets srp of the count pass (the
// missing diagonal goes before the first larger column)
template <int L>
__global__ void __launch_bounds__(256) k_sa_fill(const int64_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                  const double *__restrict__ val, int64_t M, double omega, int mode,
                                                  const int64_t *__restrict__ srp, int32_t *__restrict__ scol,
                                                  double *__restrict__ sval, int *__restrict__ err)
{
    const int sub = threadIdx.x & (L - 1);
    const int64_t stride = (int64_t)gridDim.x * (blockDim.x / L);
    for (int64_t r = (int64_t)blockIdx.x * (blockDim.x / L) + threadIdx.x / L; r < M; r += stride) {
        const int64_t b = rp[r], e1 = rp[r + 1];
        double d;
        int nless, has;
        sa_row_scan<L>(col, val, b, e1, r, sub, d, nless, has);
        if (mode == 1) d = fabs(d) + 1.0;
        if (d == 0.0) {
            if (sub == 0) atomicOr(err, kErrBadInput);
            continue;
        }
        const double w = omega / d;
        const int64_t o0 = srp[r];
        // S's row r was sized when the plan was built; a row of A that has
        // grown since (its pattern changed) is reported, not written past
        if (o0 + (e1 - b) + (has ? 0 : 1) != srp[r + 1]) {
            if (sub == 0) atomicOr(err, kErrOverflow);
            continue;
        }
        for (int64_t e = b + sub; e < e1; e += L) {
            const int c = col[e];
            const int64_t pos = o0 + (e - b) + (!has && c > r ? 1 : 0);
            scol[pos] = c;
            sval[pos] = -w * val[e] + (c == r ? 1.0 : 0.0);
        }
        if (!has && sub == 0) {
            scol[o0 + nless] = (int32_t)r;
            sval[o0 + nless] = 1.0;
        }
    }
}

// P0: one entry 1.0 per row at column agg[r]; rejects aggregates out of range
__global__ void k_p0_fill(const int64_t *__restrict__ agg, int64_t M, int64_t nagg, int64_t *__restrict__ rp,
                          int32_t *__restrict__ rp32, int32_t *__restrict__ col, double *__restrict__ val,
                          int *__restrict__ err)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r <= M; r += stride) {
        rp[r] = r;
        if (rp32) rp32[r] = (int32_t)r;
        if (r < M) {
            const int64_t a = agg[r];
            if (a < 0 || a >= nagg) atomicOr(err, kErrBadInput);
            col[r] = (int32_t)(a < 0 || a >= nagg ? 0 : a);
            val[r] = 1.0;
        }
    }
}

__global__ void k_agg_narrow(const int64_t *__restrict__ agg, int64_t M, int64_t nagg, int32_t *__restrict__ out,
                             int *__restrict__ err)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < M; r += stride) {
        const int64_t a = agg[r];
        const bool ok = a >= 0 && a < nagg;
        if (!ok) atomicOr(err, kErrBadInput);
        out[r] = ok ? (int32_t)a : 0;
    }
}

// Row r of P = (I - omega D^-1 A) P0 straight from row r of A: entry (r, k)
// contributes -omega a_rk / d_r (+ 1 on the diagonal, which counts as stored)
// to column agg[k], equal columns added in increasing k.  FILL = false: row
// lengths only.
// L = 8: rows of at most 8 entries (diagonal included) sit in 8 lanes, one
// entry each; every lane compares its aggregate with the others' by shuffles,
// so a row costs 16 shuffles and no LDS, and 8 rows share a wavefront.
// Longer rows (all of them with L = 64) take the whole wavefront and an LDS
// hash table of up to CAP slots, keyed by the aggregate; a row of CAP entries
// or more raises kErrLongRow.  (Comparing all pairs of a row staged in LDS
// took 2.2 ms on the coarse levels of a 96^3 hierarchy, the tables 0.06.)
// It replaces S = I - omega D^-1 A in HBM and the SpGEMM S P0 (count, scan,
// fill, P0, binning, hash kernel, scan, gather): HBM-bound, 12 bytes per entry
// of A and of P per pass, the gathers of agg stay in L2.  96^3 7-point
// operator: 0.70 -> 0.057 ms per recomputation.
template <int L, int CAP, bool FILL>
__global__ void __launch_bounds__(256) k_sa_rows(const int64_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                  const double *__restrict__ val, const int32_t *__restrict__ agg,
                                                  int64_t M, double omega, int mode, const int64_t *__restrict__ prp,
                                                  int32_t *__restrict__ len, int32_t *__restrict__ pcol,
                                                  double *__restrict__ pval, int *__restrict__ maxlen,
                                                  int *__restrict__ err)
{
    __shared__ double sv[4][FILL ? CAP : 1];
    __shared__ int sk[4][CAP];
    static_assert(L == 8 || L == kWave, "register rows of 8 lanes, or wavefronts");
    const int wv = threadIdx.x / kWave, l = lane(), sub = l & (L - 1), lead = l & ~(L - 1);
    constexpr int RPW = kWave / L;  // rows per wavefront
    const uint64_t part = L == kWave ? ~0ull : ((1ull << L) - 1) << lead;
    const int64_t stride = (int64_t)gridDim.x * 4 * RPW;
    int longest = 0;
    for (int64_t r0 = ((int64_t)blockIdx.x * 4 + wv) * RPW; r0 < M; r0 += stride) {
        const int64_t r = r0 + l / L;
        const int64_t b = r < M ? rp[r] : 0;
        const int64_t n64 = r < M ? rp[r + 1] - b : 0;
        const bool fits = L < kWave && n64 <= L;
        const int n = fits ? (int)n64 : 0;
        int c = -1;
        double v = 0.0;
        if (sub < n) {
            c = col[b + sub];
            if (FILL) v = val[b + sub];
        }
        const bool isd = sub < n && c == r;
        const bool has = (ballot(isd) & part) != 0;
        const int m = r < M && fits ? n + (has ? 0 : 1) : 0;  // entries with the diagonal
        const bool is_long = r < M && (!fits || m > L);
        if (sub == n && m == n + 1 && m <= L) c = (int)r;  // the missing diagonal
        const bool act = sub < m && m <= L;
        const int key = act ? agg[c] : INT32_MAX;
        double s = 0.0;
        bool bad = false;
        if (FILL) {
            double d = isd ? v : 0.0;
            for (int o = L / 2; o > 0; o >>= 1) d += __shfl_xor(d, o, L);
            if (mode == 1) d = fabs(d) + 1.0;
            bad = act && d == 0.0;
            if (bad) atomicOr(err, kErrBadInput);
            else if (act) s = -(omega / d) * v + (c == r ? 1.0 : 0.0);
        }
        bool first = act;
        double sum = 0.0;
#pragma unroll 8
        for (int i = 0; i < L; i++) {
            const int ki = __shfl(key, i, L);
            if (FILL) {
                const double si = __shfl(s, i, L);
                if (ki == key) sum += si;
            }
            if (ki == key && i < sub) first = false;
        }
        const uint64_t fm = ballot(first) & part;
        if (!FILL) {
            if (sub == 0 && r < M && !is_long) len[r] = __popcll(fm);
        } else {
            const uint64_t fl = fm >> lead;
            int rank = 0;
#pragma unroll 8
            for (int i = 0; i < L; i++) {
                const int ki = __shfl(key, i, L);
                rank += ((fl >> i) & 1) && ki < key;
            }
            if (first && !bad) {
                const int64_t o = prp[r] + rank;
                pcol[o] = key;
                pval[o] = sum;
            }
        }
        // rows beyond L lanes, one after the other
        for (uint64_t lm = ballot(is_long && sub == 0); lm; lm &= lm - 1) {
            const int64_t q = r0 + (__ffsll((unsigned long long)lm) - 1) / L;
            const int64_t qb = rp[q];
            const int64_t qn = rp[q + 1] - qb;
            if (!FILL) longest = max(longest, (int)min(qn, (int64_t)INT32_MAX));
            if (qn + 1 > CAP) {
                if (l == 0) atomicOr(err, kErrLongRow);
                if (!FILL && l == 0) len[q] = 0;
                continue;
            }
            // a table of at least the row's entries, 4/3 of them up to CAP
            int H = kWave, lg = 6;
            while (H < CAP && 3 * H < 4 * ((int)qn + 1)) {
                H *= 2;
                lg++;
            }
            int *k = sk[wv];
            double *s2 = sv[wv];
            for (int i = l; i < H; i += kWave) {
                k[i] = kEmpty;
                if (FILL) s2[i] = 0.0;
            }
            double w = 0.0;
            bool hd = false;  // the diagonal is stored
            for (int64_t e0 = qb; e0 < qb + qn; e0 += kWave) {
                const bool at = e0 + l < qb + qn && col[min(e0 + l, qb + qn - 1)] == q;
                const uint64_t am = ballot(at);
                if (am) {
                    hd = true;
                    if (FILL) w = val[e0 + __ffsll((unsigned long long)am) - 1];
                    break;
                }
            }
            if (FILL) {
                if (mode == 1) w = fabs(w) + 1.0;
                if (w == 0.0) {
                    if (l == 0) atomicOr(err, kErrBadInput);
                    continue;
                }
                w = omega / w;
            }
            wave_sync();
            int nd = 0;
            for (int e = l; e < (int)qn + (hd ? 0 : 1); e += kWave) {
                const int ce = e < (int)qn ? col[qb + e] : (int)q;
                int fresh = 0;
                const int at = hash_insert(k, (unsigned)H - 1, 32 - lg, agg[ce], &fresh);
                nd += fresh;
                if (FILL) atomicAdd(s2 + at, -w * (e < (int)qn ? val[qb + e] : 0.0) + (ce == q ? 1.0 : 0.0));
            }
            wave_sync();
            if (!FILL) {
                for (int o = 32; o > 0; o >>= 1) nd += __shfl_xor(nd, o);
                if (l == 0) len[q] = nd;
            } else {
                const int n2 = compact_table<kWave, double>(k, s2, H, nullptr);
                const int64_t o = prp[q];
                for (int j = l; j < n2; j += kWave) {
                    const int rank = key_rank(k, n2, k[j]);
                    pcol[o + rank] = k[j];
                    pval[o + rank] = s2[j];
                }
            }
            wave_sync();
        }
    }
    if (!FILL && maxlen && l == 0 && longest > __hip_atomic_load(maxlen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(maxlen, longest);
}

static unsigned grid1(int64_t n, int threads = 256)
{
    int64_t b = (n + threads - 1) / threads;
    if (b > 65536) b = 65536;
    return (unsigned)(b < 1 ? 1 : b);
}

void launch_col_count(const int32_t *col, int64_t nnz, int32_t *cnt, hipStream_t st)
{
    if (nnz > 0) hipLaunchKernelGGL(k_col_count, dim3(grid1(nnz)), dim3(256), 0, st, col, nnz, cnt);
}

void launch_transpose_scatter(const int64_t *rp, const int32_t *col, const void *val, bool f32, int64_t M,
                              int64_t nnz, const int64_t *trp, int32_t *cursor, int32_t *tcol, void *tval,
                              int32_t *tsrc, hipStream_t st)
{
    if (M == 0) return;
    // every entry waits for a returning atomic: rows of four entries take four
    // lanes (1.5e6 entries: 72 us with one lane per row, 28 with four); longer
    // rows stay at four entries per lane (rows of 9 and 70: 19 and 37 us, a
    // lane per entry 62 and 39: more of the counters' rows are hit at once)
    const int L = std::max(lanes_for(M, nnz), nnz >= 3 * M ? 4 : 1);
    const unsigned g = grid1(M, 256 / L);
    if (f32) {
        const float *v = static_cast<const float *>(val);
        float *tv = static_cast<float *>(tval);
        switch (L) {
        case 1: hipLaunchKernelGGL((k_transpose_scatter<float, 1>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 2: hipLaunchKernelGGL((k_transpose_scatter<float, 2>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 4: hipLaunchKernelGGL((k_transpose_scatter<float, 4>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 8: hipLaunchKernelGGL((k_transpose_scatter<float, 8>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 16: hipLaunchKernelGGL((k_transpose_scatter<float, 16>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 32: hipLaunchKernelGGL((k_transpose_scatter<float, 32>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        default: hipLaunchKernelGGL((k_transpose_scatter<float, 64>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        }
    } else {
        const double *v = static_cast<const double *>(val);
        double *tv = static_cast<double *>(tval);
        switch (L) {
        case 1: hipLaunchKernelGGL((k_transpose_scatter<double, 1>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 2: hipLaunchKernelGGL((k_transpose_scatter<double, 2>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 4: hipLaunchKernelGGL((k_transpose_scatter<double, 4>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 8: hipLaunchKernelGGL((k_transpose_scatter<double, 8>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 16: hipLaunchKernelGGL((k_transpose_scatter<double, 16>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        case 32: hipLaunchKernelGGL((k_transpose_scatter<double, 32>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        default: hipLaunchKernelGGL((k_transpose_scatter<double, 64>), dim3(g), dim3(256), 0, st, rp, col, v, M, trp, cursor, tcol, tv, tsrc); break;
        }
    }
}

void launch_sort_rows(const int64_t *rp, int64_t M, const int32_t *icol, const void *ival, const int32_t *isrc,
                      bool f32, int32_t *ocol, void *oval, int32_t *osrc, hipStream_t st)
{
    if (M == 0) return;
    const unsigned g = grid1(M, 4);
    if (f32)
        hipLaunchKernelGGL(k_sort_rows<float>, dim3(g), dim3(256), 0, st, rp, M, icol,
                           static_cast<const float *>(ival), isrc, ocol, static_cast<float *>(oval), osrc);
    else
        hipLaunchKernelGGL(k_sort_rows<double>, dim3(g), dim3(256), 0, st, rp, M, icol,
                           static_cast<const double *>(ival), isrc, ocol, static_cast<double *>(oval), osrc);
}

void launch_gather_vals(const void *src, const int32_t *perm, int64_t n, bool f32, void *out, hipStream_t st)
{
    if (n == 0) return;
    if (f32)
        hipLaunchKernelGGL(k_gather_vals<float>, dim3(grid1(n)), dim3(256), 0, st, static_cast<const float *>(src),
                           perm, n, static_cast<float *>(out));
    else
        hipLaunchKernelGGL(k_gather_vals<double>, dim3(grid1(n)), dim3(256), 0, st,
                           static_cast<const double *>(src), perm, n, static_cast<double *>(out));
}

void launch_sa_count(const int64_t *rp, const int32_t *col, int64_t M, int64_t nnz, int32_t *len, hipStream_t st)
{
    if (M == 0) return;
    const int L = lanes_for(M, nnz);
    SP3MM_BY_LANES(k_sa_count, dim3(grid1(M, 256 / L)), dim3(256), 0, st, rp, col, M, len)
}

void launch_sa_fill(const int64_t *rp, const int32_t *col, const double *val, int64_t M, int64_t nnz, double omega,
                    int mode, const int64_t *srp, int32_t *scol, double *sval, int *err, hipStream_t st)
{
    if (M == 0) return;
    const int L = lanes_for(M, nnz);
    SP3MM_BY_LANES(k_sa_fill, dim3(grid1(M, 256 / L)), dim3(256), 0, st, rp, col, val, M, omega, mode, srp, scol,
                   sval, err)
}

void launch_p0_fill(const int64_t *agg, int64_t M, int64_t nagg, int64_t *rp, int32_t *rp32, int32_t *col,
                    double *val, int *err, hipStream_t st)
{
    hipLaunchKernelGGL(k_p0_fill, dim3(grid1(M + 1)), dim3(256), 0, st, agg, M, nagg, rp, rp32, col, val, err);
}

void launch_agg_narrow(const int64_t *agg, int64_t M, int64_t nagg, int32_t *out, int *err, hipStream_t st)
{
    if (M > 0) hipLaunchKernelGGL(k_agg_narrow, dim3(grid1(M)), dim3(256), 0, st, agg, M, nagg, out, err);
}

// lanes by the mean row (a 7-point row and a missing diagonal fit 8 lanes;
// operators of longer rows run a wavefront per row); tables for the longest
// row when it is known (four of 1024 slots leave 12 wavefronts per CU: second
// level of a 96^3 hierarchy, 110,592 rows of 33, 125 us against 59)
void launch_sa_rows(bool fill, const int64_t *rp, const int32_t *col, const double *val, const int32_t *agg, int64_t M,
                    int64_t nnz, double omega, int mode, const int64_t *prp, int32_t *len, int32_t *pcol,
                    double *pval, int *maxlen, int longest, int *err, hipStream_t st)
{
    if (M == 0) return;
    const double avg = (double)nnz / (double)M;
    const int L = avg <= 8 ? 8 : kWave;
    const unsigned g = grid1(M, 4 * (kWave / L));
#define SP3MM_SA_ROWS(LL, CC)                                                                                      \
    do {                                                                                                           \
        if (fill)                                                                                                  \
            hipLaunchKernelGGL((k_sa_rows<LL, CC, true>), dim3(g), dim3(256), 0, st, rp, col, val, agg, M, omega,  \
                               mode, prp, len, pcol, pval, maxlen, err);                                                  \
        else                                                                                                       \
            hipLaunchKernelGGL((k_sa_rows<LL, CC, false>), dim3(g), dim3(256), 0, st, rp, col, val, agg, M, omega, \
                               mode, prp, len, pcol, pval, maxlen, err);                                                  \
    } while (0)
    if (L == 8) SP3MM_SA_ROWS(8, 128);
    else if (longest < 128) SP3MM_SA_ROWS(64, 128);
    else if (longest < 512) SP3MM_SA_ROWS(64, 512);
    else SP3MM_SA_ROWS(64, 1024);
#undef SP3MM_SA_ROWS
}

}  // namespace sp3mm

namespace sp3mm {

// ---------------------------------------------------------------------------
// consumers of a level: y = alpha A x + beta y, and damped Jacobi sweeps
// ---------------------------------------------------------------------------
// y = alpha A x + beta z (z may be y; with beta == 0 z is not read).
// L lanes per row (L a power of two up to 64), partial sums reduced by shuffles
template <int L>
__global__ void __launch_bounds__(256) k_spmv(const int64_t *__restrict__ rp, const int32_t *__restrict__ col,
                                               const double *__restrict__ val, int64_t M,
                                               const double *__restrict__ x, const double *z, double *y,
                                               double alpha, double beta)
{
    const int sub = threadIdx.x & (L - 1);
    const int64_t stride = (int64_t)gridDim.x * (blockDim.x / L);
    for (int64_t r = (int64_t)blockIdx.x * (blockDim.x / L) + threadIdx.x / L; r < M; r += stride) {
        double s = 0.0;
        for (int64_t e = rp[r] + sub; e < rp[r + 1]; e += L) s += val[e] * x[col[e]];
        for (int o = L / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (sub == 0) y[r] = alpha * s + (beta != 0.0 ? beta * z[r] : 0.0);
    }
}

// y = alpha x + beta y; a zero coefficient skips the read of its vector
__global__ void __launch_bounds__(256) k_axpby(int64_t n, double alpha, const double *x, double beta, double *y)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = (alpha != 0.0 ? alpha * x[i] : 0.0) + (beta != 0.0 ? beta * y[i] : 0.0);
}

// Dot product in two launches with a fixed summation order (the result does
// not depend on scheduling): kDotBlocks partial sums, then one block adds them.
constexpr int kDotBlocks = 1024;
__global__ void __launch_bounds__(256) k_dot_partial(int64_t n, const double *__restrict__ x,
                                                      const double *__restrict__ y, double *__restrict__ part)
{
    __shared__ double red[256 / kWave];
    double s = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        s += x[i] * y[i];
    for (int o = kWave / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane() == 0) red[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < 256 / kWave; w++) t += red[w];
        part[blockIdx.x] = t;
    }
}

__global__ void __launch_bounds__(256) k_dot_final(const double *__restrict__ part, int nb, double *__restrict__ out)
{
    __shared__ double red[256 / kWave];
    double s = 0.0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) s += part[i];
    for (int o = kWave / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane() == 0) red[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < 256 / kWave; w++) t += red[w];
        *out = t;
    }
}

// xo = xi + omega (b - A xi) / a_ii
template <int L>
__global__ void __launch_bounds__(256) k_jacobi(const int64_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                 const double *__restrict__ val, int64_t M,
                                                 const double *__restrict__ b, const double *__restrict__ xi,
                                                 double *__restrict__ xo, double omega, int *__restrict__ err)
{
    const int sub = threadIdx.x & (L - 1);
    const int64_t stride = (int64_t)gridDim.x * (blockDim.x / L);
    for (int64_t r = (int64_t)blockIdx.x * (blockDim.x / L) + threadIdx.x / L; r < M; r += stride) {
        double s = 0.0, d = 0.0;
        for (int64_t e = rp[r] + sub; e < rp[r + 1]; e += L) {
            const int c = col[e];
            s += val[e] * xi[c];
            if (c == r) d = val[e];
        }
        for (int o = L / 2; o > 0; o >>= 1) {
            s += __shfl_xor(s, o);
            d += __shfl_xor(d, o);
        }
        if (sub == 0) {
            if (d == 0.0) atomicOr(err, kErrBadInput);
            else xo[r] = xi[r] + omega * (b[r] - s) / d;
        }
    }
}

// The first sweep from x = 0: xo = omega b / a_ii.  Only the diagonal is read
// (found by bisection in the row's sorted columns), not the row: 4.8 us of
// clearing x and 34 us of sweep against 23 us on 262,144 rows of 32 entries,
// 4.5 + 23 against 7 on 32,768 rows of 180.
__global__ void __launch_bounds__(256) k_jacobi_zero(const int64_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                      const double *__restrict__ val, int64_t M,
                                                      const double *__restrict__ b, double *__restrict__ xo,
                                                      double omega, int *__restrict__ err)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= M) return;
    const int64_t e1 = rp[r + 1];
    int64_t lo = rp[r], n = e1 - lo;
    const double br = b[r];
    while (n > 0) {  // the first column not below r
        const int64_t h = n / 2;
        if (col[lo + h] < r) {
            lo += h + 1;
            n -= h + 1;
        } else {
            n = h;
        }
    }
    const double d = lo < e1 && col[lo] == r ? val[lo] : 0.0;
    if (d == 0.0) atomicOr(err, kErrBadInput);
    else xo[r] = 0.0 + omega * (br - 0.0) / d;
}

// All `sweeps` sweeps of a small system in one workgroup, with the matrix,
// b and both x vectors staged in LDS once (a coarsest-level solve is a few
// kilobytes; a launch per sweep would cost more than the sweep).  Rows are
// split over L-lane groups as in k_jacobi, with the same per-row summation
// order, so the result equals `sweeps` launches of k_jacobi.
constexpr int kSmallRows = 2048;
template <int L>
__global__ void __launch_bounds__(1024) k_jacobi_small(const int64_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                        const double *__restrict__ val, int M, int nnz,
                                                        const double *__restrict__ b, double *__restrict__ x,
                                                        double omega, int sweeps, int *__restrict__ err)
{
    extern __shared__ double lds[];
    double *sv = lds;                   // nnz values
    double *sb = sv + nnz;              // M
    double *xs0 = sb + M, *xs1 = xs0 + M;
    int *sc = reinterpret_cast<int *>(xs1 + M);  // nnz columns
    int *sr = sc + nnz;                 // M + 1 offsets from rp[0]
    const int64_t base = rp[0];
    for (int i = threadIdx.x; i < nnz; i += blockDim.x) {
        sv[i] = val[base + i];
        sc[i] = col[base + i];
    }
    for (int i = threadIdx.x; i <= M; i += blockDim.x) sr[i] = (int)(rp[i] - base);
    for (int i = threadIdx.x; i < M; i += blockDim.x) {
        sb[i] = b[i];
        xs0[i] = x[i];
    }
    __syncthreads();
    const int sub = threadIdx.x & (L - 1);
    double *xi = xs0, *xo = xs1;
    for (int k = 0; k < sweeps; k++) {
        for (int r = threadIdx.x / L; r < M; r += blockDim.x / L) {
            double s = 0.0, d = 0.0;
            for (int e = sr[r] + sub; e < sr[r + 1]; e += L) {
                const int c = sc[e];
                s += sv[e] * xi[c];
                if (c == r) d = sv[e];
            }
            for (int o = L / 2; o > 0; o >>= 1) {
                s += __shfl_xor(s, o);
                d += __shfl_xor(d, o);
            }
            if (sub == 0) {
                if (d == 0.0) atomicOr(err, kErrBadInput);
                else xo[r] = xi[r] + omega * (sb[r] - s) / d;
            }
        }
        __syncthreads();
        double *t = xi;
        xi = xo;
        xo = t;
    }
    for (int i = threadIdx.x; i < M; i += blockDim.x) x[i] = xi[i];
}

static size_t jacobi_small_lds(int64_t M, int64_t nnz) { return (size_t)nnz * 12 + (size_t)M * 24 + (size_t)(M + 1) * 4; }

// All `sweeps` sweeps of a medium system (M up to kGridRows rows, too large for
// one workgroup's LDS) in one launch: a launch per sweep costs 6.6 us on a
// 512-row operator of 300 entries per row, several times the sweep itself.
// Every L-lane group keeps one row in registers (kGridRegs entries per lane,
// what is beyond them is read again in every sweep) for all sweeps; a
// workgroup's rows see the whole x of the sweep in LDS.  Sweep k writes its x
// to buffer k, which starts filled with a signalling NaN no arithmetic
// produces (hardware quiets NaN results), and the next sweep polls every entry
// until it is there: the data is its own flag, so a sweep costs one store
// reaching one load (agent scope) and no barrier across workgroups.  The last
// sweep writes x, behind the polls of the sweep before it, which wait for every
// workgroup's read of x: a launch takes two sweeps at least (jacobi_chunk).
// The sweeps need their workgroups (at most 256 of 512 lanes and 34 KB of LDS)
// on the chip together; the launcher takes this form only where the stream's
// CUs hold them all (jacobi_grid_resident).  Other work can still keep some
// from starting, so a poll that does not see its entry within kGridSpins loads
// (some 50 ms) gives up, every other one then does, too, and k_jacobi_redo
// behind it runs all the sweeps in one workgroup from the copy of x that
// k_grid_empty took (otherwise it ends at once; counting the workgroups that
// end, to redo the sweeps in the last one, cost 7 to 30 us a launch in fences).
// Rows are summed in k_jacobi's order either way (equal results).  50 sweeps in a V-cycle's graph,
// 512 rows: 330 -> 163 us; called alone 267 -> 183, 1,000 rows 255 -> 223.
// Two or four rows per group (fewer workgroups polling): 192 to 525 us.
constexpr int kGridRegs = 8;
constexpr unsigned long long kGridEmpty = 0x7FF7A5A57FF7A5A5ull;
constexpr int kGridSpins = 1 << 16;
// behind the sweeps' buffers: x as it was, and the word of a poll that gave up
constexpr size_t kGridCopy = (size_t)(kGridSweeps - 1) * kGridRows, kGridWords = kGridCopy + kGridRows + 1;

template <int L>
__global__ void __launch_bounds__(kGridThreads) k_jacobi_grid(const int64_t *__restrict__ rp,
                                                              const int32_t *__restrict__ col,
                                                              const double *__restrict__ val, int M,
                                                              const double *__restrict__ b, double *x,
                                                              unsigned long long *buf, double omega, int sweeps,
                                                              bool from_zero, int spins, int *__restrict__ err)
{
    __shared__ double xs[2][kGridRows];
    __shared__ int dead;
    int *gave_up = reinterpret_cast<int *>(buf + kGridCopy + kGridRows);
    const int t = threadIdx.x, sub = t & (L - 1);
    const int r = blockIdx.x * (kGridThreads / L) + t / L;
    const bool act = r < M;
    const int64_t e0 = act ? rp[r] : 0;
    const int64_t e1 = act ? rp[r + 1] : 0;
    // this lane's first entries of the row, its right-hand side and diagonal
    int c[kGridRegs];
    double v[kGridRegs];
    double d = 0.0;
#pragma unroll
    for (int u = 0; u < kGridRegs; u++) {
        const int64_t e = e0 + sub + (int64_t)u * L;
        c[u] = e < e1 ? col[e] : -1;
        v[u] = e < e1 ? val[e] : 0.0;
        if (c[u] == r) d = v[u];
    }
    for (int64_t e = e0 + sub + (int64_t)kGridRegs * L; e < e1; e += L)
        if (col[e] == r) d = val[e];
    for (int o = L / 2; o > 0; o >>= 1) d += __shfl_xor(d, o);
    const double br = act ? b[r] : 0.0;
    if (act && sub == 0 && d == 0.0) atomicOr(err, kErrBadInput);
    if (t == 0) dead = 0;
    for (int i = t; i < M; i += kGridThreads) xs[0][i] = from_zero ? 0.0 : x[i];
    __syncthreads();
    for (int k = 0; k < sweeps; k++) {
        const double *xi = xs[k & 1];
        double s = 0.0;
#pragma unroll
        for (int u = 0; u < kGridRegs; u++)
            if (c[u] >= 0) s += v[u] * xi[c[u]];
        for (int64_t e = e0 + sub + (int64_t)kGridRegs * L; e < e1; e += L) s += val[e] * xi[col[e]];
        for (int o = L / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
        const bool last = k + 1 == sweeps;
        if (act && sub == 0) {
            const double xn = d == 0.0 ? xi[r] : xi[r] + omega * (br - s) / d;
            if (last) x[r] = xn;
            else
                __hip_atomic_store(buf + (int64_t)k * M + r, (unsigned long long)__double_as_longlong(xn),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (last) break;
        // the other buffer of x: nobody reads it any more (sweep k - 1 ended
        // at the barrier below)
        double *xo = xs[(k + 1) & 1];
        for (int i = t; i < M; i += kGridThreads) {
            unsigned long long w = kGridEmpty;
            for (int n = 0; n < spins; n++) {
                w = __hip_atomic_load(buf + (int64_t)k * M + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (w != kGridEmpty) break;
                if ((n & 1023) == 1023 && __hip_atomic_load(gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
                __builtin_amdgcn_s_sleep(1);
            }
            if (w == kGridEmpty) dead = 1;
            xo[i] = __longlong_as_double((long long)w);
        }
        __syncthreads();
        if (dead) {  // uniform: written before the barrier
            if (t == 0) __hip_atomic_store(gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
    }
}

// the sweeps of a k_jacobi_grid that gave up, in one workgroup
template <int L>
__global__ void __launch_bounds__(1024) k_jacobi_redo(const int64_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                       const double *__restrict__ val, int M,
                                                       const double *__restrict__ b, double *__restrict__ x,
                                                       const unsigned long long *__restrict__ buf, double omega,
                                                       int sweeps, bool from_zero)
{
    __shared__ double xs[2][kGridRows];
    if (*reinterpret_cast<const int *>(buf + kGridCopy + kGridRows) == 0) return;
    const int t = threadIdx.x, sub = t & (L - 1);
    for (int i = t; i < M; i += 1024)
        xs[0][i] = from_zero ? 0.0 : __longlong_as_double((long long)buf[kGridCopy + i]);
    __syncthreads();
    for (int k = 0; k < sweeps; k++) {
        const double *xi = xs[k & 1];
        double *xo = xs[(k + 1) & 1];
        for (int q = t / L; q < M; q += 1024 / L) {
            double s = 0.0, dq = 0.0;
            for (int64_t e = rp[q] + sub; e < rp[q + 1]; e += L) {
                const int ce = col[e];
                s += val[e] * xi[ce];
                if (ce == q) dq = val[e];
            }
            for (int o = L / 2; o > 0; o >>= 1) {
                s += __shfl_xor(s, o);
                dq += __shfl_xor(dq, o);
            }
            if (sub == 0) xo[q] = dq == 0.0 ? xi[q] : xi[q] + omega * (b[q] - s) / dq;
        }
        __syncthreads();
    }
    for (int i = t; i < M; i += 1024) x[i] = xs[sweeps & 1][i];
}

__global__ void k_grid_empty(unsigned long long *buf, int64_t n, const double *__restrict__ x, int M)
{
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = i0; i < n; i += step) buf[i] = kGridEmpty;
    for (int64_t i = i0; i < M; i += step) buf[kGridCopy + i] = (unsigned long long)__double_as_longlong(x[i]);
    if (i0 == 0) buf[kGridCopy + kGridRows] = 0;
}

size_t jacobi_grid_bytes() { return kGridWords * 8; }

// workgroups of k_jacobi_grid<L> that one CU holds, 0 if unknown
static int grid_per_cu(int L)
{
    static std::atomic<int> known[7];  // by log2 of L: the count, plus one
    std::atomic<int> &k = known[ilog2((unsigned)L)];
    int n = k.load(std::memory_order_relaxed) - 1;
    if (n >= 0) return n;
    auto occ = [&](auto fn) { return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, kGridThreads, 0); };
    const hipError_t e = L == 1    ? occ(k_jacobi_grid<1>)
                         : L == 2  ? occ(k_jacobi_grid<2>)
                         : L == 4  ? occ(k_jacobi_grid<4>)
                         : L == 8  ? occ(k_jacobi_grid<8>)
                         : L == 16 ? occ(k_jacobi_grid<16>)
                         : L == 32 ? occ(k_jacobi_grid<32>)
                                   : occ(k_jacobi_grid<64>);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    k.store(n + 1, std::memory_order_relaxed);
    return n;
}

// Lanes per row: the smallest power of two (at most 64) not below the mean
// row length divided by SP3MM_SPMV_ROW_DIV (default 4: about four entries
// per lane, measured best on SA hierarchies of 7-point operators).
void launch_spmv(const int64_t *rp, const int32_t *col, const double *val, int64_t M, int64_t nnz, const double *x,
                 const double *z, double *y, double alpha, double beta, hipStream_t st)
{
    if (M == 0) return;
    const int L = lanes_for(M, nnz);
    const unsigned g = grid1(M, 256 / L);
    SP3MM_BY_LANES(k_spmv, dim3(g), dim3(256), 0, st, rp, col, val, M, x, z, y, alpha, beta)
}

void launch_axpby(int64_t n, double alpha, const double *x, double beta, double *y, hipStream_t st)
{
    if (n == 0) return;
    hipLaunchKernelGGL(k_axpby, dim3(grid1(n, 256)), dim3(256), 0, st, n, alpha, x, beta, y);
}

void launch_dot(int64_t n, const double *x, const double *y, double *part, double *out, hipStream_t st)
{
    const unsigned nb = n ? (unsigned)std::min<int64_t>((n + 255) / 256, kDotBlocks) : 1;
    hipLaunchKernelGGL(k_dot_partial, dim3(nb), dim3(256), 0, st, n, x, y, part);
    hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(256), 0, st, part, (int)nb, out);
}

int dot_parts() { return kDotBlocks; }

bool launch_jacobi_small(const int64_t *rp, const int32_t *col, const double *val, int64_t M, int64_t nnz,
                         const double *b, double *x, double omega, int sweeps, int *err, size_t max_lds,
                         hipStream_t st)
{
    if (!jacobi_small_fits(M, nnz, max_lds)) return false;
    const int L = lanes_for(M, nnz);
    const size_t lds = jacobi_small_lds(M, nnz);
    SP3MM_BY_LANES(k_jacobi_small, dim3(1), dim3(1024), lds, st, rp, col, val, (int)M, (int)nnz, b, x, omega,
                   sweeps, err)
    return true;
}

void launch_jacobi_zero(const int64_t *rp, const int32_t *col, const double *val, int64_t M, const double *b,
                        double *xo, double omega, int *err, hipStream_t st)
{
    if (M > 0)
        hipLaunchKernelGGL(k_jacobi_zero, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, st, rp, col, val, M, b, xo,
                           omega, err);
}

bool jacobi_small_fits(int64_t M, int64_t nnz, size_t max_lds)
{
    return M > 0 && M <= kSmallRows && jacobi_small_lds(M, nnz) <= max_lds;
}

// Launches nothing and returns false when a launch per sweep is as good: fewer
// than kGridMin sweeps (clearing the buffers is a launch of its own), or more
// workgroups than the `cus` CUs at hand hold together.  SP3MM_GRID_SPINS: loads
// after which a poll gives up.
bool launch_jacobi_grid(const int64_t *rp, const int32_t *col, const double *val, int64_t M, int64_t nnz,
                        const double *b, double *x, void *buf, double omega, int sweeps, bool from_zero, int *err,
                        int cus, hipStream_t st)
{
    constexpr int kGridMin = 4;
    if (M <= 0 || sweeps < kGridMin || !buf) return false;
    const int L = lanes_for(M, nnz);
    if (M > kGridRows || !jacobi_grid_resident((int)M, L, grid_per_cu(L), cus)) return false;
    const char *env = getenv("SP3MM_GRID_SPINS");
    const int spins = env ? std::max(0, atoi(env)) : kGridSpins;
    auto *w = static_cast<unsigned long long *>(buf);
    for (int k = 0, n; k < sweeps; k += n) {
        n = jacobi_chunk(sweeps - k);
        hipLaunchKernelGGL(k_grid_empty, dim3(grid1((n - 1) * M)), dim3(256), 0, st, w, (int64_t)(n - 1) * M, x,
                           from_zero && k == 0 ? 0 : (int)M);
        const unsigned g = grid1(M, kGridThreads / L);
        SP3MM_BY_LANES(k_jacobi_grid, dim3(g), dim3(kGridThreads), 0, st, rp, col, val, (int)M, b, x, w, omega, n,
                       from_zero && k == 0, spins, err)
        SP3MM_BY_LANES(k_jacobi_redo, dim3(1), dim3(1024), 0, st, rp, col, val, (int)M, b, x, w, omega, n,
                       from_zero && k == 0)
    }
    return true;
}

void launch_jacobi(const int64_t *rp, const int32_t *col, const double *val, int64_t M, int64_t nnz, const double *b,
                   const double *xi, double *xo, double omega, int *err, hipStream_t st)
{
    if (M == 0) return;
    const int L = lanes_for(M, nnz);
    const unsigned g = grid1(M, 256 / L);
    SP3MM_BY_LANES(k_jacobi, dim3(g), dim3(256), 0, st, rp, col, val, M, b, xi, xo, omega, err)
}
#undef SP3MM_BY_LANES

// ---------------------------------------------------------------------------
// replay guards of a hierarchy plan
// ---------------------------------------------------------------------------
// 64-bit finaliser of the splitmix64 generator (Steele, Lea, Flood 2014)
__device__ __forceinline__ uint64_t mix64(uint64_t x)
{
    x ^= x >> 30;
    x *= 0xbf58476d1ce4e5b9ull;
    x ^= x >> 27;
    x *= 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}

// out += sum over the M+1 offsets and nnz columns of mix64(mix64(position) +
// entry): an order-sensitive fingerprint of a CSR pattern (wrapping sums, so
// the result does not depend on the schedule).
// One addition per workgroup, four loads in flight per lane: additions to one
// word take 15 ns each, so one per wavefront of 1024 workgroups of 256 lanes
// bounded it (96^3 7-point operator, 32 MB: 62 us, now 24).  State: out[0] the sum,
// out[1] the workgroups that have added theirs, both zero before and after;
// the last one takes the sum and writes it to dst.
constexpr int kFpThreads = 1024;
__global__ void __launch_bounds__(kFpThreads) k_fingerprint(const int64_t *__restrict__ rp, int64_t M,
                                                            const int32_t *__restrict__ col, int64_t nnz,
                                                            unsigned long long *out, unsigned long long *dst)
{
    __shared__ unsigned long long sh[kFpThreads / 64];
    const int64_t stride = (int64_t)gridDim.x * kFpThreads;
    const int64_t t0 = (int64_t)blockIdx.x * kFpThreads + threadIdx.x;
    unsigned long long acc = 0;
    auto add = [&](const auto *a, int64_t n, uint64_t first) {
        int64_t i = t0;
        for (; i + 3 * stride < n; i += 4 * stride) {
            uint64_t v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) v[u] = (uint64_t)a[i + u * stride];
#pragma unroll
            for (int u = 0; u < 4; u++) acc += mix64(mix64(first + (uint64_t)(i + u * stride)) + v[u]);
        }
        for (; i < n; i += stride) acc += mix64(mix64(first + (uint64_t)i) + (uint64_t)a[i]);
    };
    add(rp, M + 1, 0);
    add(reinterpret_cast<const uint32_t *>(col), nnz, (uint64_t)M + 1);
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane() == 0) sh[threadIdx.x / 64] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long s = 0;
        for (int w = 0; w < kFpThreads / 64; w++) s += sh[w];
        atomicAdd(out, s);
        __threadfence();
        if (atomicAdd(out + 1, 1ull) == gridDim.x - 1) {
            __threadfence();
            *dst = atomicExch(out, 0ull);
            atomicExch(out + 1, 0ull);
        }
    }
}

void launch_fingerprint(const int64_t *rp, int64_t M, const int32_t *col, int64_t nnz, unsigned long long *out,
                        unsigned long long *dst, hipStream_t st)
{
    const unsigned g = (unsigned)std::min<int64_t>((M + 1 + nnz + kFpThreads - 1) / kFpThreads, 512);
    hipLaunchKernelGGL(k_fingerprint, dim3(g), dim3(kFpThreads), 0, st, rp, M, col, nnz, out, dst);
}

// *out = bitwise OR of the n words *words[i]
__global__ void k_or_words(const int *const *words, int n, int *out)
{
    int v = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) v |= *words[i];
    for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o);
    if (threadIdx.x == 0) *out = v;
}

void launch_or_words(const int *const *words, int n, int *out, hipStream_t st)
{
    hipLaunchKernelGGL(k_or_words, dim3(1), dim3(64), 0, st, words, n, out);
}

// every plan's error word, cleared by one launch (a launch per word costs 4.6
// us each in a replay)
__global__ void k_clear_words(int *const *words, int n)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) *words[i] = 0;
}

void launch_clear_words(int *const *words, int n, hipStream_t st)
{
    hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(64), 0, st, words, n);
}

}  // namespace sp3mm
