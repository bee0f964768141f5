// Shared quadrature nodes of the three-centre passes: one node list per aux centre instead of
// twenty nodes per aux function.
//
// With s = t^2 b / (b + t^2), node t of an aux function of exponent b at R contributes w_t
// (b + t^2)^(-3/2) g(s), where g(s) = Pn(s)^(-1/2) exp(-s Qn/Pn) depends on the pair and on R only
// (dfj.hip). So the functions at one centre (the exponent scales of a product aux) ask for the same
// g at 20 nb points, most of them redundant: below t^2 ~ b the scales' nodes nearly coincide
// (s ~ t^2), above it each function's nodes crowd below s = b. g is the pair's Gaussian averaged
// over exp(-s u), u = |R - r|^2, with a positive weight (it is the integral of the product Gaussian
// against exp(-s |R - r|^2)), so any node list that reproduces
//     K_b(u) = sum_t w_t (b + t^2)^(-3/2) exp(-s_t u)
// to a relative error e at every u in reach reproduces every (P|a) to e.
// k_node_sets picks such a list for each centre: of the centre's 20 nb nodes, the columns that
// Gaussian elimination with complete pivoting takes from the matrix exp(-s_j u_i) w_j / min_b
// K_b(u_i), until what is left is below kSetTol; the others' weights are spread over those taken
// (an interpolative decomposition: the coefficients stay of order one). 40 to 60 nodes replace the
// 80 of four scales, 27 to 40 the 40 of two. Against 80-bit arithmetic the lists reproduce (P|a) of
// random pairs (exponents from 0.03 to 64, eigenvalues from 0.02 to 60, systems of 0.01 to 40 Bohr) to
// 2e-16 in the median and 7e-15 at most. A derivative has no bound of its own: 1e-15 of its terms'
// magnitudes in the median, 3e-13 at most within 3 Bohr and 2e-12 at 20, where it is small beside
// (P|a) itself.
// Every product Gaussian is, in turn, an average of isotropic Gaussians of exponent l >= its largest
// eigenvalue, so the matrix is formed for those (s -> s l / (l + s), weights (l / (l + s))^(3/2), u the
// squared distance to their centres), which takes a node or two fewer where b > l.
#include <algorithm>

#include "common.h"
#include "internal.h"

namespace gsdft {

namespace {

constexpr int kSetRows = 96;          // points in u
constexpr int kSetThreads = 320;
constexpr double kSetTol = 4e-15;
constexpr double kSetFirst = 2.0;     // u grid: u_i = c (e^(a i) - 1), c = kSetFirst / largest s
// The u grid ends kSetTail^(1/2) widths past the far corner of the pairs' centres, where the widest
// pair's Gaussian has fallen to e^-kSetTail; the lists extrapolate beyond. Over 1200 random clusters
// within 3 Bohr, splats up to fifty times as long as thick, (P|a) erred by up to 1.1e-13 with 8 and
// by 3e-15 to 6e-15 with 10 to 60, its derivatives by 7e-12 and by 2e-13 to 3e-13 of their terms, for
// 27 nodes in the mean with 8, 28 with 10, 29.5 with 16 and 32 with 36. The water octamer's step
// takes 11.20 ms with 16, 11.00 with 8; C20H42's 90.3 and 89.1.
constexpr double kSetTail = 16.0;
constexpr int kBoxBlocks = 256;

template <int kCtrl>
__device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t a = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)a, kCtrl, 0xf, 0xf,
                                                              false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(a >> 32), kCtrl,
                                                              0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The wave's largest value in every lane: lanes i ^ 1, i ^ 2, then the mirrors of 8 and 16 (each
// half of a mirror already agrees), then rows of 16 and 32 through readlane.
__device__ __forceinline__ double wave_max(double v) {
    v = __builtin_fmax(v, dpp_f64<0xb1>(v));
    v = __builtin_fmax(v, dpp_f64<0x4e>(v));
    v = __builtin_fmax(v, dpp_f64<0x141>(v));
    v = __builtin_fmax(v, dpp_f64<0x140>(v));
    return __builtin_fmax(__builtin_fmax(readlane_f64(v, 0), readlane_f64(v, 16)),
                          __builtin_fmax(readlane_f64(v, 32), readlane_f64(v, 48)));
}

// Largest |P| coordinates and widths of the pair records: per block -min P (3), max P (3),
// max I2/I3 (at least 1 / the smallest eigenvalue, the squared width), max I1 (at least the
// largest eigenvalue).
__global__ __launch_bounds__(256) void k_pair_box(int64_t n, const double* __restrict__ rec,
                                                  int rec_stride, double* __restrict__ part) {
    __shared__ double red[4][8];
    double v[8];
    for (int c = 0; c < 6; ++c) v[c] = -1e300;
    v[6] = v[7] = 0.0;
    for (int64_t a = blockIdx.x * (int64_t)256 + threadIdx.x; a < n;
         a += (int64_t)gridDim.x * 256) {
        const double* r = rec + (int64_t)rec_stride * a;
        for (int c = 0; c < 3; ++c) {
            v[c] = __builtin_fmax(v[c], -r[9 + c]);
            v[3 + c] = __builtin_fmax(v[3 + c], r[9 + c]);
        }
        v[6] = __builtin_fmax(v[6], r[1] / r[2]);
        v[7] = __builtin_fmax(v[7], r[0]);
    }
    for (int c = 0; c < 8; ++c) {
        const double x = wave_max(v[c]);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = x;
    }
    __syncthreads();
    if (threadIdx.x < 8) {
        const int c = threadIdx.x;
        part[8 * blockIdx.x + c] = __builtin_fmax(__builtin_fmax(red[0][c], red[1][c]),
                                                  __builtin_fmax(red[2][c], red[3][c]));
    }
}

__global__ __launch_bounds__(64) void k_pair_box_finish(int blocks, const double* __restrict__ part,
                                                        double* __restrict__ box) {
    for (int c = 0; c < 8; ++c) {
        double x = -1e300;
        for (int b = threadIdx.x; b < blocks; b += 64) x = __builtin_fmax(x, part[8 * b + c]);
        x = wave_max(x);
        if (threadIdx.x == 0) box[c] = x;
    }
}

// The double v with its low 13 mantissa bits replaced by an index: of two such keys the larger
// belongs to the larger value (ties within 2^-39 go by the index), so one maximum finds both.
__device__ __forceinline__ double pivot_key(double v, uint32_t index) {
    return __builtin_bit_cast(double, (__builtin_bit_cast(uint64_t, v) & ~0x1fffull) | index);
}

// One workgroup per group of up to NB aux functions that stand consecutively in slot order (the
// scales of one centre, kMaxSetScales at a time). Thread (column j, row class rg) holds the
// entries of column j in rows rg, rg + RG, ... in registers; a step finds the largest entry left
// (one key per lane, wave and workgroup maxima), publishes its row (kept in U, the pivot rows) and
// its column in LDS, and subtracts their product. With the columns taken in order, U = U11 T: the
// weights ask only for each function's sum over its twenty columns of T, so one wave per function
// solves U11 t = (sum of the function's columns of U), and the nodes go out in ascending s.
// Where the group's functions do not share a centre, an exponent is out of the range below or
// kMaxRank nodes are not enough, every function keeps its own twenty nodes in a sub-record.
// Bound by its serial steps (two barriers each, ~50 steps): 72 pivot rows keep the LDS at 50 KB, so
// three workgroups to a CU overlap them.
template <int NB>
__global__ __launch_bounds__(kSetThreads) void k_node_sets(
    int64_t N, int64_t G, int64_t per_centre, int64_t groups, int64_t stride,
    const double* __restrict__ beta,
    const double* __restrict__ kn, const double* __restrict__ R,
    const double* __restrict__ dgamma, const double* __restrict__ dscale, SetForm form,
    const double* __restrict__ box, NodeTable tb, double* __restrict__ out) {
    constexpr int kCols = kNodes * NB;
    constexpr int kMaxRank = NB == 4 ? 72 : kCols;      // pivot rows in LDS
    constexpr int RG = kSetThreads / kCols;           // row classes
    constexpr int RT = kSetRows / RG;                 // rows per thread
    static_assert(RG * RT == kSetRows && RG * kCols == kSetThreads && kCols * kSetRows <= 8192, "");
    constexpr int CH = RT % 4 == 0 ? 4 : 3;           // row classes per step of the K sums
    static_assert(RT % CH == 0, "");
    constexpr int kLd = kCols + 1;                    // odd: a column of U is free of conflicts
    constexpr int kStage = CH * kSetThreads;
    __shared__ double U[kMaxRank * kLd > kStage ? kMaxRank * kLd : kStage];
    __shared__ double pcol[kSetRows], kmin[kSetRows], us[kSetRows], cs[kCols], cw[kCols],
        rdiag[kMaxRank], wsum[kMaxRank][NB];
    __shared__ double wavekey[2][kSetThreads / 64];
    __shared__ int piv[kMaxRank];
    const int tid = threadIdx.x;
    const int64_t group = blockIdx.y * (int64_t)gridDim.x + blockIdx.x;
    if (group >= groups) return;                                       // workgroup-uniform
    int64_t slot0;
    const int nb = set_group(group, G, per_centre, &slot0);
    double* o = out + stride * group;
    // the functions of the group, and whether they can share nodes (workgroup-uniform)
    bool shared = true;
    const int64_t p0 = aux_of_slot(slot0, N, G);
    const double rc[3] = {R[3 * p0], R[3 * p0 + 1], R[3 * p0 + 2]};
    double bmax = 0.0, bmin = 1e300;
    for (int b = 0; b < nb; ++b) {
        const int64_t p = aux_of_slot(slot0 + b, N, G);
        shared = shared && beta[p] > 1e-100 && beta[p] < 1e100;
        for (int c = 0; c < 3; ++c)
            shared = shared && __builtin_bit_cast(uint64_t, R[3 * p + c]) ==
                                   __builtin_bit_cast(uint64_t, rc[c]);
        bmax = __builtin_fmax(bmax, beta[p]);
        bmin = __builtin_fmin(bmin, beta[p]);
    }
    const int col = tid % kCols, rg = tid / kCols, cb = col / kNodes, ct = col % kNodes;
    const bool real_col = cb < nb;
    double s = 1.0, wp = 0.0;
    if (real_col) {
        const double b = beta[aux_of_slot(slot0 + cb, N, G)], t2 = tb.t[ct] * tb.t[ct];
        s = t2 * b / (b + t2);
        wp = tb.w[ct] / ((b + t2) * sqrt(b + t2));
    }
    const double norm = kExpMinusHalf / kExpQuarticK;
    const int nd = set_node_doubles(NB, form);
    // node `at` of the list at y: s, and the weights w[b] of the functions
    auto put = [&](double* y, int at, double sn, const double w[NB]) {
        y += nd * at;
        const double wn = norm / sqrt(sn);
        y[0] = sn;
        if (form == kSetFold) {
            double x = 0.0;
            for (int b = 0; b < nb; ++b) {
                const int64_t p = aux_of_slot(slot0 + b, N, G);
                x += dgamma[p] * (dscale ? *dscale : 1.0) * kn[p] * w[b];
            }
            y[1] = wn * x;
            y[2] = sn * sn;
            y[3] = 1.0 / sn;
            return;
        }
        y[1] = 1.0 / sn;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const double k = form == kSetExchange && b < nb ? kn[aux_of_slot(slot0 + b, N, G)]
                                                            : 1.0;
            y[2 + b] = b < nb ? wn * w[b] * k : 0.0;
        }
        if (form == kSetExchange) {
            y[6] = sn * sn;
            y[7] = 0.0;
        }
    };
    int rank = 0;
    if (shared) {
        // reach: from R to the far corner of the pairs' centres, plus the tail of the widest
        const double lam = __builtin_fmin(__builtin_fmax(box[7], 1e-30), 1e30);
        double d2 = 0.0;
        for (int c = 0; c < 3; ++c) {
            const double d = __builtin_fmax(rc[c] + box[c], box[3 + c] - rc[c]);
            d2 += d * d;
        }
        const double reach = sqrt(d2) + sqrt(kSetTail * box[6]);
        const double c0 = kSetFirst * (lam + bmax) / (bmax * lam);
        double um = __builtin_fmax(__builtin_fmin(reach * reach, 1e12), 4.0 * c0);
        // the smallest s of the group; past s u = 600 every term has vanished
        const double t02 = tb.t[0] * tb.t[0];
        um = __builtin_fmin(um, 600.0 * (bmin + t02) / (t02 * bmin));
        if (tid < kSetRows)
            us[tid] = c0 * (exp_fast(log(um / c0 + 1.0) / (kSetRows - 1) * tid) - 1.0);
        if (rg == 0) {
            cs[col] = s;
            cw[col] = wp;
        }
        __syncthreads();
        const double f = lam / (lam + s);
        const double se = s * f;
        const double we = wp * f * sqrt(f);
        double a[RT];
        // entries, and 1 / min_b K_b(u_i) from the sums of each function's columns
#pragma unroll
        for (int i0 = 0; i0 < RT; i0 += CH) {
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                a[i0 + i] = we * exp_fast(-se * us[(i0 + i) * RG + rg]);
                U[(i * RG + rg) * kCols + col] = a[i0 + i];
            }
            __syncthreads();
            if (tid < CH * RG * NB) {          // one (row, function) per thread, NB threads a row
                const int r = tid / NB, b = tid % NB;
                double x = 0.0;
#pragma unroll
                for (int j = 0; j < kNodes; ++j) x += U[r * kCols + b * kNodes + j];
                x = b < nb ? x : 1e300;
#pragma unroll
                for (int off = 1; off < NB; off <<= 1)
                    x = __builtin_fmin(x, __shfl_xor(x, off, 64));
                if (b == 0) kmin[i0 * RG + r] = 1.0 / x;
            }
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < RT; ++i) a[i] *= kmin[i * RG + rg];
        for (;;) {
            double best = 0.0;
            int bi = 0;
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const double x = __builtin_fabs(a[i]);
                bi = x > best ? i : bi;
                best = __builtin_fmax(best, x);
            }
            const double wk = wave_max(pivot_key(best, (uint32_t)((bi * RG + rg) * kCols + col)));
            double* keys = wavekey[rank & 1];
            if ((tid & 63) == 0) keys[tid >> 6] = wk;
            __syncthreads();
            double key = keys[0];
#pragma unroll
            for (int w = 1; w < kSetThreads / 64; ++w) key = __builtin_fmax(key, keys[w]);
            if (!(key >= kSetTol)) break;                              // workgroup-uniform
            if (rank == kMaxRank) {
                shared = false;
                break;
            }
            const uint32_t at = (uint32_t)(__builtin_bit_cast(uint64_t, key) & 0x1fff);
            const int pc = at % kCols, pr = at / kCols, pi = pr / RG;
            const bool my_row = rg == pr % RG;
            if (my_row) {
                double v = a[0];
#pragma unroll
                for (int i = 1; i < RT; ++i) v = i == pi ? a[i] : v;
                U[rank * kLd + col] = v;
            }
            if (col == pc) {
#pragma unroll
                for (int i = 0; i < RT; ++i) pcol[i * RG + rg] = a[i];
            }
            if (tid == 0) piv[rank] = pc;
            __syncthreads();
            const double rp = 1.0 / U[rank * kLd + pc];
            if (tid == 0) rdiag[rank] = rp;
            const double q = col == pc ? 1.0 : U[rank * kLd + col] * rp;
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const double x = __builtin_fma(-pcol[i * RG + rg], q, a[i]);
                a[i] = my_row && i == pi ? 0.0 : x;
            }
            ++rank;
        }
        __syncthreads();
    }
    if (!shared) {                                                     // workgroup-uniform
        // one sub-record per function, in slot order
        if (rg == 0 && real_col) {
            double* x = o + cb * (kSetHeader + kNodes * nd);
            const int64_t p = aux_of_slot(slot0 + cb, N, G);
            if (ct == 0) {
                x[0] = R[3 * p]; x[1] = R[3 * p + 1]; x[2] = R[3 * p + 2];
                x[3] = __builtin_bit_cast(double, (uint64_t)kNodes |
                                                      ((uint64_t)(cb == nb - 1) << 32) |
                                                      ((uint64_t)(cb + 1) << 33));
            }
            if (form == kSetForward) {
                double* y = x + kSetHeader + 4 * ct;
                double S;
                y[0] = s;
                y[1] = fold_weight(wp / sqrt(s) * (kExpMinusHalf / kExpPolyK), &S);
                y[2] = S;
                y[3] = 1.0 / s;
            } else {
                double w[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b) w[b] = b == cb ? wp : 0.0;
                put(x + kSetHeader, ct, s, w);
            }
        }
        return;
    }
    // U11 t = sum of the function's columns of U, from the last row up: wave b, row k in lane
    // k % 64 (r1: rows from 64 on)
    if (tid < 64 * NB) {
        const int b = tid >> 6, lane = tid & 63;
        double r0 = 0.0, r1 = 0.0;
        if (lane < rank)
            for (int j = 0; j < kNodes; ++j) r0 += U[lane * kLd + b * kNodes + j];
        if (lane + 64 < rank)
            for (int j = 0; j < kNodes; ++j) r1 += U[(lane + 64) * kLd + b * kNodes + j];
        for (int m = rank - 1; m >= 0; --m) {                          // wave-uniform
            const double y = readlane_f64(m < 64 ? r0 : r1, m & 63) * rdiag[m];
            const int pc = piv[m];
            if (lane == 0) wsum[m][b] = y;
            if (lane < m) r0 = __builtin_fma(-U[lane * kLd + pc], y, r0);
            if (lane + 64 < m) r1 = __builtin_fma(-U[(lane + 64) * kLd + pc], y, r1);
        }
    }
    __syncthreads();
    if (tid == 0) {
        o[0] = rc[0]; o[1] = rc[1]; o[2] = rc[2];
        o[3] = __builtin_bit_cast(double, (uint64_t)(rank + (rank & 1)) | (1ull << 32));
    }
    if (tid < rank) {
        const double sm = cs[piv[tid]];
        int pos = 0;
        for (int m = 0; m < rank; ++m) {
            const double x = cs[piv[m]];
            pos += (x < sm || (x == sm && m < tid)) ? 1 : 0;
        }
        double w[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) w[b] = cw[piv[tid]] * wsum[tid][b];
        put(o + kSetHeader, pos, sm, w);
        if (pos == rank - 1 && (rank & 1)) {      // an odd list's last node again, weight 0
#pragma unroll
            for (int b = 0; b < NB; ++b) w[b] = 0.0;
            put(o + kSetHeader, rank, sm, w);
        }
    }
}

}  // namespace

size_t node_set_box_doubles() { return 8 * kBoxBlocks + 8; }

int launch_pair_box(int64_t n, const double* rec, int rec_stride, double* scratch,
                    hipStream_t s) {
    k_pair_box<<<kBoxBlocks, 256, 0, s>>>(n, rec, rec_stride, scratch + 8);
    k_pair_box_finish<<<1, 64, 0, s>>>(kBoxBlocks, scratch + 8, scratch);
    GSDFT_HIP(hipGetLastError());
    return GSDFT_OK;
}

int launch_node_sets(int64_t N, int64_t G, SetForm form, const double* beta, const double* kn,
                     const double* R, const double* dgamma, const double* dscale,
                     const double* box, double* out, hipStream_t s) {
    const NodeSets ns = node_sets(N, G, form);
    // groups in two dimensions: one holds at most 2^32 - 1 work-items, 13.4 million groups
    const int64_t row = std::min<int64_t>(std::max<int64_t>(ns.groups, 1), 1 << 20);
    const dim3 g((unsigned)row, (unsigned)((ns.groups + row - 1) / row));
    const NodeTable tb = coulomb_table();
    if (ns.nb == 2)
        k_node_sets<2><<<g, kSetThreads, 0, s>>>(N, G, ns.per_centre, ns.groups, ns.stride, beta, kn,
                                                 R, dgamma, dscale, form, box, tb, out);
    else
        k_node_sets<4><<<g, kSetThreads, 0, s>>>(N, G, ns.per_centre, ns.groups, ns.stride, beta, kn,
                                                 R, dgamma, dscale, form, box, tb, out);
    GSDFT_HIP(hipGetLastError());
    return GSDFT_OK;
}

}  // namespace gsdft
