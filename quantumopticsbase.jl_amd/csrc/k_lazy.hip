// Pure-sparse LazyTensor / LazySum application in gather form.
//
// Reference: mul! on a LazySum (src/operators_lazysum.jl:189-238) calls the
// LazyTensor mul! once per term (src/operators_lazytensor.jl:539-609), which
// for all-sparse factors runs the recursive scatter _gemm_recursive_lazy_dense
// (:652-685, left / Ket) or _gemm_recursive_dense_lazy (:613-648, right /
// Bra), each a full read-modify-write pass over the result.
//
// Here every term of the sum is compiled (on the host) into a gather table
// over the term's own sites, and one launch evaluates all terms for each
// output element:
//   out[J] = alpha * ( sum_t sum_{e in row(t, J)} v_e * in[K_e(J)] ) + beta * out[J]
// so the result is written once and the input is read once per term group
// (re-reads are served by LDS/L1/L2, not HBM).  Diagonal terms are folded
// into one coefficient per element before a single multiply with in[J].
//
// k_gather_rows: the gather axis is the fastest (stride 1) axis — a Ket, or
//                the row index of a density matrix (left application).
// k_gather_cols: the gather axis is the column index of a density matrix
//                (right application); lanes run along the contiguous rows and
//                the whole term walk is wave-uniform.
#include "qob_internal.h"

#include <algorithm>

namespace qob {

namespace {

template <typename T> __device__ __forceinline__ T to_t(double2 a) {
    T r; r.x = (typename real_of<T>::type)a.x; r.y = (typename real_of<T>::type)a.y; return r;
}

struct Digits {
    // non-square only: r-space offset of the element and mask of sites whose
    // l-digit is outside the r-range (identity there contributes nothing)
    int64_t jr_all;
    uint32_t invalid;
};

__device__ __forceinline__ uint32_t digit_of(uint32_t J, const int32_t *s) {
    // s: stride_l, m_stride, l_stride, d_l, m_d, l_d
    const uint32_t qv = fdiv(J, (uint32_t)s[1], (uint32_t)s[2]);
    return qv - (uint32_t)s[3] * fdiv(qv, (uint32_t)s[4], (uint32_t)s[5]);
}

__device__ __forceinline__ Digits all_digits(uint32_t J, int nsites, const int32_t *__restrict__ site_info) {
    Digits d;
    d.jr_all = 0;
    d.invalid = 0;
    for (int s = 0; s < nsites; ++s) {
        const int32_t *si = site_info + 8 * s;
        const uint32_t j = digit_of(J, si);
        d.jr_all += (int64_t)j * si[6];
        if (j >= (uint32_t)si[7]) d.invalid |= (1u << s);
    }
    return d;
}

// Sum over all terms for output J.  Returns (acc, dacc): gathered part and
// diagonal coefficient.  LD(K) loads in[K].
template <typename T, bool SQUARE, typename LD>
__device__ __forceinline__ T eval_terms(uint32_t J, const GatherPlanDev &P, const Digits &dg, LD ld) {
    const T *__restrict__ vals = (const T *)P.vals;
    T acc = czero<T>();
    T dacc = czero<T>();
    const int32_t *pg = P.prog;
    for (int t = 0; t < P.nterms; ++t) {
        const int kind = pg[0], flags = pg[1], q = pg[2], base = pg[3];
        const uint32_t fmask = (uint32_t)pg[4];
        const int32_t *sr = pg + GP_HDR;
        pg += GP_HDR + GP_SITE * q;
        if (!SQUARE && (dg.invalid & ~fmask)) continue;
        int64_t kb = SQUARE ? (int64_t)J : dg.jr_all;
        if (kind == 0) {
            int jloc = 0;
            for (int i = 0; i < q; ++i) {
                const int32_t *s = sr + GP_SITE * i;
                const uint32_t j = digit_of(J, s);
                jloc += (int)j * s[6];
                if (!SQUARE) kb -= (int64_t)j * s[8];
            }
            const int32_t p0 = P.rowptr[base + jloc], p1 = P.rowptr[base + jloc + 1];
            if (flags & 1) {
                for (int32_t p = p0; p < p1; ++p) dacc = cadd(dacc, vals[p]);
            } else {
                for (int32_t p = p0; p < p1; ++p) acc = cfma(vals[p], ld(kb + P.koff[p]), acc);
            }
        } else {
            T v = mk((typename real_of<T>::type)1, (typename real_of<T>::type)0);
            int64_t off = 0;
            bool live = true;
            for (int i = 0; i < q; ++i) {
                const int32_t *s = sr + GP_SITE * i;
                const uint32_t j = digit_of(J, s);
                const int e = s[7] + (int)j;
                const T a = vals[e];
                live = live && (a.x != 0 || a.y != 0);
                v = cmul(v, a);
                off += P.koff[e];
                if (!SQUARE) kb -= (int64_t)j * s[8];
            }
            if (live) {
                if (flags & 1) dacc = cadd(dacc, v);
                else acc = cfma(v, ld(kb + off), acc);
            }
        }
    }
    if (dacc.x != 0 || dacc.y != 0) {
        // diagonal terms only exist for square operators
        acc = cfma(dacc, ld((int64_t)J), acc);
    }
    return acc;
}

template <typename T, bool SQUARE>
__global__ void __launch_bounds__(256) k_gather_rows(GatherPlanDev P, const T *__restrict__ in, int64_t n_in,
                                                     T *__restrict__ out, int64_t n_out, int64_t nbatch,
                                                     double2 alpha_, double2 beta_, int beta_zero) {
    const int64_t J = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (J >= n_out) return;
    const T alpha = to_t<T>(alpha_), beta = to_t<T>(beta_);
    Digits dg{0, 0};
    if (!SQUARE) dg = all_digits((uint32_t)J, P.nsites, P.site_info);
    for (int64_t b = blockIdx.y; b < nbatch; b += gridDim.y) {
        const T *ib = in + b * n_in;
        T *o = out + b * n_out + J;
        const T acc = eval_terms<T, SQUARE>((uint32_t)J, P, dg, [&](int64_t K) { return ib[K]; });
        *o = axpby(alpha, acc, beta, o, beta_zero != 0);
    }
}

// The same sum from the plan's fibre tables: every table load of an element is
// issued at once, then every gathered element.  A wave's 64 elements lie in at
// most two fibres (fib >= 64): the factors of the sites above are scalar loads
// of both, which leaves the vector loads to the sites below and the elements.
template <typename T, int NP>
__global__ void __launch_bounds__(256) k_gather_fibre(GatherPlanDev P, const T *__restrict__ in, T *__restrict__ out,
                                                      int64_t nbatch, double2 alpha_, double2 beta_, int beta_zero) {
    const T alpha = to_t<T>(alpha_), beta = to_t<T>(beta_);
    const T *__restrict__ fv = (const T *)P.vals + P.fv;
    const int32_t *__restrict__ fk = P.koff + P.fk;
    const uint32_t n = P.n, len = P.fib + P.nf;
    // XCD x takes a contiguous eighth of the list of chunks, which has the
    // chunks of the top digits t = 0 .. td - 1 at the same place r side by side
    const uint32_t k = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const uint32_t chunk = fdiv(k, P.td_m, P.td_l), t = k - chunk * P.td;
    if (chunk * 256u >= P.ts) return;
    const uint32_t r = chunk * 256u + threadIdx.x;
    const uint32_t J = t * P.ts + min(r, P.ts - 1);
    const uint32_t f = fdiv(J, P.fib_m, P.fib_l), m = J - f * P.fib;
    const uint32_t f0 = __builtin_amdgcn_readfirstlane(f), f1 = min(f0 + 1, P.nf - 1);
    const bool nx = f != f0;
    const T dl = fv[m], du0 = fv[P.fib + f0], du1 = fv[P.fib + f1];
    T v[NP + 1];
    int32_t off[NP + 1];
    uint32_t live = 0;
    T lv[NP + 1], u0[NP + 1], u1[NP + 1];
    int32_t lo[NP + 1], o0[NP + 1], o1[NP + 1];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        lv[p] = fv[len * (p + 1) + m];
        lo[p] = fk[len * p + m];
        u0[p] = fv[len * (p + 1) + P.fib + f0];
        u1[p] = fv[len * (p + 1) + P.fib + f1];
        o0[p] = fk[len * p + P.fib + f0];
        o1[p] = fk[len * p + P.fib + f1];
    }
    T dv = cadd(dl, nx ? du1 : du0);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const bool l = P.has_lo >> p & 1, u = P.has_up >> p & 1;
        const T uv = nx ? u1[p] : u0[p];
        const int32_t uo = nx ? o1[p] : o0[p];
        v[p] = l && u ? cmul(lv[p], uv) : (l ? lv[p] : uv);
        bool a = lo[p] != GP_DEAD && uo != GP_DEAD;
        if (P.skip0 >> p & 1) a = a && (lv[p].x != 0 || lv[p].y != 0) && (uv.x != 0 || uv.y != 0);
        off[p] = a ? lo[p] + uo : 0;
        if (P.diag >> p & 1) {
            if (a) dv = cadd(dv, v[p]);
            a = false;
        }
        live |= (uint32_t)a << p;
    }
    for (int64_t b = blockIdx.y; b < nbatch; b += gridDim.y) {
        const T *ib = in + b * n;
        T *o = out + b * n + J;
        T x[NP + 1];
        x[NP] = ib[J];
#pragma unroll
        for (int p = 0; p < NP; ++p) x[p] = ib[(int64_t)J + off[p]];
        T acc = czero<T>();
#pragma unroll
        for (int p = 0; p < NP; ++p)
            if (live >> p & 1) acc = cfma(v[p], x[p], acc);
        if (dv.x != 0 || dv.y != 0) acc = cfma(dv, x[NP], acc);
        if (r < P.ts) *o = axpby(alpha, acc, beta, o, beta_zero != 0);
    }
}

template <typename T, bool SQUARE>
__global__ void __launch_bounds__(256) k_gather_cols(GatherPlanDev P, const T *__restrict__ in, int64_t n_in,
                                                     T *__restrict__ out, int64_t n_out, int64_t nrows,
                                                     double2 alpha_, double2 beta_, int beta_zero) {
    (void)n_in;  // the plan is compiled for this input length (the entry points check it)
    const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
    const T alpha = to_t<T>(alpha_), beta = to_t<T>(beta_);
    const bool ok = i < nrows;
    for (int64_t J = blockIdx.y; J < n_out; J += gridDim.y) {
        Digits dg{0, 0};
        if (!SQUARE) dg = all_digits((uint32_t)J, P.nsites, P.site_info);
        const T *ib = in + (ok ? i : 0);
        const T acc = eval_terms<T, SQUARE>((uint32_t)J, P, dg, [&](int64_t K) { return ib[K * nrows]; });
        if (ok) {
            T *o = out + i + J * nrows;
            *o = axpby(alpha, acc, beta, o, beta_zero != 0);
        }
    }
}

// FP64 block sum of a double2 (256 threads); lane 0 of wave 0 gets the total
__device__ __forceinline__ double2 block_sum256(double2 v) {
    __shared__ double2 sh[256];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            sh[threadIdx.x].x += sh[threadIdx.x + w].x;
            sh[threadIdx.x].y += sh[threadIdx.x + w].y;
        }
        __syncthreads();
    }
    return sh[0];
}

// mode: GatherDot
template <typename T, int MODE>
__global__ void __launch_bounds__(256) k_gather_dot(GatherPlanDev P, const T *__restrict__ u, const T *__restrict__ v,
                                                    int64_t n, double2 *__restrict__ partials) {
    double2 r = make_double2(0, 0), p = make_double2(0, 0);
    for (int64_t J = blockIdx.x * (int64_t)256 + threadIdx.x; J < n; J += (int64_t)gridDim.x * 256) {
        Digits dg{0, 0};
        T acc;
        if (MODE != GD_TRACE) {
            acc = eval_terms<T, true>((uint32_t)J, P, dg, [&](int64_t K) { return v[K]; });
            const T a = u[J];
            r.x += (double)a.x * acc.x + (double)a.y * acc.y;
            r.y += (double)a.x * acc.y - (double)a.y * acc.x;
            if (MODE == GD_BILINEAR_DOT) {
                const T b = v[J];
                p.x += (double)a.x * b.x + (double)a.y * b.y;
                p.y += (double)a.x * b.y - (double)a.y * b.x;
            }
        } else {
            const T *col = v + J * n;
            acc = eval_terms<T, true>((uint32_t)J, P, dg, [&](int64_t K) { return col[K]; });
            r.x += acc.x;
            r.y += acc.y;
        }
    }
    const double2 t = block_sum256(r);
    if (threadIdx.x == 0) partials[blockIdx.x] = t;
    if (MODE == GD_BILINEAR_DOT) {
        __syncthreads();
        const double2 q = block_sum256(p);
        if (threadIdx.x == 0) partials[gridDim.x + blockIdx.x] = q;
    }
}

}  // namespace

int gather_dot_blocks(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(1024, (n + 255) / 256)); }

hipError_t launch_gather_dot(qob_dtype dt, const GatherPlanDev &P, GatherDot mode, const void *u, const void *v, int64_t n,
                             double2 *partials, hipStream_t s) {
    if (!P.square) return hipErrorInvalidValue;
    const int g = gather_dot_blocks(n);
#define QOB_GD(TT, MD) \
    hipLaunchKernelGGL((k_gather_dot<TT, MD>), dim3(g), dim3(256), 0, s, P, (const TT *)u, (const TT *)v, n, partials)
#define QOB_GDM(TT)                                                    \
    do {                                                               \
        if (mode == GD_BILINEAR) QOB_GD(TT, GD_BILINEAR);              \
        else if (mode == GD_TRACE) QOB_GD(TT, GD_TRACE);               \
        else QOB_GD(TT, GD_BILINEAR_DOT);                              \
    } while (0)
    if (dt == QOB_C64) QOB_GDM(double2);
    else QOB_GDM(float2);
#undef QOB_GDM
#undef QOB_GD
    return hipGetLastError();
}

hipError_t launch_gather_rows(qob_dtype dt, const GatherPlanDev &P, const void *in, int64_t n_in, void *out,
                              int64_t n_out, int64_t nbatch, double2 alpha, double2 beta, hipStream_t s) {
    if (n_out == 0 || nbatch == 0) return hipSuccess;
    const int bz = (beta.x == 0.0 && beta.y == 0.0);
    if (P.np >= 0) {
        const uint32_t chunks = (P.ts + 255) / 256 * P.td;
        const dim3 gf((chunks + 7) / 8 * 8, (uint32_t)(nbatch < 65535 ? nbatch : 65535));
#define QOB_GF(NP)                                                                                                   \
    case NP:                                                                                                         \
        if (dt == QOB_C64)                                                                                           \
            hipLaunchKernelGGL((k_gather_fibre<double2, NP>), gf, dim3(256), 0, s, P, (const double2 *)in,           \
                               (double2 *)out, nbatch, alpha, beta, bz);                                             \
        else                                                                                                         \
            hipLaunchKernelGGL((k_gather_fibre<float2, NP>), gf, dim3(256), 0, s, P, (const float2 *)in,             \
                               (float2 *)out, nbatch, alpha, beta, bz);                                              \
        break;
        switch (P.np) {
            QOB_GF(0) QOB_GF(1) QOB_GF(2) QOB_GF(3) QOB_GF(4) QOB_GF(5) QOB_GF(6)
            default: return hipErrorInvalidValue;
        }
#undef QOB_GF
        return hipGetLastError();
    }
    const dim3 g((uint32_t)((n_out + 255) / 256), (uint32_t)(nbatch < 65535 ? nbatch : 65535));
#define QOB_GR(TT, SQ) \
    hipLaunchKernelGGL((k_gather_rows<TT, SQ>), g, dim3(256), 0, s, P, (const TT *)in, n_in, (TT *)out, n_out, nbatch, alpha, beta, bz)
    if (dt == QOB_C64) { if (P.square) QOB_GR(double2, true); else QOB_GR(double2, false); }
    else { if (P.square) QOB_GR(float2, true); else QOB_GR(float2, false); }
#undef QOB_GR
    return hipGetLastError();
}

hipError_t launch_gather_cols(qob_dtype dt, const GatherPlanDev &P, const void *in, int64_t n_in, void *out,
                              int64_t n_out, int64_t nrows, double2 alpha, double2 beta, hipStream_t s) {
    if (n_out == 0 || nrows == 0) return hipSuccess;
    const int bz = (beta.x == 0.0 && beta.y == 0.0);
    (void)n_in;
    const dim3 g((uint32_t)((nrows + 255) / 256), (uint32_t)(n_out < 65535 ? n_out : 65535));
#define QOB_GC(TT, SQ) \
    hipLaunchKernelGGL((k_gather_cols<TT, SQ>), g, dim3(256), 0, s, P, (const TT *)in, n_in, (TT *)out, n_out, nrows, alpha, beta, bz)
    if (dt == QOB_C64) { if (P.square) QOB_GC(double2, true); else QOB_GC(double2, false); }
    else { if (P.square) QOB_GC(float2, true); else QOB_GC(float2, false); }
#undef QOB_GC
    return hipGetLastError();
}

}  // namespace qob
