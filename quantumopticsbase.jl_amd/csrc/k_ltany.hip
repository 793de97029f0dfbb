// Dense LazyTensor factors of any width on consecutive sites, several modes
// per pass over the state.
//
// Reference: _tp_sum_matmul! (src/operators_lazytensor.jl:443-488), one mode
// product (_tp_matmul!, :281-428) per factor, each a full pass.
//
// The state is viewed as (n1, P, n3), column-major, with P the product of the
// dimensions of the group of sites that a pass covers.  A workgroup keeps a
// tile in LDS while it applies the group's factors one after another:
//   n1 == 1:  nb consecutive blocks of P elements, contiguous in memory;
//   n1 >= 16: W rows (a power of two) by the P elements of one block, W-long
//             runs at a stride of n1.
// One mode of a tile is a real matrix product on MFMA.  The complex d x d
// factor acts as its real embedding [Re -Im; Im Re] on interleaved (re, im)
// pairs: a 16-row output tile holds 8 complex outputs and a k-step of 4 takes
// two complex inputs, so a factor of width d costs ceil8(d) * ceil2(d) complex
// products per fibre (d = 20: 480 for 400; separate real and imaginary tiles
// of 16: 640 for a k padded to 4).  The rows of the embedding are ordered so
// that a lane's accumulator registers hold both parts of its outputs.
//
// Bound by the MFMA rate plus what a wave issues between its MFMAs (the left
// pass of (12, 20, 9) on 2160^2 in ComplexF64, 67 us: MFMA pipes busy 51% of the
// cycles in which a CU is, 42% of the kernel, other vector instructions 18%) and
// by the barrier between modes; three or four small workgroups per CU overlap
// one's loads and stores with another's modes.
// Left application on a square rho, ComplexF64 / ComplexF32, mode-by-mode
// chain -> this: (12, 20, 9) 114 / 76 -> 62 / 36 us (2.4 / 2.1 TB/s),
// (8, 8, 8, 8) 423 / 283 -> 160 / 87 us (3.4 / 3.1 TB/s), (33, 12, 15) 1545 /
// 788 -> 597 / 297 us, (5, 7, 6) 15 / 19 -> 7.5 / 7.6 us; from the right
// (12, 20, 9) 100 / 63 -> 75 / 47 us.  Not kept: a lane per fibre on vector
// FMAs with the factor read through the scalar cache (same time on narrow
// factors, three times as long on 40 wide ones), two groups of fibres per
// wave at a time, 3 signed planes of the factor in LDS.
#include "qob_mfma.h"
#include "qob_rules.h"

#include <atomic>
#include <type_traits>

namespace qob {

namespace {

constexpr int ANY_B = 6;  // tile elements per thread loaded before the first is stored

// x with its sign flipped where neg
__device__ __forceinline__ double neg_if(double x, uint32_t neg) {
    return __hiloint2double(__double2hiint(x) ^ (int)neg, __double2loint(x));
}
__device__ __forceinline__ float neg_if(float x, uint32_t neg) { return __uint_as_float(__float_as_uint(x) ^ neg); }

// One mode: output tiles of 8 complex outputs for a group of 16 fibres per wave
// at a time.  F: the factor with 8 NT8 rows and an even number of columns,
// zeros outside the d x d factor; fib: each fibre's first element, ofib: the
// same without the LDS padding.  NS > 0: the number of k-steps, the factor's
// fragments stay in registers for all of the wave's groups; NS = 0: any
// number of k-steps, fragments read one k-step ahead.
template <typename R, int NT8, int NS>
__device__ __forceinline__ void any_mode(const AnyPass &S, const AnyMode &M, cplx<R> *tile, const cplx<R> *F,
                                         const uint16_t *fib, const uint16_t *ofib, int nf, bool direct,
                                         cplx<R> *__restrict__ out, int rows_ok, bool scale, cplx<R> alpha,
                                         cplx<R> beta, int beta_zero) {
    using T = cplx<R>;
    using V = typename mf<R>::v4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int d = M.d, ng = (nf + 15) >> 4, ldf = 8 * NT8;
    // row lr of an A tile: output 8 t + ao, real (ac = 0) or imaginary part
    const int ao = sizeof(R) == 8 ? (lr & 3) + 4 * (lr >> 3) : lr >> 1;
    const int ac = sizeof(R) == 8 ? (lr >> 2) & 1 : lr & 1;
    // column lk: input 2 ks + kh, real (kc = 0) or imaginary part
    const int kh = lk >> 1, kc = lk & 1;
    const uint32_t neg = (ac == 0 && kc == 1) ? 0x80000000u : 0u;
    const R *a0 = (const R *)F + 2 * (ao + kh * ldf) + (ac ^ kc);
    // outputs 8 t + ol + 4 h (f64) or 8 t + ol + h (f32) of this lane
    const int ol = sizeof(R) == 8 ? lk : 2 * lk;
    constexpr int OH = sizeof(R) == 8 ? 4 : 1;
    const int nsteps = NS ? NS : (d + 1) >> 1, xst = 4 * M.m1p;
    // odd width: the lanes of the input past the last one read the one before
    // it, and give zeros
    const bool odd = d & 1;
    const int xstl = odd && kh ? 0 : xst;
    const int64_t ost = S.n1 * (int64_t)(M.m1 >> S.lw);
    // from one output of the lane to the next: OH, then 8 - OH
    const int64_t ost0 = OH * ost, ost1 = (8 - OH) * ost;
    const int wst0 = OH * M.m1p, wst1 = (8 - OH) * M.m1p;
    constexpr int NR = NS ? NS : 1;
    R ar[NR][NT8];
    if constexpr (NS > 0) {
#pragma unroll
        for (int ks = 0; ks < NS; ++ks)
#pragma unroll
            for (int t = 0; t < NT8; ++t) ar[ks][t] = neg_if(a0[4 * ldf * ks + 16 * t], neg);
    }
    for (int g = wave; g < ng; g += nw) {
        const int f = g * 16 + lr;
        const bool fok = f < nf;
        const int base = fib[fok ? f : nf - 1];
        const R *xp = (const R *)tile + 2 * (base + (d > 1 ? M.m1p * kh : 0)) + kc;
        V acc[NT8];
        if constexpr (NS > 0) {
            R x[NS];
#pragma unroll
            for (int ks = 0; ks < NS; ++ks) {
                x[ks] = *xp;
                xp += ks + 2 == NS ? xstl : xst;
            }
            if (odd) x[NS - 1] = kh ? (R)0 : x[NS - 1];
#pragma unroll
            for (int ks = 0; ks < NS; ++ks)
#pragma unroll
                for (int t = 0; t < NT8; ++t) acc[t] = mf<R>::mma(ar[ks][t], x[ks], ks ? acc[t] : V{0, 0, 0, 0});
        } else {
            const R *ap = a0;
            R xn = *xp, an[NT8];
#pragma unroll
            for (int t = 0; t < NT8; ++t) {
                an[t] = ap[16 * t];
                acc[t] = V{0, 0, 0, 0};
            }
            for (int ks = 1; ks <= nsteps; ++ks) {
                R x = xn, a[NT8];
#pragma unroll
                for (int t = 0; t < NT8; ++t) a[t] = neg_if(an[t], neg);
                if (ks < nsteps) {
                    xp += ks + 1 == nsteps ? xstl : xst;
                    ap += 4 * ldf;
                    xn = *xp;
#pragma unroll
                    for (int t = 0; t < NT8; ++t) an[t] = ap[16 * t];
                } else if (odd) {
                    x = kh ? (R)0 : x;
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < NT8; ++t) acc[t] = mf<R>::mma(a[t], x, acc[t]);
            }
        }
        if (scale) {  // last mode, alpha != 1
#pragma unroll
            for (int t = 0; t < NT8; ++t)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const T v = cmul(alpha, mk((R)acc[t][2 * h], (R)acc[t][2 * h + 1]));
                    acc[t][2 * h] = v.x;
                    acc[t][2 * h + 1] = v.y;
                }
        }
        // a group's inputs are read by its own wave only: write in place
        if (!direct) {
            T *w = tile + base + M.m1p * ol;
            if (fok) {
#pragma unroll
                for (int t = 0; t < NT8; ++t)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (t + 1 < NT8 || 8 * t + ol + OH * h < d) *w = mk((R)acc[t][2 * h], (R)acc[t][2 * h + 1]);
                        w += h ? wst1 : wst0;
                    }
            }
        } else {
            const int e = ofib[fok ? f : nf - 1], i = e & (S.W - 1);
            T *w = out + i + S.n1 * (e >> S.lw) + ost * ol;
            if (fok && i < rows_ok) {
#pragma unroll
                for (int t = 0; t < NT8; ++t)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (t + 1 < NT8 || 8 * t + ol + OH * h < d) {
                            T r = mk((R)acc[t][2 * h], (R)acc[t][2 * h + 1]);
                            if (!beta_zero) r = cfma(beta, ldg(w), r);
                            stg_stream(w, r);
                        }
                        w += h ? ost1 : ost0;
                    }
            }
        }
    }
}

template <typename R>
__global__ void __launch_bounds__(1024) k_lt_any(AnyPass S, const cplx<R> *__restrict__ in, cplx<R> *__restrict__ out,
                                                 int64_t ntiles, double2 alpha_, double2 beta_, int beta_zero) {
    using T = cplx<R>;
    extern __shared__ unsigned char lds_raw[];
    T *F = (T *)lds_raw;  // every factor, padded (any_fac), then the tile, then the fibre tables
    T *tile = F + S.nfac;
    uint16_t *fibs = (uint16_t *)(tile + S.ntile);
    const int tid = threadIdx.x, nt = blockDim.x;
    const T alpha = mk((R)alpha_.x, (R)alpha_.y), beta = mk((R)beta_.x, (R)beta_.y);
    const bool scale = alpha_.x != 1.0 || alpha_.y != 0.0;
    for (int s = 0, off = 0, fo = 0; s < S.nmodes; ++s) {
        const AnyMode &M = S.m[s];
        const int d = M.d, ld = (d + 7) & ~7, n = ld * ((d + 1) & ~1);
        const T *A = (const T *)M.A;
        for (int e = tid; e < n; e += nt) {
            const int k = e / ld, a = e - k * ld;
            F[off + e] = a < d && k < d ? ldg(A + a + k * d) : czero<T>();
        }
        off += n;
        const int nf = M.pf * S.units;
        for (int f = tid; f < nf; f += nt) {
            const int i3 = f / M.m1, e = f - M.m1 * i3 + M.m1 * d * i3;
            fibs[fo + f] = (uint16_t)(S.padd ? e + (int)fdiv((uint32_t)e, S.fm0, S.fl0) : e);
            if (s + 1 == S.nmodes) fibs[fo + nf + f] = (uint16_t)e;
        }
        fo += nf;
    }
    // each XCD walks its own contiguous range of tiles
    const int x = blockIdx.x & 7, nx = gridDim.x >> 3;
    const int t1 = (int)(ntiles * (x + 1) / 8);
    for (int t = (int)(ntiles * x / 8) + (blockIdx.x >> 3); t < t1; t += nx) {
        int units = S.units, rows_ok = 1;
        int64_t go;
        if (S.n1 == 1) {
            const int64_t b0 = (int64_t)t * S.units;
            if (S.n3 - b0 < units) units = (int)(S.n3 - b0);
            go = b0 * S.P;
        } else {
            const int q = (int)fdiv((uint32_t)t, S.fmr, S.flr);
            const int64_t r0 = (int64_t)(t - q * S.nrb) * S.W;
            rows_ok = (int)(S.n1 - r0 < S.W ? S.n1 - r0 : S.W);
            go = r0 + S.n1 * S.P * (int64_t)q;
        }
        const int E = units * S.P;
        const T *src = in + go;
        for (int b0 = 0; b0 < E; b0 += ANY_B * nt) {
            T v[ANY_B];
#pragma unroll
            for (int j = 0; j < ANY_B; ++j) {
                if (b0 + j * nt >= E) continue;  // uniform
                const int e = b0 + j * nt + tid < E ? b0 + j * nt + tid : E - 1;
                if (S.n1 == 1) {
                    v[j] = ldg(src + e);
                } else {
                    const int i = e & (S.W - 1);
                    v[j] = ldg(src + (i < rows_ok ? i : rows_ok - 1) + S.n1 * (int64_t)(e >> S.lw));
                }
            }
            if (b0 == 0) __syncthreads();  // the previous tile's last mode has been read
#pragma unroll
            for (int j = 0; j < ANY_B; ++j) {
                if (b0 + j * nt >= E) continue;
                const int e = b0 + j * nt + tid;
                if (e < E) tile[S.padd ? e + (int)fdiv((uint32_t)e, S.fm0, S.fl0) : e] = v[j];
            }
        }
        for (int s = 0, off = 0, fo = 0; s < S.nmodes; ++s) {
            __syncthreads();
            const AnyMode &M = S.m[s];
            const bool direct = s + 1 == S.nmodes && !S.lin;
            const int nf = units * M.pf;
#define NSW(n) (sizeof(R) == 4 ? n : 0)
#define QOB_AM(N, NS)                                                                                             \
    any_mode<R, N, NS>(S, M, tile, F + off, fibs + fo, fibs + fo + S.units * M.pf, nf, direct, out + go, rows_ok,     \
                       scale && s + 1 == S.nmodes, alpha, beta, beta_zero)
            switch ((M.d + 1) >> 1) {
            case 1: QOB_AM(1, 1); break;
            case 2: QOB_AM(1, 2); break;
            case 3: QOB_AM(1, 3); break;
            case 4: QOB_AM(1, 4); break;
            case 5: QOB_AM(2, 5); break;
            case 6: QOB_AM(2, 6); break;
            case 7: QOB_AM(2, 7); break;
            case 8: QOB_AM(2, 8); break;
            case 9: QOB_AM(3, NSW(9)); break;
            case 10: QOB_AM(3, NSW(10)); break;
            case 11:
            case 12: QOB_AM(3, 0); break;
            case 13:
            case 14:
            case 15:
            case 16: QOB_AM(4, 0); break;
            default: QOB_AM(5, 0); break;
            }
#undef QOB_AM
            off += ((M.d + 7) & ~7) * ((M.d + 1) & ~1);
            fo += S.units * M.pf;
        }
        if (S.lin) {  // contiguous tile whose last mode's fibres are not: written out in order
            __syncthreads();
            for (int e = tid; e < E; e += nt) {
                T r = tile[S.padd ? e + (int)fdiv((uint32_t)e, S.fm0, S.fl0) : e];
                T *o = out + go + e;
                if (!beta_zero) r = cfma(beta, ldg(o), r);
                stg_stream(o, r);
            }
        }
    }
}

}  // namespace

// Fills the parts of S that follow from n1, n3, P, the modes' widths and
// strides; returns the LDS bytes of a workgroup, or 0 when the pass does not
// fit one.
size_t any_plan(qob_dtype dt, AnyPass &S) {
    const size_t es = dt == QOB_C64 ? 16 : 8;
    S.nfac = 0;
    for (int s = 0; s < S.nmodes; ++s) {
        AnyMode &M = S.m[s];
        if (M.d < 1 || M.d > ANY_MAXD) return 0;
        S.nfac += ((M.d + 7) & ~7) * ((M.d + 1) & ~1);
    }
    const size_t fb = S.nfac * es, cap = 160 * 1024;
    if (fb >= cap) return 0;
    S.W = 1;
    S.lw = 0;
    S.units = 1;
    S.nrb = 1;
    S.padd = 0;
    int64_t E = S.P, pad = 0, nfib = 0;
    if (S.n1 == 1) {
        // up to 32 KiB per tile, but two tiles per CU, and not less than the
        // factors' size (each workgroup loads them)
        if (S.n3 > 0x7fffffff) return 0;
        const int64_t bb = (int64_t)(S.P * es);
        S.units = (int)std::max<int64_t>(1, std::min<int64_t>(std::max<int64_t>(S.n3 / (2 * device_cu_count()), fb / bb),
                                                           (32 * 1024) / bb));
        E = (int64_t)S.units * S.P;
        if (S.m[0].m1 == 1 && S.m[0].d % 2 == 0) {
            S.padd = 1;
            const FastDiv f = make_fastdiv((uint32_t)S.m[0].d);
            S.fm0 = f.m;
            S.fl0 = f.l;
            pad = E / S.m[0].d;
        }
    } else {
        const int W = any_rows(es == 16, S.n1, S.P, S.n3, device_cu_count());
        S.W = W;
        while ((1 << S.lw) < W) ++S.lw;
        S.units = W;
        const int64_t nrb = (S.n1 + W - 1) / W;
        if (nrb > 0x7fffffff / std::max<int64_t>(S.n3, 1)) return 0;
        S.nrb = (int)nrb;
        const FastDiv f = make_fastdiv((uint32_t)S.nrb);
        S.fmr = f.m;
        S.flr = f.l;
        E = (int64_t)W * S.P;
    }
    for (int s = 0; s < S.nmodes; ++s) {
        AnyMode &M = S.m[s];
        M.m1 *= S.W;  // innermost: the tile's rows
        M.m1p = S.padd && M.m1 > 1 ? M.m1 + M.m1 / S.m[0].d : M.m1;
        M.pf = S.P / M.d;
        nfib += (int64_t)S.units * M.pf * (s + 1 == S.nmodes ? 2 : 1);
    }
    S.lin = S.n1 == 1 && S.m[S.nmodes - 1].m1 < 16;
    if (E > 0xffff - pad) return 0;  // the fibre tables hold 16-bit offsets
    S.ntile = (int)(E + pad);
    const size_t lds = fb + (size_t)S.ntile * es + (size_t)nfib * 2;
    return lds <= cap ? lds : 0;
}

hipError_t launch_lt_any(qob_dtype dt, AnyPass S, const void *in, void *out, double2 alpha, double2 beta,
                         hipStream_t s) {
    const size_t lds = any_plan(dt, S);
    if (!lds) return hipErrorNotSupported;
    const int bz = (beta.x == 0.0 && beta.y == 0.0);
    const int64_t nt = S.n1 == 1 ? (S.n3 + S.units - 1) / S.units : S.nrb * S.n3;
    if (nt <= 0) return hipSuccess;
    if (nt > 0x7fffffff) return hipErrorNotSupported;
    // 16 waves per CU (128 registers), in as many workgroups as the LDS holds
    // (allocated in units of 1280 bytes)
    const int per_cu = (int)std::max<size_t>(1, (160 * 1024) / ((lds + 1279) / 1280 * 1280));
    const int res = std::min(per_cu, 4), threads = res >= 3 ? 256 : 1024 / res;
    const int64_t g = std::min<int64_t>((nt + 7) / 8 * 8, (int64_t)device_cu_count() * res);
    const unsigned grid = (unsigned)std::max<int64_t>(8, g / 8 * 8);
#define QOB_LA(RR)                                                                                                  \
    do {                                                                                                            \
        auto k = k_lt_any<RR>;                                                                                      \
        static std::atomic<int> set{0};                                                                             \
        if (!set.load()) {                                                                                          \
            hipError_t e =                                                                                          \
                hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);       \
            if (e != hipSuccess) return e;                                                                          \
            set.store(1);                                                                                           \
        }                                                                                                           \
        hipLaunchKernelGGL(k, dim3(grid), dim3(threads), lds, s, S, (const cplx<RR> *)in, (cplx<RR> *)out, nt, alpha, \
                           beta, bz);                                                                               \
        return hipGetLastError();                                                                                   \
    } while (0)
    if (dt == QOB_C64) QOB_LA(double);
    QOB_LA(float);
#undef QOB_LA
}

}  // namespace qob
