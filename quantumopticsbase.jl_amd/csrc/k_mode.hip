// Dense mode products and dense operator products on MFMA.
//
// Reference: the mode product of a tensor-product factor, _tp_matmul!
// (src/operators_lazytensor.jl:406-428), which dispatches to
// _tp_matmul_first! (:281-290), _tp_matmul_last! (:292-301) or
// _tp_matmul_mid! (:333-404, permutes through cached temporaries), and the
// DenseOperator mul! through BLAS gemm / gemv (src/operators_dense.jl:394-396).
// All of them are one operation here:
//   out[i1, a, i3] = alpha * sum_b F[a, b] in[i1, b, i3] + beta * out[i1, a, i3]
// with in viewed (n1, d_in, n3) and out (n1, d_out, n3), column-major, and F
// the d_out x d_in factor (column-major; a transposed or conjugated variant
// is materialised by the caller).  No permutation is ever materialised.
//
// Kernels (every complex product from four real MFMAs, see qob_mfma.h):
//   k_mode_fib    n1 >= 16, d_in, d_out <= 64.  A wave takes 16 fibres with
//                 consecutive i1 (one i3): their elements are read from HBM
//                 straight into MFMA B-fragments (16 consecutive i1 = 256 B
//                 runs), the factor's A-fragments come from LDS (staged once
//                 per workgroup), and the D tiles go straight back to HBM
//                 (again 256 B runs).  Each element is read and written once.
//   k_mode_chunk  n1 < 16 (the factor on the first, fastest site, or sites
//                 of small dimension before it), d_in, d_out <= 64.  A chunk
//                 of consecutive i3 blocks is contiguous in memory: it is
//                 loaded linearly into LDS planes, the mode product runs from
//                 LDS into output planes, and the output chunk is written
//                 back linearly.
//   k_zgemm       everything wider: an LDS-tiled complex GEMM
//                 with arbitrary element strides and a batch index, used for
//                 factors wider than 64 and for DenseOperator on a density
//                 matrix (and qob_gemm).
//   k_zgemm_small the same with one 16 x 16 tile per workgroup, for products
//                 of few tiles per CU.
//   k_zgemv       a single vector (DenseOperator on a Ket or Bra): columns
//                 of F split over workgroups, deterministic two-stage sum;
//                 up to 1536 rows and columns in one launch (k_zgemv_one).
#include "qob_mfma.h"
#include "qob_rules.h"

#include <map>
#include <mutex>
#include <numeric>
#include <type_traits>
#include <unordered_set>

namespace qob {

namespace {

__device__ __forceinline__ int pad16(int i) { return i + (i >> 4); }

constexpr int MODE_NT = 512;  // threads per workgroup of the mode kernels

// F (d_out x d_in, column-major) into Fs[i + k * ldf] for i < rows,
// k < cols, zero outside F.
template <typename T>
__device__ void stage_factor(T *Fs, int ldf, int rows, int cols, const T *__restrict__ F, int d_out, int d_in) {
    for (int e = threadIdx.x; e < rows * cols; e += blockDim.x) {
        const int i = e % rows, k = e / rows;
        Fs[i + k * ldf] = (i < d_out && k < d_in) ? F[i + (int64_t)k * d_out] : czero<T>();
    }
}

// ------------------------------------------------------------ k_mode_fib
// NT16 = ceil(max(d_in, d_out) / 16): output tiles per fibre group and
// k-steps / 4.  A fibre group is 16 fibres: with n1 >= 16, 16 consecutive
// i1 of one i3 (gpi groups per i3); with n1 < 16 (flat), 16 consecutive
// fibres f = i1 + n1 * i3 of the nf = n1 * n3 fibres.  The loads of the next
// chunk of 16 k -- the next group's first chunk after a group's last -- are
// in flight during the current chunk's MFMAs and the group's stores.
struct FibreAt {
    const void *p;  // first element of the fibre (in), or null past the end
    int64_t o;      // offset of the fibre in out
};
template <typename R, int NT16>
__global__ void __launch_bounds__(MODE_NT) k_mode_fib(const cplx<R> *__restrict__ F, int d_out, int d_in,
                                                       const cplx<R> *__restrict__ in, cplx<R> *__restrict__ out,
                                                       int n1, int gpi, int64_t ngroups, int64_t nf,
                                                       double2 alpha_, double2 beta_, int beta_zero, int flat) {
    using T = cplx<R>;
    using V = typename mf<R>::v4;
    constexpr int KS = 4 * NT16, LDF = 16 * NT16 + 1;
    extern __shared__ unsigned char lds_raw[];
    T *Fs = (T *)lds_raw;
    stage_factor(Fs, LDF, 16 * NT16, 4 * KS, F, d_out, d_in);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const T alpha = mk((R)alpha_.x, (R)alpha_.y), beta = mk((R)beta_.x, (R)beta_.y);
    const int64_t sin = (int64_t)n1 * d_in, sout = (int64_t)n1 * d_out;
    constexpr int WPB = MODE_NT / 64;
    const int64_t gstep = (int64_t)gridDim.x * WPB;
    // this lane's fibre of group g
    auto fibre = [&](int64_t g) -> FibreAt {
        int64_t i3;
        int i1;
        bool ok;
        if (g >= ngroups) return {nullptr, 0};
        if (flat) {
            const int64_t f = g * 16 + lr;
            ok = f < nf;
            i3 = n1 == 1 ? f : f / n1;
            i1 = (int)(f - i3 * n1);
        } else {
            i3 = g / gpi;
            i1 = (int)(g - i3 * gpi) * 16 + lr;
            ok = i1 < n1;
        }
        if (!ok) return {nullptr, 0};
        return {in + i1 + i3 * sin, i1 + i3 * sout};
    };
    // Every lane issues all of its loads (from an in-bounds address where
    // the element does not exist, followed by a zero select): with loads
    // under a branch the compiler must assume that none was issued after
    // the chunk in use, and waited for the next chunk's loads before this
    // chunk's MFMAs.  (16, 32, 16) chain on an 8192^2 rho: 1.211 -> 1.185 ms.
    auto load = [&](const FibreAt &fa, int kc, T (&x)[4]) {
        const T *base = fa.p ? (const T *)fa.p : in;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int b = 16 * kc + 4 * j + lk;
            const bool ok = fa.p && b < d_in;
            const T v = ldg(base + (int64_t)n1 * (ok ? b : 0));
            x[j] = ok ? v : czero<T>();
        }
    };
    int64_t g = (int64_t)blockIdx.x * WPB + wave;
    FibreAt cur = fibre(g);
    T x[4], xn[4];
    load(cur, 0, x);
    for (; g < ngroups; g += gstep) {
        const FibreAt nxt = fibre(g + gstep);
        V ar[NT16], ai[NT16];
#pragma unroll
        for (int t = 0; t < NT16; ++t) {
            ar[t] = V{0, 0, 0, 0};
            ai[t] = V{0, 0, 0, 0};
        }
#pragma unroll 1
        for (int kc = 0; kc < NT16; ++kc) {
            if (kc + 1 < NT16) load(cur, kc + 1, xn);
            else load(nxt, 0, xn);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int t = 0; t < NT16; ++t)
                    cmma4<R>(Fs[(16 * t + lr) + (16 * kc + 4 * j + lk) * LDF], x[j], ar[t], ai[t]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = xn[j];
        }
        if (cur.p) {
            T *ob = out + cur.o;
#pragma unroll
            for (int t = 0; t < NT16; ++t) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int a = 16 * t + mf<R>::row(lane, r);
                    if (a < d_out) {
                        T *o = ob + (int64_t)n1 * a;
                        T v = cmul(alpha, mk((R)ar[t][r], (R)ai[t][r]));
                        if (!beta_zero) v = cfma(beta, *o, v);
                        st_stream(o, v);
                    }
                }
            }
        }
        cur = nxt;
    }
}

// ---------------------------------------------------------- k_mode_chunk
// Chunks of cpc consecutive i3 blocks (cpc * n1 * d elements, contiguous).
constexpr int CHUNK_NT = 256;  // threads per workgroup: small chunks, several workgroups per CU
// input elements per thread loaded one chunk ahead (a ComplexF64 chunk of
// 32 KB of planes holds 512 input elements for square factors, ComplexF32 1024)
template <typename R> constexpr int chunk_pf() { return sizeof(R) == 8 ? 2 : 4; }
template <typename R, int NT16>
__global__ void __launch_bounds__(CHUNK_NT) k_mode_chunk(const cplx<R> *__restrict__ F, int d_out, int d_in,
                                                         const cplx<R> *__restrict__ in, cplx<R> *__restrict__ out,
                                                         int n1, int64_t n3, int cpc, int64_t nchunks,
                                                         double2 alpha_, double2 beta_, int beta_zero) {
    using T = cplx<R>;
    using V = typename mf<R>::v4;
    constexpr int KS = 4 * NT16, LDF = 16 * NT16 + 1;
    extern __shared__ unsigned char lds_raw[];
    T *Fs = (T *)lds_raw;
    const int pin = pad16(cpc * n1 * d_in) + 1, pout = pad16(cpc * n1 * d_out) + 1;
    R *ire = (R *)(Fs + 4 * KS * LDF);
    R *iim = ire + pin;
    R *ore = iim + pin;
    R *oim = ore + pout;
    stage_factor(Fs, LDF, 16 * NT16, 4 * KS, F, d_out, d_in);  // ordered by the first barrier below
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const T alpha = mk((R)alpha_.x, (R)alpha_.y), beta = mk((R)beta_.x, (R)beta_.y);
    // The first CHUNK_PF * CHUNK_NT input elements of the next chunk are
    // loaded into registers while this chunk is multiplied and written out
    // (the rest of a larger chunk is loaded when it is staged).
    auto chunk_in = [&](int64_t c, int &ne) -> const T * {
        const int64_t i30 = c * cpc;
        const int nb = (int)(n3 - i30 < cpc ? n3 - i30 : cpc);
        ne = nb * n1 * d_in;
        return in + i30 * n1 * d_in;
    };
    constexpr int CHUNK_PF = chunk_pf<R>();
    T pre[CHUNK_PF];
    auto prefetch = [&](int64_t c) {
        int ne = 0;
        const T *src = c < nchunks ? chunk_in(c, ne) : in;
#pragma unroll
        for (int j = 0; j < CHUNK_PF; ++j) {
            const int e = tid + j * CHUNK_NT;
            pre[j] = e < ne ? ldg(src + e) : czero<T>();
        }
    };
    prefetch(blockIdx.x);
    for (int64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        const int64_t i30 = c * cpc;
        const int nb = (int)(n3 - i30 < cpc ? n3 - i30 : cpc);
        const int ne_out = nb * n1 * d_out;
        int ne_in;
        const T *src = chunk_in(c, ne_in);
#pragma unroll
        for (int j = 0; j < CHUNK_PF; ++j) {
            const int e = tid + j * CHUNK_NT;
            if (e < ne_in) {
                ire[pad16(e)] = pre[j].x;
                iim[pad16(e)] = pre[j].y;
            }
        }
        for (int e = tid + CHUNK_PF * CHUNK_NT; e < ne_in; e += CHUNK_NT) {
            const T v = ldg(src + e);
            ire[pad16(e)] = v.x;
            iim[pad16(e)] = v.y;
        }
        prefetch(c + gridDim.x);
        // input planes loaded; the previous chunk's output planes are copied out
        __syncthreads();
        const int nf = nb * n1, ng = (nf + 15) >> 4;
        for (int g = wave; g < ng; g += CHUNK_NT / 64) {
            const int f = g * 16 + lr;
            const bool ok = f < nf;
            const int i3l = ok ? f / n1 : 0, i1 = ok ? f - i3l * n1 : 0;
            const int bin = i1 + n1 * d_in * i3l;
            V ar[NT16], ai[NT16];
#pragma unroll
            for (int t = 0; t < NT16; ++t) {
                ar[t] = V{0, 0, 0, 0};
                ai[t] = V{0, 0, 0, 0};
            }
#pragma unroll 1
            for (int kc = 0; kc < NT16; ++kc) {
                T x[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int b = 16 * kc + 4 * j + lk;
                    if (ok && b < d_in) {
                        const int idx = pad16(bin + n1 * b);
                        x[j] = mk(ire[idx], iim[idx]);
                    } else {
                        x[j] = czero<T>();
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int t = 0; t < NT16; ++t)
                        cmma4<R>(Fs[(16 * t + lr) + (16 * kc + 4 * j + lk) * LDF], x[j], ar[t], ai[t]);
                }
            }
            if (ok) {
                const int bout = i1 + n1 * d_out * i3l;
#pragma unroll
                for (int t = 0; t < NT16; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int a = 16 * t + mf<R>::row(lane, r);
                        if (a < d_out) {
                            const int idx = pad16(bout + n1 * a);
                            ore[idx] = ar[t][r];
                            oim[idx] = ai[t][r];
                        }
                    }
                }
            }
        }
        // output planes complete; every wave is done reading the input planes
        __syncthreads();
        T *dst = out + i30 * n1 * d_out;
        for (int e = tid; e < ne_out; e += CHUNK_NT) {
            T v = cmul(alpha, mk(ore[pad16(e)], oim[pad16(e)]));
            if (!beta_zero) v = cfma(beta, dst[e], v);
            st_stream(dst + e, v);
        }
    }
}

// --------------------------------------------------------------- k_zgemm
// C[m, n] = alpha * sum_k A[m, k] B[k, n] + beta * C[m, n] for every batch
// index z, with element (m, k) of A at A + z sa + m sam + k sak, (k, n) of B
// at B + z sb + k sbk + n sbn, (m, n) of C at C + z sc + m scm + n scn.
// Tiles of BM x BN outputs, K in chunks of 16 through two LDS buffers.  Four
// waves in a 2 x 2 grid; the MFMA rows run along n and its columns (lane % 16)
// along m, so a C column with scm = 1 is stored as 16-element runs.
//
// Bound by the MFMA rate.  A wave issues in order, so whatever it issues
// between its MFMAs and does not overlap costs matrix time:
//   - LDS rows hold interleaved complex elements and are BM + 1 long: a chunk
//     whose threads run along k is staged without bank conflicts (separate
//     real and imaginary planes with 64 + 16 columns: 8-way conflicts, a
//     third of the kernel), and one 16-byte read gives a fragment's both parts;
//   - a whole chunk costs one pointer addition per load and nothing else
//     (with the bounds checks of the last chunk on every chunk: 64 instead of
//     68 TFLOP/s);
//   - a chunk is staged before the MFMAs of the previous chunk's last k-step;
//   - registers are capped (WPE waves per SIMD), which also keeps the
//     accumulators out of the accumulation registers (the compiler copied
//     them there and back on every chunk).
// Measured (ComplexF64 / ComplexF32, square, against one 64 x 64 tile shape
// with none of these): 4096: 7.64 / 4.22 ms (71.9 / 130 TFLOP/s) from 9.76 /
// 4.69; 3001: 3.21 / 1.76 from 4.05 / 1.97; 1000: 130 / 76 us from 186 / 110;
// 200: 11 / 7.8 us from 40 / 25 (k_zgemm_small since).  Not kept: loads two chunks ahead (no
// change), k split over wave groups of one workgroup (no gain from 64^3 to
// 4096^3), 8 k per chunk, a 64 x 64 tile (1-3% faster above 3000^3 in
// ComplexF32, slower below 2000^3).
constexpr int GNT = 256, GBK = 16, GPAD = 1;

template <typename R, int BM, int BN, int WPE>
__global__ void __launch_bounds__(GNT, WPE) k_zgemm(int64_t M, int64_t N, int64_t K, const cplx<R> *__restrict__ A,
                                               int64_t sam, int64_t sak, int64_t sa, const cplx<R> *__restrict__ B,
                                               int64_t sbk, int64_t sbn, int64_t sb, cplx<R> *__restrict__ C,
                                               int64_t scm, int64_t scn, int64_t sc, int64_t tiles_m, int64_t tiles_n,
                                               double2 alpha_, double2 beta_, int beta_zero) {
    using T = cplx<R>;
    using V = typename mf<R>::v4;
    constexpr int LA = BM + GPAD, LB = BN + GPAD;
    constexpr int BK = GBK, KS = BK / 4;  // k and MFMA k-steps per chunk
    constexpr int AE = BM * BK / GNT, BE = BN * BK / GNT;
    constexpr int TMW = BM / 32, TNW = BN / 32;  // 16 x 16 tiles per wave along m and n
    constexpr int BUF = BK * (LA + LB);          // elements per buffer: A [k][m], then B [k][n]
    extern __shared__ unsigned char lds_raw[];
    T *lds = (T *)lds_raw;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1;
    int64_t bid = blockIdx.x;
    const int64_t tn = bid % tiles_n;
    bid /= tiles_n;
    const int64_t tm = bid % tiles_m, z = bid / tiles_m;
    C += z * sc;
    const int64_t m0 = tm * BM, n0 = tn * BN;
    // Element i of this thread's share of a chunk: (am + i amst, ak + i akst)
    // of A, consecutive threads along the dimension of the smaller stride.
    // Rows past M and columns past N read the last one instead (they only
    // reach outputs that are not stored).
    const bool amf = sam <= sak, bnf = sbn <= sbk;
    const int am = amf ? tid % BM : tid / BK, ak = amf ? tid / BM : tid % BK;
    const int bn = bnf ? tid % BN : tid / BK, bk = bnf ? tid / BN : tid % BK;
    const int amst = amf ? 0 : GNT / BK, akst = amf ? GNT / BM : 0;
    const int bnst = bnf ? 0 : GNT / BK, bkst = bnf ? GNT / BN : 0;
    const T *pa[AE], *pb[BE];
#pragma unroll
    for (int i = 0; i < AE; ++i) {
        const int64_t m = m0 + am + i * amst;
        pa[i] = A + z * sa + (m < M ? m : M - 1) * sam + (ak + i * akst) * sak;
    }
#pragma unroll
    for (int i = 0; i < BE; ++i) {
        const int64_t n = n0 + bn + i * bnst;
        pb[i] = B + z * sb + (n < N ? n : N - 1) * sbn + (bk + i * bkst) * sbk;
    }
    const int64_t stepa = BK * sak, stepb = BK * sbk;
    // The chunk at k0 into registers.  When the whole chunk lies
    // below K nothing but loads and pointer additions is issued; else every
    // load past K takes the operand's first element and is zeroed when it is
    // staged (a load under a branch would be waited for at the branch's end,
    // before the MFMAs it should overlap).
    T ra[AE], rb[BE];
    auto load = [&](auto whole, int64_t k0) {
#pragma unroll
        for (int i = 0; i < AE; ++i) {
            ra[i] = ldg(whole || k0 + ak + i * akst < K ? pa[i] : A);
            pa[i] += stepa;
        }
#pragma unroll
        for (int i = 0; i < BE; ++i) {
            rb[i] = ldg(whole || k0 + bk + i * bkst < K ? pb[i] : B);
            pb[i] += stepb;
        }
    };
    const int wa = ak * LA + am, wast = akst * LA + amst;
    const int wb = BK * LA + bk * LB + bn, wbst = bkst * LB + bnst;
    auto store = [&](auto buf, auto whole, int64_t k0) {
        T *l = lds + buf * BUF;
#pragma unroll
        for (int i = 0; i < AE; ++i)
            l[wa + i * wast] = whole || k0 + ak + i * akst < K ? ra[i] : czero<T>();
#pragma unroll
        for (int i = 0; i < BE; ++i)
            l[wb + i * wbst] = whole || k0 + bk + i * bkst < K ? rb[i] : czero<T>();
    };
    V cr[TNW][TMW], ci[TNW][TMW];
#pragma unroll
    for (int p = 0; p < TNW; ++p)
#pragma unroll
        for (int q = 0; q < TMW; ++q) {
            cr[p][q] = V{0, 0, 0, 0};
            ci[p][q] = V{0, 0, 0, 0};
        }
    const int fa = lk * LA + wm * (BM / 2) + lr, fb = BK * LA + lk * LB + wn * (BN / 2) + lr;
    // fragments of k-step ks of a buffer, read one k-step ahead of the MFMAs
    // that use them
    T af[2][TNW], bf[2][TMW];
    auto frag = [&](auto buf, int ks, int s) {
        const T *l = lds + buf * BUF + 4 * ks * LA, *m = lds + buf * BUF + 4 * ks * LB;
#pragma unroll
        for (int p = 0; p < TNW; ++p) af[s][p] = m[fb + 16 * p];
#pragma unroll
        for (int q = 0; q < TMW; ++q) bf[s][q] = l[fa + 16 * q];
    };
    const int64_t nk = (K + BK - 1) / BK, nfull = K / BK;
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    // Chunk c, in buffer buf = c mod 2.  fast: chunk c + 1 exists and is whole.
    auto chunk = [&](auto buf, auto fast, int64_t c) {
        using Next = std::integral_constant<int, 1 - buf>;
        if (fast || c + 1 < nk) load(fast, (c + 1) * BK);  // in flight during this chunk's MFMAs
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int s = ks & 1;
            if (ks + 1 < KS) {
                frag(buf, ks + 1, s ^ 1);
            } else if (fast || c + 1 < nk) {
                // The next chunk is staged and its first fragments are read
                // before the last k-step's MFMAs, which hide both: the other
                // buffer was last read before the previous barrier, and every
                // read of this one is complete at this barrier.
                store(Next(), fast, (c + 1) * BK);
                __syncthreads();
                frag(Next(), 0, s ^ 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            // the four real products of cmma4, each over all tiles before the
            // next, so that an accumulator's two updates are far apart
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int p = 0; p < TNW; ++p)
#pragma unroll
                    for (int q = 0; q < TMW; ++q) {
                        cr[p][q] = h == 0 ? mf<R>::mma(af[s][p].x, bf[s][q].x, cr[p][q])
                                          : mf<R>::mma(-af[s][p].y, bf[s][q].y, cr[p][q]);
                        ci[p][q] = h == 0 ? mf<R>::mma(af[s][p].x, bf[s][q].y, ci[p][q])
                                          : mf<R>::mma(af[s][p].y, bf[s][q].x, ci[p][q]);
                    }
        }
    };
    load(std::false_type(), 0);
    store(I0(), std::false_type(), 0);
    __syncthreads();
    frag(I0(), 0, 0);
    int64_t c = 0;
    for (; c + 2 < nfull; c += 2) {
        chunk(I0(), std::true_type(), c);
        chunk(I1(), std::true_type(), c + 1);
    }
    if (c + 1 < nfull) chunk(I0(), std::true_type(), c++);
    for (; c < nk; ++c) {
        if (c & 1) chunk(I1(), std::false_type(), c);
        else chunk(I0(), std::false_type(), c);
    }
    const T alpha = mk((R)alpha_.x, (R)alpha_.y), beta = mk((R)beta_.x, (R)beta_.y);
#pragma unroll
    for (int p = 0; p < TNW; ++p)
#pragma unroll
        for (int q = 0; q < TMW; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t n = n0 + wn * (BN / 2) + 16 * p + mf<R>::row(lane, r);
                const int64_t m = m0 + wm * (BM / 2) + 16 * q + lr;
                if (m < M && n < N) {
                    T *c = C + m * scm + n * scn;
                    T v = cmul(alpha, mk((R)cr[p][q][r], (R)ci[p][q][r]));
                    if (!beta_zero) v = cfma(beta, *c, v);
                    *c = v;
                }
            }
}

// ---------------------------------------------------------- k_zgemm_small
// The same product where its tiles would leave most CUs idle: a workgroup has
// one 16 x 16 tile of C, its four waves runs of 16 k of it in turn, with the
// fragments straight from memory.  Bound by load latency: k_zgemm waits for
// about one round trip per 16 k, here a wave has SM_U k-steps of both operands
// in flight and the waves share the k range.  Their partial sums are added
// through LDS in wave order.  Against k_zgemm, ComplexF64 / ComplexF32: (3000, 16,
// 3000) 149 / 99 -> 54 / 34 us, (128, 128, 2000) 80 / 48 -> 34 / 20, 200^3 11.1 /
// 8.0 -> 7.0 / 5.1.  Long k ranges, whose operands leave the caches, gain as much
// or nothing: (128, 128, 10^5) 4.9 / 3.2 -> 1.6 / 1.0 ms, (64, 64, 10^6) 50 / 44
// -> 15 / 12, (400, 400, 10^5) in ComplexF64 4.9 -> 3.4, (500, 500, 10^5) 4.9 -> 4.6.
constexpr int SM_U = 4;
template <typename R>
__global__ void __launch_bounds__(256) k_zgemm_small(int64_t M, int64_t N, int64_t K, const cplx<R> *__restrict__ A,
                                                     int64_t sam, int64_t sak, int64_t sa, const cplx<R> *__restrict__ B,
                                                     int64_t sbk, int64_t sbn, int64_t sb, cplx<R> *__restrict__ C,
                                                     int64_t scm, int64_t scn, int64_t sc, int64_t tiles_m,
                                                     int64_t tiles_n, double2 alpha_, double2 beta_, int beta_zero) {
    using T = cplx<R>;
    using V = typename mf<R>::v4;
    __shared__ T red[4][16 * 17];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lk = lane >> 4;
    int64_t bid = blockIdx.x;
    const int64_t tm = bid % tiles_m;
    bid /= tiles_m;
    const int64_t tn = bid % tiles_n, z = bid / tiles_n;
    const int64_t m0 = tm * 16, n0 = tn * 16;
    // rows past M and columns past N read the last one (they only reach
    // outputs that are not stored)
    const T *a = A + z * sa + (m0 + lr < M ? m0 + lr : M - 1) * sam;
    const T *b = B + z * sb + (n0 + lr < N ? n0 + lr : N - 1) * sbn;
    V cr = V{0, 0, 0, 0}, ci = V{0, 0, 0, 0};
    // a wave's groups of 4 SM_U k at k0, k0 + 16 SM_U, ...: full of them lie
    // inside K and need one address addition per load
    constexpr int G = 4 * SM_U;
    const int64_t k0 = G * wave;
    const int64_t full = K >= k0 + G ? (K - k0 - G) / (4 * G) + 1 : 0;
    const T *pa = a + (k0 + lk) * sak, *pb = b + (k0 + lk) * sbk;
    T x[SM_U], y[SM_U], xn[SM_U], yn[SM_U];
    auto load = [&](T (&x)[SM_U], T (&y)[SM_U]) {
#pragma unroll
        for (int u = 0; u < SM_U; ++u) {
            x[u] = ldg(pa + 4 * u * sak);
            y[u] = ldg(pb + 4 * u * sbk);
        }
    };
    if (full > 0) load(x, y);
    for (int64_t g = 0; g < full; ++g) {
        // the last group is loaded once more in place of one that is not there
        pa += g + 1 < full ? 4 * G * sak : 0;
        pb += g + 1 < full ? 4 * G * sbk : 0;
        load(xn, yn);
#pragma unroll
        for (int u = 0; u < SM_U; ++u) cmma4<R>(x[u], y[u], cr, ci);
#pragma unroll
        for (int u = 0; u < SM_U; ++u) {
            x[u] = xn[u];
            y[u] = yn[u];
        }
    }
    const int64_t kt = k0 + 4 * G * full;
    if (kt < K) {  // k past K reads the last one as a zero
#pragma unroll
        for (int u = 0; u < SM_U; ++u) {
            const int64_t k = kt + 4 * u + lk, kc = k < K ? k : K - 1;
            x[u] = ldg(a + kc * sak);
            y[u] = ldg(b + kc * sbk);
        }
#pragma unroll
        for (int u = 0; u < SM_U; ++u) {
            if (kt + 4 * u + lk >= K) x[u] = y[u] = czero<T>();
            cmma4<R>(x[u], y[u], cr, ci);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][mf<R>::row(lane, r) + 17 * lr] = mk((R)cr[r], (R)ci[r]);
    __syncthreads();
    const int i = tid & 15, j = tid >> 4;
    if (m0 + i < M && n0 + j < N) {
        T s = red[0][i + 17 * j];
        for (int w = 1; w < 4; ++w) s = cadd(s, red[w][i + 17 * j]);
        const T alpha = mk((R)alpha_.x, (R)alpha_.y), beta = mk((R)beta_.x, (R)beta_.y);
        T *o = C + z * sc + (m0 + i) * scm + (n0 + j) * scn;
        *o = axpby(alpha, s, beta, o, beta_zero != 0);
    }
}

// --------------------------------------------------------------- k_zgemv
// A matrix far larger than the caches is read once at the copy rate; below
// about 3000 columns the time is load latency, so the kernels here keep
// several loads of each lane in flight, issued at a valid address where there
// is nothing left to add.  A Ket and a Bra by an n x n matrix, before -> now:
// ComplexF32 803 14.7 -> 11.3 us, 2013 26.1 -> 17.4, 6143 125 -> 114;
// ComplexF64 2013 31.2 -> 26.1, 3009 63.9 -> 53.0.
constexpr int GV_U = 8;

// part[s][i] = sum over the columns j of split s of F[i, j] x[j]; with one
// split the result goes straight to y (y = alpha part + beta y).  A
// workgroup covers 64 rows (one row per lane, so every column of F is read as
// a 1 KiB run); its 4 waves take every 4th column of the split; the wave
// partials are summed in LDS in wave order.
constexpr int GV_NT = 256;
template <typename R>
__global__ void __launch_bounds__(GV_NT) k_zgemv(const cplx<R> *__restrict__ F, int64_t m, int64_t n,
                                                 const cplx<R> *__restrict__ x, int64_t split_len,
                                                 cplx<double> *__restrict__ part, cplx<R> *__restrict__ y,
                                                 double2 alpha_, double2 beta_, int beta_zero) {
    using T = cplx<R>;
    __shared__ T red[GV_NT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t i = (int64_t)blockIdx.x * 64 + lane;
    const int64_t j0 = (int64_t)blockIdx.y * split_len;
    const int64_t j1 = j0 + split_len < n ? j0 + split_len : n;
    T acc = czero<T>();
    const T *Fi = F + (i < m ? i : m - 1);
    int64_t j = j0 + wave;
    for (; j + 4 * (GV_U - 1) < j1; j += 4 * GV_U) {
        T f[GV_U];
#pragma unroll
        for (int u = 0; u < GV_U; ++u) f[u] = Fi[(j + 4 * u) * m];
#pragma unroll
        for (int u = 0; u < GV_U; ++u) acc = cfma(f[u], x[j + 4 * u], acc);
    }
    if (j < j1) {
        T f[GV_U];
#pragma unroll
        for (int u = 0; u < GV_U; ++u) f[u] = Fi[(j + 4 * u < j1 ? j + 4 * u : j) * m];
#pragma unroll
        for (int u = 0; u < GV_U; ++u)
            if (j + 4 * u < j1) acc = cfma(f[u], x[j + 4 * u], acc);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    if (wave == 0 && i < m) {
        T s = red[lane];
        s = cadd(s, red[64 + lane]);
        s = cadd(s, red[128 + lane]);
        s = cadd(s, red[192 + lane]);
        if (gridDim.y == 1) {
            const T alpha = mk((R)alpha_.x, (R)alpha_.y), beta = mk((R)beta_.x, (R)beta_.y);
            y[i] = axpby(alpha, s, beta, y + i, beta_zero != 0);
        } else {
            part[(int64_t)blockIdx.y * m + i] = mk((double)s.x, (double)s.y);
        }
    }
}

// y[i] = alpha * sum_s part[s][i] + beta * y[i]: 32 rows per workgroup, eight
// runs of splits per row, each in order, their sums added in order.
template <typename R>
__global__ void __launch_bounds__(256) k_zgemv_sum(const cplx<double> *__restrict__ part, int nsplit, int64_t m,
                                                   cplx<R> *__restrict__ y, double2 alpha_, double2 beta_,
                                                   int beta_zero) {
    using T = cplx<R>;
    __shared__ double2 red[256];
    const int r = threadIdx.x & 31, q = threadIdx.x >> 5;
    const int64_t i = (int64_t)blockIdx.x * 32 + r;
    const double2 *p = part + (i < m ? i : m - 1);
    const int k0 = (int)((int64_t)nsplit * q / 8), k1 = (int)((int64_t)nsplit * (q + 1) / 8);
    double2 s = make_double2(0, 0);
    for (int k = k0; k < k1; k += 4) {
        double2 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = p[(int64_t)min(k + u, k1 - 1) * m];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (k + u < k1) s = cadd(s, v[u]);
    }
    red[threadIdx.x] = s;
    __syncthreads();
    if (q == 0 && i < m) {
        for (int k = 1; k < 8; ++k) s = cadd(s, red[32 * k + r]);
        const T alpha = mk((R)alpha_.x, (R)alpha_.y), beta = mk((R)beta_.x, (R)beta_.y);
        y[i] = axpby(alpha, mk((R)s.x, (R)s.y), beta, y + i, beta_zero != 0);
    }
}

// The same in one launch: a workgroup covers 16 rows, lane l of wave w row
// l % 16 and the columns 4 w + l / 16 + 64 t (runs of 16 rows).  The 64
// partial sums of a row are added in FP64, in column order within a wave: a
// lane's run in the element type is at most 24 products (zgemv_in_one), as
// long as the split kernel's.
template <typename R>
__global__ void __launch_bounds__(1024) k_zgemv_one(const cplx<R> *__restrict__ F, int64_t m, int64_t n,
                                                    const cplx<R> *__restrict__ x, cplx<R> *__restrict__ y,
                                                    double2 alpha_, double2 beta_, int beta_zero) {
    using T = cplx<R>;
    __shared__ double2 red[16][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15;
    const int64_t i = (int64_t)blockIdx.x * 16 + r;
    const T *Fi = F + (i < m ? i : m - 1);
    T acc = czero<T>();
    for (int64_t j = wave * 4 + (lane >> 4); j < n; j += 64 * GV_U) {
        T f[GV_U], v[GV_U];
#pragma unroll
        for (int u = 0; u < GV_U; ++u) {
            const int64_t jj = j + 64 * u < n ? j + 64 * u : j;
            f[u] = Fi[jj * m];
            v[u] = x[jj];
        }
#pragma unroll
        for (int u = 0; u < GV_U; ++u)
            if (j + 64 * u < n) acc = cfma(f[u], v[u], acc);
    }
    double2 s = make_double2(acc.x, acc.y);
    for (int o = 16; o <= 32; o <<= 1) {
        s.x += __shfl_xor(s.x, o, 64);
        s.y += __shfl_xor(s.y, o, 64);
    }
    if (lane < 16) red[wave][r] = s;
    __syncthreads();
    if (threadIdx.x < 16 && i < m) {
        for (int k = 1; k < 16; ++k) s = cadd(s, red[k][r]);
        const T alpha = mk((R)alpha_.x, (R)alpha_.y), beta = mk((R)beta_.x, (R)beta_.y);
        y[i] = axpby(alpha, mk((R)s.x, (R)s.y), beta, y + i, beta_zero != 0);
    }
}

// y[i] = alpha * sum_l A[l + i k] x[l] + beta * y[i] (y = A^T x for a
// column-major k x m A): one wave per output, lanes along the column (1 KiB
// runs), U loads of each in flight, then a butterfly sum over the wave in a
// fixed order.  A load is VL elements: 16 bytes, one complex double or two complex
// floats (8-byte aligned in a matrix of odd height; ComplexF32 6143 65.8 ->
// 51.1 us, 7389 95.7 -> 75.9, 2013 unchanged.  The same for k_zgemv: 6143 58.4 ->
// 55.2, but 8192 92 -> 99, not kept), or one complex float of a short column.
typedef float gv_f4 __attribute__((ext_vector_type(4), aligned(8)));
__device__ __forceinline__ void gv_load(const double2 *p, double2 (&v)[1]) { v[0] = *p; }
__device__ __forceinline__ void gv_load(const float2 *p, float2 (&v)[1]) { v[0] = *p; }
__device__ __forceinline__ void gv_load(const float2 *p, float2 (&v)[2]) {
    const gv_f4 w = *(const gv_f4 *)p;
    v[0] = make_float2(w.x, w.y);
    v[1] = make_float2(w.z, w.w);
}
template <typename R, int U, int VL>
__global__ void __launch_bounds__(256) k_zgemv_t(const cplx<R> *__restrict__ A, int64_t k, int64_t m,
                                                 const cplx<R> *__restrict__ x, cplx<R> *__restrict__ y,
                                                 double2 alpha_, double2 beta_, int beta_zero) {
    using T = cplx<R>;
    constexpr int64_t ST = 64 * VL;
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= m) return;
    const T *Ai = A + i * k;
    T acc = czero<T>();
    int64_t b = 0;
    for (; b + ST * U <= k; b += ST * U) {
        T a[U][VL], v[U][VL];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            gv_load(Ai + b + lane * VL + ST * u, a[u]);
            gv_load(x + b + lane * VL + ST * u, v[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < VL; ++e) acc = cfma(a[u][e], v[u][e], acc);
    }
    // what is left of the column, element by element, no loads for runs that
    // start behind its end (uniform)
    if (b < k) {
        T a[U][VL], v[U][VL];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u == 0 || b + ST * u < k) {
#pragma unroll
                for (int e = 0; e < VL; ++e) {
                    const int64_t p = b + ST * u + lane * VL + e, c = p < k ? p : k - 1;
                    a[u][e] = Ai[c];
                    v[u][e] = x[c];
                }
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < VL; ++e)
                if (b + ST * u + lane * VL + e < k) acc = cfma(a[u][e], v[u][e], acc);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        acc.x += __shfl_xor(acc.x, o);
        acc.y += __shfl_xor(acc.y, o);
    }
    if (lane == 0) {
        const T alpha = mk((R)alpha_.x, (R)alpha_.y), beta = mk((R)beta_.x, (R)beta_.y);
        y[i] = axpby(alpha, acc, beta, y + i, beta_zero != 0);
    }
}

// Workgroups of a kernel resident per CU at the given block size and LDS
// (the runtime's occupancy query, cached per kernel and LDS size).
template <typename K> int resident_per_cu(K kfn, int nt, size_t lds) {
    static std::mutex mu;
    static std::map<std::pair<const void *, size_t>, int> cache;
    std::lock_guard<std::mutex> g(mu);
    auto key = std::make_pair((const void *)kfn, lds);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kfn, nt, lds) != hipSuccess || nb < 1) nb = 1;
    cache.emplace(key, nb);
    return nb;
}

// Dynamic LDS above 64 KiB needs the kernel's limit raised once (to the full
// 160 KiB, so later launches with any size are covered).
template <typename K> hipError_t raise_lds(K kfn, size_t bytes) {
    if (bytes <= 64 * 1024) return hipSuccess;
    static std::mutex mu;
    static std::unordered_set<const void *> done;
    std::lock_guard<std::mutex> g(mu);
    if (done.count((const void *)kfn)) return hipSuccess;
    hipError_t e = hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e == hipSuccess) done.insert((const void *)kfn);
    return e;
}

}  // namespace

// 0: automatic (fibre groups for n1 >= 16, LDS chunks below); 1: always the
// tiled GEMM; 2: flat fibre groups for n1 < 16 as well (1 and 2 for tests
// and timing; the LDS chunks measured 2% faster on a (16, 32, 16) chain)
int g_mode_kernel = 0;

int64_t zgemv_splits(int64_t m, int64_t n) {
    if (zgemv_in_one(m, n)) return 1;
    const int64_t rt = (m + 63) / 64;
    int64_t s = 1;
    while (rt * s < 1024 && n / (s * 2) >= 64) s *= 2;
    return s;
}

hipError_t launch_zgemm(qob_dtype dt, int64_t M, int64_t N, int64_t K, const void *A, int64_t sam, int64_t sak,
                        int64_t sa, const void *B, int64_t sbk, int64_t sbn, int64_t sb, void *C, int64_t scm,
                        int64_t scn, int64_t sc, int64_t batch, double2 alpha, double2 beta, hipStream_t s) {
    if (M <= 0 || N <= 0 || batch <= 0) return hipSuccess;
    const int bz = (beta.x == 0.0 && beta.y == 0.0);
    if (K <= 0) {
        // no product: C = beta C, element by element (beta = 0 writes zeros)
        return hipErrorInvalidValue;
    }
#define QOB_ZG(RR, BMV, BNV, WV)                                                                               \
    do {                                                                                                        \
        const int64_t tmn = (M + BMV - 1) / BMV, tnn = (N + BNV - 1) / BNV, nblk = tmn * tnn * batch;           \
        if (nblk > 0x7fffffff) return hipErrorInvalidValue;                                                     \
        const size_t lds = (size_t)2 * GBK * ((BMV + GPAD) + (BNV + GPAD)) * sizeof(cplx<RR>);                  \
        auto k = k_zgemm<RR, BMV, BNV, WV>;                                                                    \
        hipError_t e = raise_lds(k, lds);                                                                       \
        if (e != hipSuccess) return e;                                                                          \
        hipLaunchKernelGGL(k, dim3((unsigned)nblk), dim3(GNT), lds, s, M, N, K, (const cplx<RR> *)A, sam, sak, sa, \
                           (const cplx<RR> *)B, sbk, sbn, sb, (cplx<RR> *)C, scm, scn, sc, tmn, tnn, alpha, beta, bz); \
        return hipGetLastError();                                                                               \
    } while (0)
    const int64_t ncu = device_cu_count();
    // Few 16 x 16 tiles and a k range worth splitting: one tile per workgroup,
    // up to two tiles per CU, in ComplexF64 up to four where A's rows are
    // contiguous (square, k_zgemm / k_zgemm_small: ComplexF64 200 11.1 / 6.6 us,
    // 350 18.1 / 11.0, 400 (625 tiles) 19.8 / 15.9, 500 24.5 / 22.4, but A
    // transposed 512 23.7 / 34.3; ComplexF32 200 8.0 / 5.0, 350 13.9 / 8.7, 400
    // 14.8 / 15.0, 512 17.2 / 22.4; (350, 350, 64) in ComplexF32 4.7 / 6.3, so
    // short ranges only where half of the CUs would have no tile).
    const int64_t t16m = (M + 15) / 16, t16n = (N + 15) / 16, t16 = t16m * t16n * batch;
    const int64_t most = (dt == QOB_C64 && sam <= sak ? 4 : 2) * ncu;
    if (t16 <= most && (K >= 128 || 2 * t16 <= ncu)) {
#define QOB_ZS(RR)                                                                                                  \
    hipLaunchKernelGGL(k_zgemm_small<RR>, dim3((unsigned)t16), dim3(256), 0, s, M, N, K, (const cplx<RR> *)A, sam,  \
                       sak, sa, (const cplx<RR> *)B, sbk, sbn, sb, (cplx<RR> *)C, scm, scn, sc, t16m, t16n, alpha,  \
                       beta, bz)
        if (dt == QOB_C64) QOB_ZS(double);
        else QOB_ZS(float);
#undef QOB_ZS
        return hipGetLastError();
    }
    // Tile: a launch takes about (rounds of tiles over the CUs) x (tile area),
    // the 32 x 32 tile at 0.92 of the 64 x 32 tile's rate (68 against 72
    // TFLOP/s at 4096^3 in ComplexF64).  With few tiles per CU the smaller
    // one also keeps more waves in flight (700^3: 52 against 58 us).
    const int64_t nl = ((M + 63) / 64) * ((N + 31) / 32) * batch, ns = ((M + 31) / 32) * ((N + 31) / 32) * batch;
    // A launch has less than 2^32 threads: more tiles go in two halves (of the
    // batch, of C's columns or of its rows).
    if (ns > 0xffffffffll / GNT && ns <= 0x7fffffff) {
        const size_t es = dt == QOB_C64 ? sizeof(double2) : sizeof(float2);
        auto at = [&](const void *p, int64_t e) { return (void *)((char *)p + e * (int64_t)es); };
        auto part = [&](int64_t m, int64_t n, int64_t z, int64_t m0, int64_t n0, int64_t z0) {
            return launch_zgemm(dt, m, n, K, at(A, z0 * sa + m0 * sam), sam, sak, sa, at(B, z0 * sb + n0 * sbn), sbk, sbn,
                                sb, at(C, z0 * sc + m0 * scm + n0 * scn), scm, scn, sc, z, alpha, beta, s);
        };
        const int64_t hz = batch / 2, hn = (N / 2 + 31) / 32 * 32, hm = (M / 2 + 31) / 32 * 32;
        hipError_t e;
        if (batch > 1) {
            e = part(M, N, hz, 0, 0, 0);
            return e != hipSuccess ? e : part(M, N, batch - hz, 0, 0, hz);
        }
        if (N >= M) {
            e = part(M, hn, 1, 0, 0, 0);
            return e != hipSuccess ? e : part(M, N - hn, 1, 0, hn, 0);
        }
        e = part(hm, N, 1, 0, 0, 0);
        return e != hipSuccess ? e : part(M - hm, N, 1, hm, 0, 0);
    }
    const int64_t rl = (nl + ncu - 1) / ncu, rs = (ns + ncu - 1) / ncu;
    const bool large = rl > 2 && 200 * rl < 109 * rs;
    if (dt == QOB_C64) {
        if (large) QOB_ZG(double, 64, 32, 3);
        QOB_ZG(double, 32, 32, 4);
    }
    if (large) QOB_ZG(float, 64, 32, 3);
    QOB_ZG(float, 32, 32, 4);
#undef QOB_ZG
}

hipError_t launch_zgemv(qob_dtype dt, const void *F, int64_t m, int64_t n, const void *x, void *y, void *part,
                        double2 alpha, double2 beta, hipStream_t s) {
    if (m <= 0) return hipSuccess;
    const int bz = (beta.x == 0.0 && beta.y == 0.0);
    if (zgemv_in_one(m, n)) {
        const unsigned g = (unsigned)((m + 15) / 16);
        if (dt == QOB_C64)
            hipLaunchKernelGGL(k_zgemv_one<double>, dim3(g), dim3(1024), 0, s, (const double2 *)F, m, n,
                               (const double2 *)x, (double2 *)y, alpha, beta, bz);
        else
            hipLaunchKernelGGL(k_zgemv_one<float>, dim3(g), dim3(1024), 0, s, (const float2 *)F, m, n,
                               (const float2 *)x, (float2 *)y, alpha, beta, bz);
        return hipGetLastError();
    }
    const int64_t ns = zgemv_splits(m, n);
    const int64_t len = (n + ns - 1) / ns;
    if (ns > 1 && !part) return hipErrorInvalidValue;
    dim3 g((unsigned)((m + 63) / 64), (unsigned)ns), gs((unsigned)((m + 31) / 32));
    if (dt == QOB_C64) {
        hipLaunchKernelGGL(k_zgemv<double>, g, dim3(GV_NT), 0, s, (const double2 *)F, m, n, (const double2 *)x, len,
                           (double2 *)part, (double2 *)y, alpha, beta, bz);
        if (ns > 1)
            hipLaunchKernelGGL(k_zgemv_sum<double>, gs, dim3(256), 0, s, (const double2 *)part, (int)ns, m,
                               (double2 *)y, alpha, beta, bz);
    } else {
        hipLaunchKernelGGL(k_zgemv<float>, g, dim3(GV_NT), 0, s, (const float2 *)F, m, n, (const float2 *)x, len,
                           (double2 *)part, (float2 *)y, alpha, beta, bz);
        if (ns > 1)
            hipLaunchKernelGGL(k_zgemv_sum<float>, gs, dim3(256), 0, s, (const double2 *)part, (int)ns, m,
                               (float2 *)y, alpha, beta, bz);
    }
    return hipGetLastError();
}

hipError_t launch_zgemv_t(qob_dtype dt, const void *A, int64_t k, int64_t m, const void *x, void *y, double2 alpha,
                          double2 beta, hipStream_t s) {
    if (m <= 0) return hipSuccess;
    const int bz = (beta.x == 0.0 && beta.y == 0.0);
    const unsigned g = (unsigned)((m + 3) / 4);
#define QOB_GT(RR, U, VL)                                                                                    \
    hipLaunchKernelGGL((k_zgemv_t<RR, U, VL>), dim3(g), dim3(256), 0, s, (const cplx<RR> *)A, k, m,          \
                       (const cplx<RR> *)x, (cplx<RR> *)y, alpha, beta, bz)
    const GemvT f = zgemv_t_form(dt == QOB_C64, k, m);
    if (dt == QOB_C64) {
        if (f.loads == 1) QOB_GT(double, 1, 1);
        else QOB_GT(double, 4, 1);
    } else {
        if (f.elems == 1) QOB_GT(float, 1, 1);
        else if (f.loads == 1) QOB_GT(float, 1, 2);
        else QOB_GT(float, 4, 2);
    }
#undef QOB_GT
    return hipGetLastError();
}

// chunk of i3 blocks for k_mode_chunk: up to 32 KiB of planes (in + out),
// at least one block, and where that fits a whole number of fibre groups
// per wave (4 waves), else of single fibre groups
static int mode_chunk_blocks(int64_t n1, int64_t d_in, int64_t d_out, size_t esz) {
    const int64_t per = n1 * (d_in + d_out) * 2 * (int64_t)esz;  // plane bytes per i3 block
    int64_t c = std::max<int64_t>(1, (32 * 1024) / std::max<int64_t>(per, 1));
    const int64_t uw = 64 / std::gcd<int64_t>(n1, 64), u1 = 16 / std::gcd<int64_t>(n1, 16);
    if (c >= uw) c -= c % uw;
    else if (c >= u1) c -= c % u1;
    return (int)c;
}

size_t mode_workspace_bytes(int64_t d_out, int64_t d_in, int64_t n1, int64_t n3) {
    if (n1 == 1 && n3 == 1) {
        const int64_t ns = zgemv_splits(d_out, d_in);
        return ns > 1 ? (size_t)(ns * d_out) * 16 : 0;
    }
    return 0;
}

hipError_t launch_mode(qob_dtype dt, const void *F, int64_t d_out, int64_t d_in, const void *in, void *out,
                       int64_t n1, int64_t n3, double2 alpha, double2 beta, hipStream_t s, void *ws) {
    if (n1 <= 0 || n3 <= 0 || d_out <= 0) return hipSuccess;
    if (d_in <= 0) return hipErrorInvalidValue;
    const bool small = d_in <= 64 && d_out <= 64 && g_mode_kernel != 1;
    if (n1 == 1 && n3 == 1 && g_mode_kernel != 1) return launch_zgemv(dt, F, d_out, d_in, in, out, ws, alpha, beta, s);
    if (!small) {
        if (n1 == 1)  // out (d_out x n3) = F in
            return launch_zgemm(dt, d_out, n3, d_in, F, 1, d_out, 0, in, 1, d_in, 0, out, 1, d_out, 0, 1, alpha,
                                beta, s);
        if (n1 >= 64 || n3 == 1)  // per i3: out_i3 (n1 x d_out) = in_i3 (n1 x d_in) F^T
            return launch_zgemm(dt, n1, d_out, d_in, in, 1, n1, n1 * d_in, F, d_out, 1, 0, out, 1, n1, n1 * d_out,
                                n3, alpha, beta, s);
        // per i1: out[i1, :, :] (d_out x n3, strided) = F in[i1, :, :]
        return launch_zgemm(dt, d_out, n3, d_in, F, 1, d_out, 0, in, n1, n1 * d_in, 1, out, n1, n1 * d_out, 1, n1,
                            alpha, beta, s);
    }
    const int bz = (beta.x == 0.0 && beta.y == 0.0);
    const int nt16 = (int)((std::max(d_in, d_out) + 15) / 16);
    const size_t esz = dt == QOB_C64 ? 8 : 4;
    const size_t fbytes = (size_t)(4 * 4 * nt16) * (16 * nt16 + 1) * 2 * esz;
    const int ncu = device_cu_count();
    if (n1 >= 16 || g_mode_kernel == 2) {
        // n1 >= 16: groups of 16 consecutive i1; else of 16 consecutive fibres
        const int flat = n1 < 16;
        const int64_t nf = n1 * n3;
        const int64_t gpi = (n1 + 15) / 16, ng = flat ? (nf + 15) / 16 : gpi * n3;
#define QOB_MF(RR, NT)                                                                                          \
    do {                                                                                                        \
        auto k = k_mode_fib<RR, NT>;                                                                            \
        hipError_t e = raise_lds(k, fbytes);                                                                    \
        if (e != hipSuccess) return e;                                                                          \
        const int64_t grid = std::max<int64_t>(                                                                 \
            1, std::min<int64_t>((ng + 7) / 8, (int64_t)ncu * resident_per_cu(k, MODE_NT, fbytes)));           \
        hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(MODE_NT), fbytes, s, (const cplx<RR> *)F, (int)d_out, \
                           (int)d_in, (const cplx<RR> *)in, (cplx<RR> *)out, (int)n1, (int)gpi, ng, nf, alpha, beta, \
                           bz, flat);                                                                          \
        return hipGetLastError();                                                                               \
    } while (0)
        if (n1 > 0x7fffffff) return hipErrorInvalidValue;
        if (dt == QOB_C64) {
            if (nt16 == 1) QOB_MF(double, 1);
            if (nt16 == 2) QOB_MF(double, 2);
            if (nt16 == 3) QOB_MF(double, 3);
            QOB_MF(double, 4);
        } else {
            if (nt16 == 1) QOB_MF(float, 1);
            if (nt16 == 2) QOB_MF(float, 2);
            if (nt16 == 3) QOB_MF(float, 3);
            QOB_MF(float, 4);
        }
#undef QOB_MF
    }
    const int cpc = mode_chunk_blocks(n1, d_in, d_out, esz);
    const int64_t nch = (n3 + cpc - 1) / cpc;
    const size_t pin = (size_t)(cpc * n1 * d_in + ((cpc * n1 * d_in) >> 4) + 1);
    const size_t pout = (size_t)(cpc * n1 * d_out + ((cpc * n1 * d_out) >> 4) + 1);
    const size_t lds = fbytes + 2 * (pin + pout) * esz;
    if (lds > 160 * 1024) return hipErrorInvalidValue;
#define QOB_MC(RR, NT)                                                                                        \
    do {                                                                                                      \
        auto k = k_mode_chunk<RR, NT>;                                                                        \
        hipError_t e = raise_lds(k, lds);                                                                     \
        if (e != hipSuccess) return e;                                                                        \
        const int64_t grid =                                                                                  \
            std::max<int64_t>(1, std::min<int64_t>(nch, (int64_t)ncu * resident_per_cu(k, CHUNK_NT, lds)));   \
        hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(CHUNK_NT), lds, s, (const cplx<RR> *)F, (int)d_out,  \
                           (int)d_in, (const cplx<RR> *)in, (cplx<RR> *)out, (int)n1, n3, cpc, nch, alpha, beta, bz); \
        return hipGetLastError();                                                                             \
    } while (0)
    if (dt == QOB_C64) {
        if (nt16 == 1) QOB_MC(double, 1);
        if (nt16 == 2) QOB_MC(double, 2);
        if (nt16 == 3) QOB_MC(double, 3);
        QOB_MC(double, 4);
    } else {
        if (nt16 == 1) QOB_MC(float, 1);
        if (nt16 == 2) QOB_MC(float, 2);
        if (nt16 == 3) QOB_MC(float, 3);
        QOB_MC(float, 4);
    }
#undef QOB_MC
}

}  // namespace qob
