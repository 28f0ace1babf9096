// Lindhard response of the ScreenedPotential application on the device:
// ScreenedPotential::ResponseFunction (src/Screened_potential/Screened_potential.cpp:17-58)
//
//   X_ab(q) = 1/Nk sum_k sum_{v < nf <= c}
//             U_k(a,v) U_k'(b,c) conj(U_k'(a,c)) conj(U_k(b,v)) / (e_v(k) - e_c(k'))
//
// with k' = k + q on the periodic mesh (MeshGrid::find, MeshGrid.cpp:282-297),
// U_k the eigenvectors in columns (ascending bands) and e the band energies.
// Writing A_v(k)_ab = U_k(a,v) conj(U_k(b,v)) and B_c(k')_ab = conj(U_k'(a,c)) U_k'(b,c),
//
//   X_ab(q) = 1/Nk sum_k sum_c B_c(k+q)_ab sum_v r_vc(k, k+q) A_v(k)_ab,
//   r_vc(k, k') = 1 / (e_v(k) - e_c(k')).
//
// O(Nk^2) pairs (q, k) with O(nb^2 nv nc) FP64 work each: the kernels are bound
// by the FP64 pipes and what feeds them, not by HBM.  Two forms follow: this
// one on the vector pipes, elementwise in (a, b), and one that takes the sum
// over v on the matrix cores (below); lindhard_mfma_shape chooses.  Mapping of
// the vector form:
//   * a split pass stores the valence columns of every U_k as Uv[k][v][a]
//     and the conduction columns as planes Uc[c nb + a][k], so that a step's
//     valence block is one contiguous run and the conduction elements of the
//     consecutive k + q of a work-group are adjacent;
//   * one work-group = W waves; each lane owns one element pair (a, b) (the
//     upper triangle when that packs the lanes better, the lower triangle
//     then follows from X_ba(q) = conj X_ab(q)), for G q-groups per wave when
//     the pairs fit G times in 64 lanes (W = 1), or spread over the W waves of
//     the work-group when they need more than 64 lanes (G = 1); the waves
//     share the staged columns and reciprocals;
//   * the work-group's GT = G * TQ q lie on one grid row at consecutive q1,
//     so for every k their k + q are consecutive on one row: per k the
//     work-group copies Uv(k) and the conduction columns of the k + q
//     straight from memory into LDS (global_load_lds, no registers),
//     double-buffered: step k + 1 is in flight while step k is computed;
//   * the reciprocals r_vc of each (q, k) are formed once per work-group,
//     from energies loaded into registers one step ahead, into one of two
//     tables, and read by all lanes of that q (one address for all:
//     broadcast); one barrier per k publishes both the columns and the
//     table; A_v(k) is built once per k in registers and used for all TQ q
//     of a lane;
//   * work-groups of neighbouring q go to the same XCD: their Uc(k + q)
//     windows overlap and stay in that XCD's L2;
//   * when the q-blocks would leave the last round of resident work-groups
//     mostly empty, each block's k range is split in two and the partial sums
//     are added into a zeroed X (0 + p1 + p2 is the same in either order).
// The summation order differs from the reference's (k outermost over pairs
// of bands, r multiplied instead of divided), so results agree to rounding,
// not bit for bit.
#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <stdexcept>
#include <vector>

#include "../../../include/edus_gpu.h"
#include "common.hpp"
#include "engine_internal.hpp"
#include "kernels.hpp"

namespace edus {

namespace {

constexpr int kLindStageR = 4;  // reciprocals formed per thread per k
constexpr int kLindGatherU = 8;  // conduction-column elements gathered per thread per k
typedef double dbl4 __attribute__((ext_vector_type(4)));

struct LindhardArgs {
    const double2* Uv;  // [Nk][nv][nb]: U_k(a, v) at (k nv + v) nb + a
    const double2* Uc;  // planes [nc * nb][Nk]: U_k(a, nv + c) at (c nb + a) Nk + k
    const double* eps;  // [Nk][nb]
    double2* X;         // planes [nb * nb][Nk]
    int nb, nv, nc, N0, N1, Nk;
    int Pg;             // element pairs per q
    int G;              // q groups per wave (Pg <= 64), else 1
    int W;              // waves per work-group (Pg > 64), else 1
    int tri;            // pairs are the upper triangle
    int nqb_row;        // q-blocks per grid row
    int KS;             // k-range parts (work-groups per q-block); > 1: partial sums added into X
    int nR;             // reciprocals per k (whole work-group)
    int nvp;            // nv rounded up to even (reciprocal row length)
    int buf;            // one LDS buffer, in double2
    double inv_nk;
};

// pair index i -> (a, b): row-major full list, or the upper triangle a <= b
__device__ inline void pair_of(int i, int nb, int tri, int& a, int& b)
{
    if (!tri) {
        a = i / nb;
        b = i % nb;
        return;
    }
    a = 0;
    while (i >= nb - a) {
        i -= nb - a;
        ++a;
    }
    b = a + i;
}

// U[k][a][n] -> Uv[k][v][a] and the conduction planes Uc[(c nb + a)][k]
__global__ void lindhard_zero_kernel(double2* __restrict__ X, long n)
{
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) X[i] = make_double2(0.0, 0.0);
}

__global__ void lindhard_split_kernel(const double2* __restrict__ U, double2* __restrict__ Uv,
                                      double2* __restrict__ Uc, int nb, int nv, int Nk)
{
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    const long total = long(Nk) * nb * nb;
    if (i >= total) return;
    const int M = nb * nb;
    const long k = i / M;
    const int r = int(i - k * M), al = r / nb, n = r % nb;
    const double2 v = U[i];
    if (n < nv)
        Uv[(k * nv + n) * nb + al] = v;
    else
        Uc[long((n - nv) * nb + al) * Nk + k] = v;
}

// copy count 16-byte elements src[0..count) to LDS dst: wave w of nw takes
// the 64-element chunks w, w + nw, ... (wave-uniform LDS base per chunk)
__device__ inline void copy16(const double2* src, double2* dst, int count, int lane, int w, int nw)
{
    for (int i = 64 * w; i < count; i += 64 * nw)
        if (i + lane < count) __builtin_amdgcn_global_load_lds(src + i + lane, dst + i, 16, 0, 0);
}

template <int NV, int TQ>
__global__ void __launch_bounds__(256) lindhard_kernel(LindhardArgs a)
{
    extern __shared__ double2 lds[];
    constexpr int NVP = (NV + 1) & ~1;
    const int nb = a.nb, nc = a.nc, N1 = a.N1, GT = a.G * TQ;
    // buffer layout (double2 units): Uv(k) [NV][nb]; the conduction columns
    // of the GT slots, slot fastest: [nc][nb][GT].  With the slot fastest,
    // the TQ q of a lane sit at fixed offsets from one address.  After both
    // buffers: two reciprocal tables [nc][GT][NVP] (doubles), one per step
    // parity.
    const int oUc = NV * nb;
    const int nRt = nc * GT * NVP;
    double* sR0 = reinterpret_cast<double*>(lds + 2 * a.buf);

    // XCD-aware order: consecutive logical blocks on one XCD
    long L;
    {
        const long nblk = gridDim.x, q = nblk / 8, r = nblk % 8;
        const long x = blockIdx.x % 8, i = blockIdx.x / 8;
        L = x * q + min(x, r) + i;
    }
    const int qbi = int(L / a.KS), ks = int(L % a.KS);
    const int kb = int(long(a.Nk) * ks / a.KS), ke = int(long(a.Nk) * (ks + 1) / a.KS);
    const int q0 = qbi / a.nqb_row, q1f = (qbi % a.nqb_row) * GT;  // row and first q1 of the block
    const int nvalid = min(GT, N1 - q1f);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = a.W, nthr = 64 * a.W;
    int s, pi;
    if (a.W > 1) {
        s = 0;
        pi = tid;
    } else {
        s = lane / a.Pg;
        pi = lane % a.Pg;
    }
    const bool active = s < a.G && pi < a.Pg;
    int al = 0, be = 0;
    if (active) pair_of(pi, nb, a.tri, al, be);

    // per-thread work lists, fixed for the whole k loop:
    //  reciprocal entries: valence band, slot, conduction band (as a column
    //  of the energy row) and destination in the table
    int rv[kLindStageR], rs[kLindStageR], rc[kLindStageR], rd[kLindStageR];
#pragma unroll
    for (int t = 0; t < kLindStageR; ++t) {
        const int e = tid + nthr * t;
        rv[t] = rs[t] = rc[t] = rd[t] = -1;
        if (e < a.nR && (e / NV) % GT < nvalid) {
            const int c = e / (GT * NV), slot = (e / NV) % GT, v = e % NV;
            rv[t] = v;
            rs[t] = slot;
            rc[t] = NV + c;
            rd[t] = (c * GT + slot) * NVP + v;
        }
    }
    //  gathered conduction-column elements: offset of plane (c nb + a) and slot
    const int nU = nc * nb * GT;
    int gp[kLindGatherU], gs[kLindGatherU];
#pragma unroll
    for (int t = 0; t < kLindGatherU; ++t) {
        const int e = tid + nthr * t;
        gp[t] = gs[t] = -1;
        if (e < nU && e % GT < nvalid) {
            gp[t] = (e / GT) * a.Nk;  // < nb^2 Nk, fits an int for any grid the engine takes
            gs[t] = e % GT;
        }
    }

    // first grid point of row r0 + shift s1 of step (k0, k1)
    auto shift = [&](int k0, int k1, int& row, int& s1) {
        int r0 = k0 + q0;
        if (r0 >= a.N0) r0 -= a.N0;
        s1 = k1 + q1f;
        if (s1 >= N1) s1 -= N1;
        row = r0 * N1;
    };
    // issue the direct copies of step k into buffer b
    auto issue = [&](int k, int k0, int k1, int b) {
        double2* buf = lds + b * a.buf;
        int row, s1;
        shift(k0, k1, row, s1);
        copy16(a.Uv + long(k) * NV * nb, buf, NV * nb, lane, wave, nw);
        // element e = tid + nthr t lands at LDS slot oUc + e: wave-uniform base
        // oUc + nthr t + 64 wave, lane offset 16 bytes
#pragma unroll
        for (int t = 0; t < kLindGatherU; ++t) {
            if (nthr * t >= nU) break;
            if (gp[t] >= 0) {
                int kk = s1 + gs[t];
                if (kk >= N1) kk -= N1;
                __builtin_amdgcn_global_load_lds(a.Uc + (gp[t] + row + kk),
                                                 buf + oUc + nthr * t + 64 * wave, 16, 0, 0);
            }
        }
    };
    // the energies of this thread's reciprocal entries for step k, into registers
    double ev[kLindStageR], ec[kLindStageR];
    auto load_energies = [&](int k, int k0, int k1) {
        int row, s1;
        shift(k0, k1, row, s1);
#pragma unroll
        for (int t = 0; t < kLindStageR; ++t) {
            if (rd[t] >= 0) {
                int kk = s1 + rs[t];
                if (kk >= N1) kk -= N1;
                ev[t] = a.eps[long(k) * nb + rv[t]];
                ec[t] = a.eps[long(row + kk) * nb + rc[t]];
            }
        }
    };
    auto store_reciprocals = [&](double* sR) {
#pragma unroll
        for (int t = 0; t < kLindStageR; ++t)
            if (rd[t] >= 0) sR[rd[t]] = 1.0 / (ev[t] - ec[t]);
    };

    double2 acc[TQ];
#pragma unroll
    for (int j = 0; j < TQ; ++j) acc[j] = make_double2(0.0, 0.0);

    // grid coordinates of the next step to issue, advanced without divisions
    int n0 = kb / N1, n1 = kb - (kb / N1) * N1;
    auto advance = [&]() {
        if (++n1 == N1) {
            n1 = 0;
            ++n0;
        }
    };
    issue(kb, n0, n1, 0);
    load_energies(kb, n0, n1);
    store_reciprocals(sR0);
    advance();
    for (int k = kb; k < ke; ++k) {
        const int par = (k - kb) & 1;
        const double2* buf = lds + par * a.buf;
        const double* sR = sR0 + par * nRt;
        __builtin_amdgcn_s_waitcnt(0);  // this wave's copies of step k are in LDS
        __syncthreads();                // and every lane is done with step k - 1
        const bool next = k + 1 < ke;
        if (next) {
            issue(k + 1, n0, n1, par ^ 1);
            load_energies(k + 1, n0, n1);
            advance();
        }
        if (active) {
            double2 A[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) A[v] = cmul(buf[v * nb + al], cconj(buf[v * nb + be]));
            // c outer, the TQ q inner: TQ independent chains per iteration;
            // the TQ slots of a lane are adjacent in the Uc tile and the
            // reciprocals, so their reads share one address
            const double2* ua = buf + oUc + al * GT + s * TQ;
            const double2* ub = buf + oUc + be * GT + s * TQ;
            const double* rr = sR + s * TQ * NVP;
            for (int c = 0; c < nc; ++c) {
                double2 B[TQ], S[TQ];
#pragma unroll
                for (int j = 0; j < TQ; ++j) B[j] = cmul(cconj(ua[j]), ub[j]);
#pragma unroll
                for (int j = 0; j < TQ; ++j) {
                    const double2* r2 = reinterpret_cast<const double2*>(rr + j * NVP);  // 16-byte aligned
                    S[j] = make_double2(0.0, 0.0);
#pragma unroll
                    for (int v = 0; v < NV; v += 2) {
                        const double2 r = r2[v / 2];
                        S[j].x = fma(r.x, A[v].x, S[j].x);
                        S[j].y = fma(r.x, A[v].y, S[j].y);
                        if (v + 1 < NV) {
                            S[j].x = fma(r.y, A[v + 1].x, S[j].x);
                            S[j].y = fma(r.y, A[v + 1].y, S[j].y);
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < TQ; ++j) {
                    acc[j].x = fma(S[j].x, B[j].x, fma(-S[j].y, B[j].y, acc[j].x));
                    acc[j].y = fma(S[j].x, B[j].y, fma(S[j].y, B[j].x, acc[j].y));
                }
                ua += nb * GT;
                ub += nb * GT;
                rr += GT * NVP;
            }
        }
        // reciprocals of step k + 1 into the other table: its readers finished
        // step k - 1 before this step's barrier; the next barrier publishes it
        if (next) store_reciprocals(sR0 + (par ^ 1) * nRt);
    }

    if (!active) return;
#pragma unroll
    for (int j = 0; j < TQ; ++j) {
        const int q1 = q1f + s * TQ + j;
        if (q1 >= N1) continue;
        const int q = q0 * N1 + q1;
        const double2 x = cscale(acc[j], a.inv_nk);
        double2* x1 = a.X + long(al * nb + be) * a.Nk + q;
        double2* x2 = a.X + long(be * nb + al) * a.Nk + q;
        if (a.KS == 1) {
            *x1 = x;
            if (a.tri && al != be) *x2 = cconj(x);
        } else {
            // two parts onto a zeroed X: 0 + p1 + p2 is the same sum in
            // either order, so the result does not depend on timing
            atomicAdd(&x1->x, x.x);
            atomicAdd(&x1->y, x.y);
            if (a.tri && al != be) {
                atomicAdd(&x2->x, x.x);
                atomicAdd(&x2->y, -x.y);
            }
        }
    }
}

// Work-groups of one launch run in rounds of (resident work-groups per CU) x
// CUs; when the q-blocks leave the last round mostly empty, each q-block's k
// range is split in two (partial sums added into a zeroed X) if that fills
// the rounds better.
template <int NV, int TQ>
void launch_nv(const LindhardArgs& a0, int blocks, size_t lds, hipStream_t s)
{
    LindhardArgs a = a0;
    auto kern = &lindhard_kernel<NV, TQ>;
    int per_cu = 0, dev = 0, ncu = 0;
    EDUS_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kern),
                                                                64 * a.W, lds));
    EDUS_HIP_CHECK(hipGetDevice(&dev));
    EDUS_HIP_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    const long cap = long(std::max(per_cu, 1)) * std::max(ncu, 1);
    auto fill = [&](long n) { return double(n) / double(((n + cap - 1) / cap) * cap); };
    a.KS = (a.Nk >= 64 && fill(2L * blocks) > fill(blocks) + 0.05) ? 2 : 1;
    if (a.KS > 1) {  // a kernel: callers may capture this
        const long n = long(a.nb) * a.nb * a.Nk;
        hipLaunchKernelGGL(lindhard_zero_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, a.X, n);
    }
    hipLaunchKernelGGL(kern, dim3(blocks * a.KS), dim3(64 * a.W), lds, s, a);
}

template <int TQ>
void launch_tq(const LindhardArgs& a, int blocks, size_t lds, hipStream_t s)
{
    switch (a.nv) {
#define EDUS_NV(n) \
    case n: launch_nv<n, TQ>(a, blocks, lds, s); break;
        EDUS_NV(1) EDUS_NV(2) EDUS_NV(3) EDUS_NV(4) EDUS_NV(5) EDUS_NV(6) EDUS_NV(7) EDUS_NV(8)
        EDUS_NV(9) EDUS_NV(10) EDUS_NV(11) EDUS_NV(12) EDUS_NV(13) EDUS_NV(14) EDUS_NV(15)
#undef EDUS_NV
        default: throw EngineError(EDUS_ERR_ARG, "lindhard: filled bands out of range");
    }
}

// ---- the matrix-core form
//
// For one k and the (q, c) rows of 4 consecutive q and 4 conduction bands, the
// inner sum S_c(q)_ab = sum_v r_vc(k, k+q) A_v(k)_ab is a 16 x nv by nv x 16
// real product (real and imaginary part of A) for every 16 element pairs:
// v_mfma_f64_16x16x4.  The FP64 matrix cores and the vector pipes share their
// rate on this chip, so the products cost what they cost in vector FMAs (less
// the padding of nv and nc to multiples of 4); what the matrix form saves is
// LDS bandwidth, which bounds the vector form: there every lane reads every
// r_vc from LDS, here a lane reads one per 16 x 16 products.  Result slot v of
// lane group g is row g + 4 v = (q g, c v), so each lane accumulates X(q)_ab
// over c and k in its own registers.
//   * a work-group takes GT consecutive q of one grid row (and a range of k
//     rows) and walks k along each row: k + q then slides by one point per
//     step, and B_c(k')_ab = conj U_k'(a,c) U_k'(b,c) is formed once per
//     point, into a ring of GT + 1 slots, instead of once per (k, q);
//   * A_v(k) and the reciprocals of step k + 1 are formed from registers loaded
//     one step ahead while step k multiplies; one barrier per step;
//   * units of (4 q, 16 pairs) are dealt to the waves, at most UPW each;
//   * parts of the k range are summed by a second kernel, in a fixed order.
struct LindhardMfmaArgs {
    const double2* U;    // [Nk][nb][nb], bands in columns
    const double* eps;   // [Nk][nb]
    double2* X;          // planes [nb * nb][Nk]
    double2* work;       // another nb * nb planes, for partial sums
    int nb, nv, nc, N0, N1, Nk;
    int P, T;            // element pairs a <= b, tiles of 16
    int GT, KS, nqb_row;
    double inv_nk;
};

// where part ks of the sum for pair p, point q is kept (parts 0 and 1 in the
// first P planes of X and work, part 2 in the planes these leave, P <= 2 (nb^2 - P))
__device__ inline double2* lindhard_part(const LindhardMfmaArgs& a, int ks, int p, int q)
{
    const int left = a.nb * a.nb - a.P;
    if (ks == 0) return a.X + long(p) * a.Nk + q;
    if (ks == 1) return a.work + long(p) * a.Nk + q;
    return (p < left ? a.X + long(a.P + p) * a.Nk : a.work + long(a.P + p - left) * a.Nk) + q;
}

// LDS of the matrix-core kernel: the ring of B, two of A and two tables of r
struct LindhardMfmaLds {
    int ring, A, r;  // entries of one ring slot, one A buffer (double2), one r table (double)
    __host__ __device__ LindhardMfmaLds(int nv, int nc, int T, int GT)
    {
        const int cv = (nv + 3) / 4 * 4, cc = (nc + 3) / 4 * 4;
        ring = nc * 16 * T;
        A = cv * 16 * T;
        r = GT * cc * cv;
    }
    __host__ __device__ int elems(int GT) const { return (GT + 1) * ring + 2 * A + (2 * r + 1) / 2; }
};

// By the numbers of valence and conduction quadruples, for at most NB (8 or 12)
// bands: threads, and products A_v (n = CV) or B_c (n = CC) per thread and step
constexpr int lind_threads(int CV, int CC) { return CV + CC <= 3 ? 256 : 512; }
constexpr int lind_items(int n, int CV, int CC, int NB)
{
    const int nb = 4 * (CV + CC) < NB ? 4 * (CV + CC) : NB, bands = 4 * n < nb ? 4 * n : nb - 1;
    return (nb * (nb + 1) / 2 * bands + lind_threads(CV, CC) - 1) / lind_threads(CV, CC);
}
// Waves per SIMD that the registers leave (116 to 166 at NB = 8, up to 217 at 12).
// Lists sized for 12 bands and a choice of shapes that counted on three waves: 6
// bands, 1 filled, 52 x 52 2362 us; with lists for 8 bands 1538; vector form 1357.
constexpr int lind_waves(int NB) { return NB <= 8 ? 3 : 2; }
// the same as a limit for the compiler (two conduction quadruples: 163 without the
// limit, with it some spill)
constexpr int lind_min_waves(int CC, int NB) { return CC == 2 ? 2 : lind_waves(NB); }

template <int CV, int CC, int UPW, int NBANDS>
__global__ void __launch_bounds__(lind_threads(CV, CC), (lind_min_waves(CC, NBANDS))) lindhard_mfma_kernel(LindhardMfmaArgs a)
{
    constexpr int NT = lind_threads(CV, CC), NA = lind_items(CV, CV, CC, NBANDS), NB = lind_items(CC, CV, CC, NBANDS);
    extern __shared__ double2 lds[];
    const int nb = a.nb, nv = a.nv, nc = a.nc, N0 = a.N0, N1 = a.N1, P = a.P, T = a.T, GT = a.GT;
    const int Pp = 16 * T;
    const LindhardMfmaLds sz(nv, nc, T, GT);
    double2* ring = lds;
    double2* bufA = ring + (GT + 1) * sz.ring;
    double* bufR = reinterpret_cast<double*>(bufA + 2 * sz.A);
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int L = xcd_contiguous_block();
    const int qb = L / a.KS, ks = L - qb * a.KS;
    const int q0 = qb / a.nqb_row, q1f = (qb - q0 * a.nqb_row) * GT;
    const int row_b = N0 * ks / a.KS, row_e = N0 * (ks + 1) / a.KS;
    // padded bands and pairs are zero in every buffer and never written again
    for (int e = tid; e < sz.elems(GT); e += NT) lds[e] = make_double2(0.0, 0.0);

    // products of this thread, A_v(k)_ab = U(a,v) conj U(b,v) and, at the point
    // that enters the window, B_c_ab = conj U(a,c) U(b,c): offsets of the two
    // factors in a point's matrix and of the result in its buffer
    int a1[NA], a2[NA], ad[NA], b1[NB], b2[NB], bd[NB];
    auto items = [&](int bands, int first, auto& o1, auto& o2, auto& od) {
        constexpr int N = sizeof(od) / sizeof(int);
#pragma unroll
        for (int t = 0; t < N; ++t) {
            const int e = tid + t * NT;
            const bool use = e < P * bands;
            const int n = use ? e / P : 0, p = use ? e - n * P : 0;
            int al, be;
            pair_of(p, nb, 1, al, be);
            o1[t] = al * nb + first + n;
            o2[t] = be * nb + first + n;
            od[t] = use ? n * Pp + p : -1;
        }
    };
    items(nv, 0, a1, a2, ad);
    items(nc, nv, b1, b2, bd);
    // reciprocals of this thread: (slot, c, v) of the GT x nc x nv
    constexpr int NR = 2;
    int rv[NR], rc[NR], rs[NR], rd[NR];
#pragma unroll
    for (int t = 0; t < NR; ++t) {
        const int e = tid + t * NT;
        rd[t] = -1;
        rv[t] = rc[t] = rs[t] = 0;
        if (e < GT * nc * nv) {
            rs[t] = e / (nc * nv);
            const int m = e - rs[t] * nc * nv;
            rc[t] = m / nv;
            rv[t] = m - rc[t] * nv;
            rd[t] = (rs[t] * 4 * CC + rc[t]) * 4 * CV + rv[t];
        }
    }
    // the wave's units: q group and tile (a wave with fewer repeats unit 0 and
    // drops the result: no branch between units, whose loads then overlap)
    int uq[UPW], ut[UPW];
    bool uok[UPW];
#pragma unroll
    for (int u = 0; u < UPW; ++u) {
        const int n = wave + u * (NT / 64);
        uok[u] = n < (GT / 4) * T;
        uq[u] = uok[u] ? n / T : 0;
        ut[u] = uok[u] ? n - uq[u] * T : 0;
    }
    double2 acc[UPW];
    int oA[UPW], oR[UPW];  // this lane's operands of the first quadruple in a buffer of A and a table of r
#pragma unroll
    for (int u = 0; u < UPW; ++u) {
        acc[u] = make_double2(0.0, 0.0);
        oA[u] = g * Pp + 16 * ut[u] + i;
        oR[u] = ((4 * uq[u] + (i & 3)) * 4 * CC + (i >> 2)) * 4 * CV + g;
    }
    // offsets of the conduction bands in a ring slot; the bands that pad the
    // last quadruple repeat the last one (their rows of r are zero)
    int oc[4 * CC];
#pragma unroll
    for (int c = 0; c < 4 * CC; ++c) oc[c] = min(c, nc - 1) * Pp;
    const int ring_end = (GT + 1) * sz.ring;

    for (int k0 = row_b; k0 < row_e; ++k0) {
        int r0 = k0 + q0;
        if (r0 >= N0) r0 -= N0;
        const long rowk = long(k0) * N1, rowq = long(r0) * N1;
        if (k0 == row_b) __syncthreads();  // the zeroed buffers
        // the first step's operands: all GT points of the window
        for (int e = tid; e < GT * nc * P; e += NT) {
            const int s = e / (nc * P), m = e - s * (nc * P), c = m / P, p = m - c * P;
            int al, be;
            pair_of(p, nb, 1, al, be);
            const double2* u = a.U + (rowq + (q1f + s) % N1) * nb * nb;
            ring[s * sz.ring + c * Pp + p] = cmul(cconj(u[al * nb + nv + c]), u[be * nb + nv + c]);
        }
#pragma unroll
        for (int t = 0; t < NA; ++t)
            if (ad[t] >= 0) {
                const double2* u = a.U + rowk * nb * nb;
                bufA[ad[t]] = cmul(u[a1[t]], cconj(u[a2[t]]));
            }
#pragma unroll
        for (int t = 0; t < NR; ++t)
            if (rd[t] >= 0)
                bufR[rd[t]] = 1.0 / (a.eps[rowk * nb + rv[t]] - a.eps[(rowq + (q1f + rs[t]) % N1) * nb + nv + rc[t]]);
        __syncthreads();
        // The operands of step k1 + 1 are formed at the start of step k1, from
        // loads issued one step earlier: the loads of step k1 + 2 are in flight
        // while step k1 multiplies.
        int oB[UPW];  // this lane's point in the ring
#pragma unroll
        for (int u = 0; u < UPW; ++u) oB[u] = (4 * uq[u] + g) * sz.ring + 16 * ut[u] + i;
        double2 xa[NA], ya[NA], xb[NB], yb[NB];
        double ev[NR], ec[NR];
        int lk = 1, newc = (q1f + GT) % N1;  // step to load next, and the column that enters the window with it
        int qc[NR];                          // column of each reciprocal's point in that step
#pragma unroll
        for (int t = 0; t < NR; ++t) qc[t] = (q1f + rs[t] + 1) % N1;
        auto load = [&]() {
            if (lk >= N1) return;
            const double2* uk = a.U + (rowk + lk) * nb * nb;
            const double2* un = a.U + (rowq + newc) * nb * nb;
            const double* ek = a.eps + (rowk + lk) * nb;
            const double* eq = a.eps + rowq * nb + nv;
#pragma unroll
            for (int t = 0; t < NA; ++t)
                if (ad[t] >= 0) {
                    xa[t] = uk[unsigned(a1[t])];
                    ya[t] = uk[unsigned(a2[t])];
                }
#pragma unroll
            for (int t = 0; t < NB; ++t)
                if (bd[t] >= 0) {
                    xb[t] = un[unsigned(b1[t])];
                    yb[t] = un[unsigned(b2[t])];
                }
#pragma unroll
            for (int t = 0; t < NR; ++t)
                if (rd[t] >= 0) {
                    ev[t] = ek[unsigned(rv[t])];
                    ec[t] = eq[unsigned(qc[t] * nb + rc[t])];
                    if (++qc[t] >= N1) qc[t] = 0;
                }
            ++lk;
            if (++newc >= N1) newc = 0;
        };
        load();
        int slot = GT * sz.ring;  // the ring slot behind the window, free during a step
        for (int k1 = 0; k1 < N1; ++k1) {
            const int par = k1 & 1;
            if (k1 + 1 < N1) {
                double2* An = bufA + (par ^ 1) * sz.A;
                double2* Bn = ring + slot;
#pragma unroll
                for (int t = 0; t < NA; ++t)
                    if (ad[t] >= 0) An[ad[t]] = cmul(xa[t], cconj(ya[t]));
#pragma unroll
                for (int t = 0; t < NB; ++t)
                    if (bd[t] >= 0) Bn[bd[t]] = cmul(cconj(xb[t]), yb[t]);
                double* Rn = bufR + (par ^ 1) * sz.r;
#pragma unroll
                for (int t = 0; t < NR; ++t)
                    if (rd[t] >= 0) Rn[rd[t]] = 1.0 / (ev[t] - ec[t]);
                slot += sz.ring;
                if (slot >= ring_end) slot = 0;
                load();
            }
            const double2* A = bufA + par * sz.A;
            const double* R = bufR + par * sz.r;
#pragma unroll
            for (int u = 0; u < UPW; ++u) {
                double2 x[CV], b[4 * CC];
                double r[CC][CV];
#pragma unroll
                for (int vc = 0; vc < CV; ++vc) x[vc] = A[oA[u] + 4 * vc * Pp];
#pragma unroll
                for (int cc = 0; cc < CC; ++cc)
#pragma unroll
                    for (int vc = 0; vc < CV; ++vc) r[cc][vc] = R[oR[u] + cc * 16 * CV + 4 * vc];
#pragma unroll
                for (int c = 0; c < 4 * CC; ++c) b[c] = ring[oB[u] + oc[c]];
                dbl4 sr[CC], si[CC];
#pragma unroll
                for (int cc = 0; cc < CC; ++cc) {
                    sr[cc] = si[cc] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int vc = 0; vc < CV; ++vc) {
                        sr[cc] = __builtin_amdgcn_mfma_f64_16x16x4f64(r[cc][vc], x[vc].x, sr[cc], 0, 0, 0);
                        si[cc] = __builtin_amdgcn_mfma_f64_16x16x4f64(r[cc][vc], x[vc].y, si[cc], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int c = 0; c < 4 * CC; ++c) {
                    const double re = sr[c / 4][c % 4], im = si[c / 4][c % 4];
                    acc[u].x = fma(re, b[c].x, fma(-im, b[c].y, acc[u].x));
                    acc[u].y = fma(re, b[c].y, fma(im, b[c].x, acc[u].y));
                }
                oB[u] += sz.ring;
                if (oB[u] >= ring_end) oB[u] -= ring_end;
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int u = 0; u < UPW; ++u) {
        const int p = 16 * ut[u] + i, q1 = q1f + 4 * uq[u] + g;
        if (!uok[u] || p >= P || q1 >= N1) continue;
        const int q = q0 * N1 + q1;
        if (a.KS > 1) {
            *lindhard_part(a, ks, p, q) = acc[u];
            continue;
        }
        int al, be;
        pair_of(p, nb, 1, al, be);
        const double2 x = cscale(acc[u], a.inv_nk);
        a.X[long(al * nb + be) * a.Nk + q] = x;
        if (al != be) a.X[long(be * nb + al) * a.Nk + q] = cconj(x);
    }
}

constexpr int kLindSumQ = 16;  // points per work-group of the sum

// X from the parts of the k range; a work-group reads every part of its points
// before it writes (the parts lie in planes of X)
__global__ void __launch_bounds__(256) lindhard_sum_kernel(LindhardMfmaArgs a)
{
    extern __shared__ double2 lds[];  // [P][kLindSumQ]
    const int qa = blockIdx.x * kLindSumQ;
    for (int e = threadIdx.x; e < a.P * kLindSumQ; e += 256) {
        const int p = e / kLindSumQ, q = qa + e - p * kLindSumQ;
        if (q >= a.Nk) continue;
        double2 x = make_double2(0.0, 0.0);
        for (int ks = 0; ks < a.KS; ++ks) x = cadd(x, *lindhard_part(a, ks, p, q));
        lds[e] = cscale(x, a.inv_nk);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < a.P * kLindSumQ; e += 256) {
        const int p = e / kLindSumQ, q = qa + e - p * kLindSumQ;
        if (q >= a.Nk) continue;
        int al, be;
        pair_of(p, a.nb, 1, al, be);
        a.X[long(al * a.nb + be) * a.Nk + q] = lds[e];
        if (al != be) a.X[long(be * a.nb + al) * a.Nk + q] = cconj(lds[e]);
    }
}

constexpr int kLindMaxUPW = 3;
constexpr size_t kLindMfmaLds = 160 * 1024;

// Whether the vector form is the faster one.  How full it runs the chip goes by
// its waves (one or more per q-block): 4 to 6 per CU in one round are its best
// case, a second round just started its worst; with four q per lane (TQ = 4) any
// large grid fills it.  The matrix form pads the bands of either side to
// quadruples: with one quadruple each it was the faster one at every size, with
// two on one side up to half of its products are padding, and with two on both, or
// 13 bands and more, its registers hold fewer waves than its latency needs.  us,
// vector and matrix form (waves of the vector form):
//   3, 1 filled   64 x 64 (448): 1327, 1168; 72 x 72 (576): 1906, 2153
//   4, 2          56 x 56 (560): 1300, 898; 72 x 72 (864): 2151, 2191
//   6, 3          72 x 72: 3293, 2922        8, 4   48 x 48: 2800, 971
//   6, 5          48 x 48 (768): 922, 921; 52 x 52 (936): 1076, 1385
//   7, 6          48 x 48 (1152): 1106, 925; 52 x 52 (1352): 1309, 1417
//   8, 1          40 x 40 (1600): 1171, 1169; 48 x 48 (2304): 2085, 2200
//   8, 2          42 x 42 (1764): 1411, 1180; 45 x 45 (2025): 1637, 2016; 52 x 52 (2704): 3726, 2518
//   8, 7          32 x 32 (1024): 448, 406; 45 x 26 (1170): 599, 683; 40 x 40 (1600): 1384, 977
//   10, 5         48 x 48: 3582, 3672
//   11, 8         36 x 21 (1512): 533, 576; 28 x 28 (1568): 894, 670; 44 x 44 (3872): 1.31 times
//   12, 11        22 x 18 (792): 241, 282; 45 x 26 (2340): 1.09 times; 42 x 42 (3528): 1.44 times
//   13, 12        24 x 24: 393, 370; 26 x 26: 455, 635
//   14, 5         30 x 30: 1177, 2133        14, 13   40 x 40: 2690, 5432
bool lindhard_vector_better(const LindhardPlan& p)
{
    const int nb = p.nb, nv = p.nv, nc = p.nc;
    const long waves = long(p.blocks) * p.W;
    if (nb < 3 || nb > 12) return true;
    if (nb > 8) return nb <= 10 || nc > 4 || p.TQ != 1 || waves < 1536;
    if (nb <= 4) return p.TQ != 1 || waves >= (nb == 3 ? 512 : 1024);
    if (nv <= 4 && nc <= 4) return false;
    if (p.TQ != 1) return true;
    if (nb == 6) return waves >= 900;
    if (nb == 7) return nc == 1 && waves >= 1300;
    if (nv == 1) return true;
    if (nv == 2) return waves >= 1900 && waves < 2400;
    return nc <= 2 && waves >= 1100 && waves < 1560;
}

// The shape of the matrix-core form, and whether it is used: functions of the
// sizes alone, so that a call under stream capture runs the kernels that it runs
// elsewhere.  Among the window lengths GT that fit, and 1 to 3 parts of the k
// range, the one with the least estimated time: rounds of resident work-groups x
// steps x the longer of a step's FP64 issue time on a SIMD and its latency.
bool lindhard_mfma_shape(const LindhardPlan& p, LindhardMfmaArgs& best)
{
    const int nb = p.nb, nv = p.nv, nc = p.nc, N0 = p.N0, N1 = p.N1;
    if (nv < 1 || nc < 1 || lindhard_vector_better(p)) return false;
    const int P = nb * (nb + 1) / 2, T = (P + 15) / 16, CV = (nv + 3) / 4, CC = (nc + 3) / 4;
    const int nt = lind_threads(CV, CC), W = nt / 64, simd_waves = lind_waves(nb);
    double best_cost = 1e300;
    for (int GT = 4; GT <= 32; GT += 4) {
        const LindhardMfmaLds sz(nv, nc, T, GT);
        const size_t lds = size_t(sz.elems(GT)) * sizeof(double2);
        const int units = (GT / 4) * T, upw = (units + W - 1) / W;
        if (lds > kLindMfmaLds || upw > kLindMaxUPW || GT * nc * nv > 2 * nt) continue;
        const int per_cu = std::max(1, std::min(int(kLindMfmaLds / lds), 4 * simd_waves / W));
        const int blocks = N0 * ((N1 + GT - 1) / GT);
        for (int KS = 1; KS <= 3; ++KS) {
            if (KS > 1 && N0 < 4 * KS) continue;
            const long n = long(blocks) * KS;
            const long rounds = (n + 256L * per_cu - 1) / (256L * per_cu);
            const double resident = std::min<double>(per_cu, double((n + 255) / 256));  // work-groups per CU
            const double unit = 128.0 * CV * CC + 64.0 * CC + 60.0;             // issue cycles of one unit
            const double build = 4.0 * (14.0 * P * nb + 30.0 * GT * nc * nv) / nt;  // per wave
            const double wave = upw * unit + build;
            const double step = std::max(600.0 + wave, resident * W / 4 * wave);
            const double cost = double(rounds) * ((N0 + KS - 1) / KS) * (N1 + 3) * step;
            if (cost < best_cost) {
                best_cost = cost;
                best.GT = GT;
                best.KS = KS;
            }
        }
    }
    if (best_cost >= 1e300) return false;
    best.nb = nb;
    best.nv = nv;
    best.nc = nc;
    best.N0 = N0;
    best.N1 = N1;
    best.Nk = N0 * N1;
    best.P = P;
    best.T = T;
    best.nqb_row = (N1 + best.GT - 1) / best.GT;
    best.inv_nk = 1.0 / double(best.Nk);
    return true;
}

template <int CV, int CC, int UPW, int NB>
void launch_mfma_one(const LindhardMfmaArgs& a, hipStream_t s)
{
    const size_t lds = size_t(LindhardMfmaLds(a.nv, a.nc, a.T, a.GT).elems(a.GT)) * sizeof(double2);
    auto kern = &lindhard_mfma_kernel<CV, CC, UPW, NB>;
    // a first call may be under stream capture: the launch captured there runs with
    // its LDS all the same (checked by replays of 80 KB launches)
    static std::once_flag raised;  // calls may come from several host threads
    std::call_once(raised, [&] {
        EDUS_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, int(kLindMfmaLds)));
    });
    hipLaunchKernelGGL(kern, dim3(a.N0 * a.nqb_row * a.KS), dim3(lind_threads(CV, CC)), lds, s, a);
}

template <int CV, int CC, int NB>
void launch_mfma_upw(const LindhardMfmaArgs& a, hipStream_t s)
{
    const int W = lind_threads(CV, CC) / 64;
    switch (((a.GT / 4) * a.T + W - 1) / W) {
        case 1: launch_mfma_one<CV, CC, 1, NB>(a, s); break;
        case 2: launch_mfma_one<CV, CC, 2, NB>(a, s); break;
        default: launch_mfma_one<CV, CC, kLindMaxUPW, NB>(a, s); break;
    }
}

void launch_lindhard_mfma(const LindhardMfmaArgs& a, hipStream_t s)
{
    switch ((a.nb > 8 ? 64 : 0) + (a.nv + 3) / 4 * 8 + (a.nc + 3) / 4) {  // (those lindhard_vector_better leaves)
        case 1 * 8 + 1: launch_mfma_upw<1, 1, 8>(a, s); break;
        case 1 * 8 + 2: launch_mfma_upw<1, 2, 8>(a, s); break;
        case 2 * 8 + 1: launch_mfma_upw<2, 1, 8>(a, s); break;
        case 64 + 2 * 8 + 1: launch_mfma_upw<2, 1, 12>(a, s); break;
        case 64 + 3 * 8 + 1: launch_mfma_upw<3, 1, 12>(a, s); break;
        default: throw EngineError(EDUS_ERR_STATE, "lindhard: no matrix-core kernel for these bands");
    }
    if (a.KS > 1)
        hipLaunchKernelGGL(lindhard_sum_kernel, dim3((a.Nk + kLindSumQ - 1) / kLindSumQ), dim3(256),
                           size_t(a.P) * kLindSumQ * sizeof(double2), s, a);
    EDUS_HIP_CHECK(hipGetLastError());
}

// waves per q for L element pairs (fractional when several q share a wave)
double waves_per_q(int L) { return L <= 64 ? 1.0 / double(64 / L) : double((L + 63) / 64); }

}  // namespace

LindhardPlan lindhard_plan(int nb, int nf, int N0, int N1)
{
    if (nb < 2 || nb > kMaxNb) throw EngineError(EDUS_ERR_ARG, "lindhard: nb must be in [2, 16]");
    if (nf < 0 || nf > nb) throw EngineError(EDUS_ERR_ARG, "lindhard: filledbands out of range");
    if (N0 < 1 || N1 < 1) throw EngineError(EDUS_ERR_ARG, "lindhard: grid sizes must be positive");
    if (long(nb) * nb * N0 * N1 >= (1L << 31))
        throw EngineError(EDUS_ERR_UNSUPPORTED, "lindhard: nb^2 * Nk must stay below 2^31");
    LindhardPlan p{};
    p.nb = nb;
    p.nv = nf;
    p.nc = nb - nf;
    p.N0 = N0;
    p.N1 = N1;
    p.Nk = N0 * N1;
    const int P = nb * (nb + 1) / 2, M = nb * nb;
    p.tri = waves_per_q(P) < waves_per_q(M) ? 1 : 0;
    p.Pg = p.tri ? P : M;
    p.G = p.Pg <= 64 ? 64 / p.Pg : 1;
    p.W = p.Pg <= 64 ? 1 : (p.Pg + 63) / 64;
    // four q per lane when that keeps >= 1024 waves, wastes under 10% of the
    // slots at the row ends and the per-thread staging lists hold a step;
    // else one (eight measured slower at nb = 14: 220 VGPRs, 2 waves per SIMD)
    if (p.W > 4) throw EngineError(EDUS_ERR_UNSUPPORTED, "lindhard: more than 256 element pairs");
    auto row_blocks = [&](int tq) { return (N1 + p.G * tq - 1) / (p.G * tq); };
    const int nthr = 64 * p.W;
    auto fits = [&](int tq) {
        const int gt = p.G * tq;
        return gt * p.nc * p.nv <= nthr * kLindStageR && p.nc * nb * gt <= nthr * kLindGatherU;
    };
    auto good = [&](int tq) {
        const double fill = double(N1) / double(row_blocks(tq) * p.G * tq);
        return long(N0) * row_blocks(tq) * p.W >= 1024 && fill >= 0.9 && fits(tq);
    };
    p.TQ = good(4) ? 4 : 1;
    const int GT = p.G * p.TQ;
    p.nqb_row = row_blocks(p.TQ);
    p.nR = GT * p.nc * p.nv;
    p.nvp = (p.nv + 1) & ~1;
    p.buf = p.nv * nb + p.nc * nb * GT;
    p.blocks = N0 * p.nqb_row;
    p.lds = size_t(2 * p.buf) * sizeof(double2) + size_t(2 * GT) * p.nc * p.nvp * sizeof(double);
    if (p.nv > 0 && p.nc > 0 && !fits(p.TQ))
        throw EngineError(EDUS_ERR_UNSUPPORTED, "lindhard: a step needs more per-thread staging than the kernel holds");
    return p;
}

size_t lindhard_work_bytes(const LindhardPlan& p) { return size_t(p.Nk) * p.nb * p.nb * sizeof(double2); }

void launch_lindhard(const LindhardPlan& p, const double2* U, const double* eps, double2* work, double2* X,
                     hipStream_t s)
{
    const size_t bytes = size_t(p.nb) * p.nb * p.Nk * sizeof(double2);
    if (p.nv == 0 || p.nc == 0) {  // no valence-conduction pair: X = 0 (a kernel: callers may capture this)
        const long n = long(bytes / sizeof(double2));
        hipLaunchKernelGGL(lindhard_zero_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, X, n);
        EDUS_HIP_CHECK(hipGetLastError());
        return;
    }
    LindhardMfmaArgs m{};
    if (lindhard_mfma_shape(p, m)) {
        m.U = U;
        m.eps = eps;
        m.X = X;
        m.work = work;
        launch_lindhard_mfma(m, s);
        return;
    }
    double2* Uv = work;
    double2* Uc = work + size_t(p.Nk) * p.nv * p.nb;
    const long total = long(p.Nk) * p.nb * p.nb;
    hipLaunchKernelGGL(lindhard_split_kernel, dim3(unsigned((total + 255) / 256)), dim3(256), 0, s, U, Uv, Uc, p.nb,
                       p.nv, p.Nk);
    LindhardArgs a{};
    a.Uv = Uv;
    a.Uc = Uc;
    a.eps = eps;
    a.X = X;
    a.nb = p.nb;
    a.nv = p.nv;
    a.nc = p.nc;
    a.N0 = p.N0;
    a.N1 = p.N1;
    a.Nk = p.Nk;
    a.Pg = p.Pg;
    a.G = p.G;
    a.W = p.W;
    a.tri = p.tri;
    a.nqb_row = p.nqb_row;
    a.nR = p.nR;
    a.nvp = p.nvp;
    a.buf = p.buf;
    a.inv_nk = 1.0 / double(p.Nk);
    if (p.TQ == 4)
        launch_tq<4>(a, p.blocks, p.lds, s);
    else
        launch_tq<1>(a, p.blocks, p.lds, s);
    EDUS_HIP_CHECK(hipGetLastError());
}

}  // namespace edus

extern "C" int edus_lindhard_device(int nb, int N0, int N1, int filledbands, const double* U, const double* eps,
                                    double* work, double* X, void* stream)
{
    EDUS_REQUIRE(U && eps && work && X);
    return edus::guarded([&] {
        const edus::LindhardPlan p = edus::lindhard_plan(nb, filledbands, N0, N1);
        edus::launch_lindhard(p, reinterpret_cast<const double2*>(U), eps, reinterpret_cast<double2*>(work),
                              reinterpret_cast<double2*>(X), static_cast<hipStream_t>(stream));
    });
}

// ---- the Lindhard response without allocation ----------------------------
// Callers that cannot allocate device memory (code under HIP graph capture,
// serving loops) use edus_lindhard_device_noalloc: the band-split copy of U
// that edus_lindhard_device keeps in its `work` argument lives here instead,
// in a fixed array of every GPU the library runs on, held until the process
// ends.  Its device address is taken once per device with
// hipGetSymbolAddress; host code passes that address, never the array's
// name (a host-side stand-in).
namespace edus {
constexpr size_t kLindhardScratchElems = size_t(3) << 20;  // 3,145,728 complex doubles = 48 MiB
static __device__ __align__(256) double2 scratch[kLindhardScratchElems];

namespace {
// address of `scratch` on the current device
double2* scratch_address()
{
    static std::mutex mu;
    static std::map<int, double2*> addr;
    int dev = 0;
    EDUS_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(mu);
    auto it = addr.find(dev);
    if (it != addr.end()) return it->second;
    void* p = nullptr;
    EDUS_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) throw EngineError(EDUS_ERR_HIP, "hipGetSymbolAddress returned no address for the Lindhard scratch");
    addr[dev] = static_cast<double2*>(p);
    return addr[dev];
}
}  // namespace
}  // namespace edus

extern "C" int edus_lindhard_device_noalloc(int nb, int N0, int N1, int filledbands, const double* U,
                                            const double* eps, double* X, void* stream)
{
    EDUS_REQUIRE(U && eps && X);
    return edus::guarded([&] {
        const edus::LindhardPlan p = edus::lindhard_plan(nb, filledbands, N0, N1);
        const size_t need = edus::lindhard_work_bytes(p);
        if (need > edus::kLindhardScratchElems * sizeof(double2))
            throw edus::EngineError(EDUS_ERR_ARG,
                                    "edus_lindhard_device_noalloc: Nk * nb^2 = " +
                                        std::to_string(size_t(p.Nk) * nb * nb) + " exceeds its fixed scratch of " +
                                        std::to_string(edus::kLindhardScratchElems) +
                                        " complex doubles (48 MiB); use edus_lindhard_device with a workspace");
        edus::launch_lindhard(p, reinterpret_cast<const double2*>(U), eps, edus::scratch_address(),
                              reinterpret_cast<double2*>(X), static_cast<hipStream_t>(stream));
    });
}

extern "C" int edus_lindhard(int nb, int N0, int N1, int filledbands, const double* U, const double* eps, double* X)
{
    EDUS_REQUIRE(U && eps && X);
    return edus::guarded([&] {
        const edus::LindhardPlan p = edus::lindhard_plan(nb, filledbands, N0, N1);
        const size_t M = size_t(nb) * nb, Nk = size_t(p.Nk);
        double2 *dU = nullptr, *dX = nullptr, *dW = nullptr;
        double* de = nullptr;
        auto release = [&] {
            (void)hipFree(dU);
            (void)hipFree(dX);
            (void)hipFree(dW);
            (void)hipFree(de);
        };
        try {
            EDUS_HIP_CHECK(hipMalloc(&dU, Nk * M * sizeof(double2)));
            EDUS_HIP_CHECK(hipMalloc(&dX, Nk * M * sizeof(double2)));
            EDUS_HIP_CHECK(hipMalloc(&dW, edus::lindhard_work_bytes(p)));
            EDUS_HIP_CHECK(hipMalloc(&de, Nk * nb * sizeof(double)));
            EDUS_HIP_CHECK(hipMemcpy(dU, U, Nk * M * sizeof(double2), hipMemcpyHostToDevice));
            EDUS_HIP_CHECK(hipMemcpy(de, eps, Nk * nb * sizeof(double), hipMemcpyHostToDevice));
            edus::launch_lindhard(p, dU, de, dW, dX, nullptr);
            std::vector<double2> planes(Nk * M);
            EDUS_HIP_CHECK(hipMemcpy(planes.data(), dX, Nk * M * sizeof(double2), hipMemcpyDeviceToHost));
            // planes [M][Nk] -> [Nk][nb][nb]
            for (size_t h = 0; h < M; ++h)
                for (size_t q = 0; q < Nk; ++q) {
                    X[2 * (q * M + h)] = planes[h * Nk + q].x;
                    X[2 * (q * M + h) + 1] = planes[h * Nk + q].y;
                }
        } catch (...) {
            release();
            throw;
        }
        release();
    });
}
