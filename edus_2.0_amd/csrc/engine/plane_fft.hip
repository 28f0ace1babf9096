// Two-dimensional spectral passes with a whole plane in LDS.
//
// The right-hand side needs, per plane, the derivative
//   D = F^-1 diag(i (c0 R0 + c1 R1)) F rho
// (kGradient_definitions.hpp:35-41 inside Functional_SourceTerm.hpp:20-24),
// with exchange also the convolution T = F^-1[-W o F rho / N]
// (Coulomb.cpp:134-180), and in the Peierls gauge S_A[H] = F^-1 exp(i A.R) F H
// (Simulation.cpp:876-899).  Where a plane fits in the LDS of one CU, one
// work-group does the whole two-dimensional sandwich there: the plane is read
// once and its result written once, in one launch, where the axis passes
// (fft_two.hip, fft_axis.hip) take two to five launches with a plane set
// through memory between each.  With exchange the derivative and the
// convolution of one plane are two work-groups of the same launch.
//
// Every line is n = RA * RB with both factors at most 16, chosen on the host
// (plane_args); the factors are run-time values and each step is dispatched on
// its radix, so that every axis length with such a split shares one kernel.
// Element j = ja RB + jb, frequency k = ka + RA kb:
//   A   DFT_RA over ja, times w^(jb ka), to position ka RB + jb;
//   B   DFT_RB over jb, to position ka RB + kb, which then holds frequency
//       ka + RA kb; the inverse runs B, then A, back to natural order.
// Steps work in place on the plane's array in LDS (a task reads and writes its
// own positions; one barrier between steps).  Axis 0 is outermost: its A step
// loads from memory and its inverse A step stores, coalesced over columns;
// the multiplier is applied between B and its inverse of axis 1, in registers.
// Neighbouring lanes take neighbouring lines: columns are adjacent words, and
// rows are N1 | 1 elements apart, so neither axis has bank conflicts.
//
// What bounds it: a chain of up to seven steps of one plane on one CU, a barrier
// between each and about one round of tasks in a step (90 x 90 with exchange: the
// FP64 operations alone would take 4 of its 19 us, its bytes 5); with fewer planes
// than CUs the chip is partly idle, which the saved launches and passes outweigh.  Measured
// (derivative): 45 x 63, 21 planes 10 us, two Stockham passes 27; 90 x 90 with
// exchange, 64 planes 18.9 us, four axis passes 32; 96 x 96, 784 planes 82 us
// (2.8 TB/s), two axis passes 90.  A derivative alone on a small grid with
// two-step kernels on both axes is left to them (30 x 30: 6.3 against 7.5 us for
// both axes but 5.1 against 3.5 for one; 60 x 60, 64 planes: 11.2 against 9.7).
#include <algorithm>
#include <mutex>

#include "common.hpp"
#include "fft_reg.hpp"
#include "kernels.hpp"

namespace edus {

namespace {

using reg::sfor;

constexpr size_t kPlaneLds = 160 * 1024;
constexpr int kAxesMaxThreads = 256;

// q = t / d for 0 <= t < 2^20 and 0 < d < 2^12, inv = 1 / d in FP32: t + 1/2
// is at least 1/2 away from any multiple of d, far above the rounding
__device__ inline int fast_div(int t, float inv) { return int((float(t) + 0.5f) * inv); }

// f(std::integral_constant<int, R>) for a radix 2 <= r <= MAXR (MAXR 12: without
// 11, whose registers would spill under that kernel's limit of 128)
template <int MAXR, class F>
__device__ __forceinline__ void with_radix(int r, F&& f)
{
    switch (r) {
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 3: f(std::integral_constant<int, 3>{}); break;
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 5: f(std::integral_constant<int, 5>{}); break;
        case 6: f(std::integral_constant<int, 6>{}); break;
        case 7: f(std::integral_constant<int, 7>{}); break;
        case 8: f(std::integral_constant<int, 8>{}); break;
        case 9: f(std::integral_constant<int, 9>{}); break;
        case 10: f(std::integral_constant<int, 10>{}); break;
        case 11: if constexpr (MAXR > 12) f(std::integral_constant<int, 11>{}); break;
        case 12: if constexpr (MAXR >= 12) f(std::integral_constant<int, 12>{}); break;
        case 13: if constexpr (MAXR >= 13) f(std::integral_constant<int, 13>{}); break;
        case 14: if constexpr (MAXR >= 14) f(std::integral_constant<int, 14>{}); break;
        case 15: if constexpr (MAXR >= 15) f(std::integral_constant<int, 15>{}); break;
        case 16: if constexpr (MAXR >= 16) f(std::integral_constant<int, 16>{}); break;
        default: break;
    }
}

// One axis of the plane in LDS: `lines` lines of n = RA * RB elements,
// `estr` apart inside a line, consecutive lines `lstr` apart.
struct PlaneAxis {
    int n, RA, RB, lines, estr, lstr;
    float inv_lines, inv_RB;
    const double2* tw;  // exp(-2 pi i j / n) in LDS
};

// Forward A step (S = -1: DFT, then the twiddle) or inverse one (S = +1: the
// conjugate twiddle, then the DFT) from src to dst, each the plane in LDS or
// in memory with its own element and line strides.  Addresses advance by
// wave-uniform strides (an index product per element would cost as much as
// the transform: 32-bit integer multiplies run at a quarter of the FP64 rate).
// ROW: neighbouring lanes run along the line (coalesced where src or dst is a
// row in memory) instead of across lines.  NT threads, or with NT = 0 as many as
// the work-group has.
template <int NT, int MAXR, int S, bool ROW = false>
__device__ __forceinline__ void step_a(const PlaneAxis& ax, int tid, const double2* src, int se, int sl, double2* dst,
                                       int de, int dl)
{
    const int nt = NT ? NT : blockDim.x;
    with_radix<MAXR>(ax.RA, [&](auto r_) {
        constexpr int R = decltype(r_)::value;
        const int RB = ax.RB, ntask = ax.lines * RB;
        for (int t = tid; t < ntask; t += nt) {
            int jb, line;
            if (ROW) {
                line = fast_div(t, ax.inv_RB);
                jb = t - line * RB;
            } else {
                jb = fast_div(t, ax.inv_lines);
                line = t - jb * ax.lines;
            }
            const double2* p = src + (line * sl + jb * se);
            double2* q = dst + (line * dl + jb * de);
            double2 v[R];
            sfor<R>([&](auto j_) {
                constexpr int j = decltype(j_)::value;
                v[j] = p[j * (RB * se)];
            });
            const double2* w = ax.tw;
            if constexpr (S > 0) {
                sfor<R - 1>([&](auto j_) {
                    constexpr int j = decltype(j_)::value + 1;
                    w += jb;
                    v[j] = cmul(v[j], cconj(*w));
                });
            }
            reg::rdft<R, S>(v);
            if constexpr (S < 0) {
                sfor<R - 1>([&](auto j_) {
                    constexpr int j = decltype(j_)::value + 1;
                    w += jb;
                    v[j] = cmul(v[j], *w);
                });
            }
            sfor<R>([&](auto j_) {
                constexpr int j = decltype(j_)::value;
                q[j * (RB * de)] = v[j];
            });
        }
    });
}

// Forward (S = -1) or inverse (S = +1) B step in place in LDS, or with S = 0
// both around mul(line, ka, kb, x), the element at frequency ka + RA kb
template <int NT, int MAXR, int S, class Mul>
__device__ __forceinline__ void step_b(const PlaneAxis& ax, int tid, double2* pl, Mul mul)
{
    const int nt = NT ? NT : blockDim.x;
    with_radix<MAXR>(ax.RB, [&](auto r_) {
        constexpr int R = decltype(r_)::value;
        const int ntask = ax.lines * ax.RA;
        for (int t = tid; t < ntask; t += nt) {
            const int ka = fast_div(t, ax.inv_lines), line = t - ka * ax.lines;
            const int es = ax.estr;
            double2* p = pl + (line * ax.lstr + ka * R * es);
            double2 u[R];
            sfor<R>([&](auto j_) {
                constexpr int j = decltype(j_)::value;
                u[j] = p[j * es];
            });
            reg::rdft<R, S == 0 ? -1 : S>(u);
            if constexpr (S == 0) {
                mul(line, ka, u);
                reg::rdft<R, 1>(u);
            }
            sfor<R>([&](auto j_) {
                constexpr int j = decltype(j_)::value;
                p[j * es] = u[j];
            });
        }
    });
}

template <int NT, int MAXR, bool PHASE>
__global__ void __launch_bounds__(NT, MAXR <= 12 ? 4 : 2) plane_kernel(PlaneArgs a)
{
    extern __shared__ double2 lds[];
    const int N0 = a.N0, N1 = a.N1, N1P = N1 | 1, Nk = N0 * N1;
    const int tid = threadIdx.x;
    double2* pl = lds;  // the plane, rows N1P apart
    double2* tw0 = pl + N0 * N1P;
    double2* tw1 = tw0 + N0;
    double2* e0 = tw1 + N1;  // phase: exp(i th R) / n per axis
    double2* e1 = e0 + N0;
    for (int i = tid; i < N0; i += NT) tw0[i] = a.tw0[i];
    for (int i = tid; i < N1; i += NT) tw1[i] = a.tw1[i];
    // work-groups [0, P) take the first result of their plane, [P, 2P) the
    // second one (exchange beside the derivative)
    const int second = blockIdx.x >= unsigned(a.P) ? 1 : 0;
    const int plane = int(blockIdx.x) - second * a.P;
    const bool conv = !PHASE && a.conv && (second || !a.out[0]);
    constexpr bool phase = PHASE;
    const double2* in = a.in + long(plane) * Nk;
    double2* out = a.out[conv ? 1 : 0] + long(plane) * Nk;
    const PlaneAxis x0{N0, a.RA0, a.RB0, N1, N1P, 1, a.inv_N1, a.inv_RB0, tw0};
    const PlaneAxis x1{N1, a.RA1, a.RB1, N0, 1, N1P, a.inv_N0, 0.f, tw1};
    // the axis whose B step applies the multiplier, the other one around it.
    // A derivative along one axis only runs that axis alone: a zero
    // coefficient adds nothing, wherever it comes from.
    PlaneAxis in_ax = x1;
    bool both = true;
    double dl = 0.0, di = 0.0;  // derivative: coefficients of the outer and the inner axis
    if (!conv && !phase) {
        double c0 = a.coef[0], c1 = a.coef[1];
        if (a.coef_tab) {
            const const_double* t = uniform_doubles(a.coef_tab + long(plane / a.ppi) * a.coef_stride);
            c0 = t[0];
            c1 = t[1];
        }
        // (the same in every lane: kept in scalar registers)
        const bool use0 = __builtin_amdgcn_readfirstlane(c0 != 0.0), use1 = __builtin_amdgcn_readfirstlane(c1 != 0.0);
        if (!use0 && !use1) {
            for (int i = tid; i < Nk; i += NT) out[i] = make_double2(0.0, 0.0);
            return;
        }
        both = use0 && use1;
        if (both) {
            dl = c0 / double(N1);
            di = c1 / double(N0);
        } else if (use1) {
            di = c1;
        } else {
            di = c0;
            in_ax = x0;
            if (in_ax.RB == 1) {  // one step: the one that multiplies
                in_ax.RB = in_ax.RA;
                in_ax.RA = 1;
            }
        }
    }
    if (phase)
        for (int i = tid; i < N0 + N1; i += NT) {
            const bool first = i < N0;
            const int j = first ? i : i - N0, n = first ? N0 : N1;
            double sn, cs;
            sincos((first ? a.coef[0] : a.coef[1]) * double(gamma_centred(j, n)), &sn, &cs);
            const double sc = 1.0 / double(n);
            (first ? e0 : e1)[j] = make_double2(sc * cs, sc * sn);
        }
    const bool copy_in = !both || phase;
    if (copy_in) {
        for (int i = tid; i < Nk; i += NT) {
            double2 v = in[i];
            if (phase)
                for (int d = 0; d < 3; ++d) {
                    if (!a.in_add[d]) continue;
                    const double2 w = a.in_add[d][long(plane) * Nk + i];
                    v.x += a.in_add_c[d] * w.x;
                    v.y += a.in_add_c[d] * w.y;
                }
            const int r = fast_div(i, a.inv_N1);
            pl[r * N1P + (i - r * N1)] = v;
        }
    }
    __syncthreads();  // the twiddles, the phases and a copied plane are in LDS
    if (both) {
        if (copy_in)
            step_a<NT, MAXR, -1>(x0, tid, pl, N1P, 1, pl, N1P, 1);
        else
            step_a<NT, MAXR, -1>(x0, tid, in, N1, 1, pl, N1P, 1);
        __syncthreads();
        if (x0.RB > 1) {
            step_b<NT, MAXR, -1>(x0, tid, pl, [](int, int, auto&) {});
            __syncthreads();
        }
    }
    if (in_ax.RA > 1) {
        step_a<NT, MAXR, -1>(in_ax, tid, pl, in_ax.estr, in_ax.lstr, pl, in_ax.estr, in_ax.lstr);
        __syncthreads();
    }
    step_b<NT, MAXR, 0>(in_ax, tid, pl, [&](int line, int ka, auto& u) {
        constexpr int R = sizeof(u) / sizeof(double2);
        // row position `line` of axis 0 holds frequency f0 after its forward steps
        const int k0 = fast_div(line, a.inv_RB0), f0 = k0 + a.RA0 * (line - k0 * a.RB0);
        if (conv) {
            // zero frequency of both axes: the plane's sum over k
            if (ka == 0 && line == 0) a.r0[plane] = u[0];
            const double* W = a.Wp + long(plane) * Nk + (ka * R) * N0 + line;
            sfor<R>([&](auto k_) {
                constexpr int k = decltype(k_)::value;
                u[k] = cscale(u[k], a.conv_scale * W[k * N0]);
            });
        } else if (phase) {
            const double2 p0 = e0[f0];
            sfor<R>([&](auto k_) {
                constexpr int k = decltype(k_)::value;
                u[k] = cmul(u[k], cmul(p0, e1[ka + x1.RA * k]));
            });
        } else {
            const double r0 = dl * double(gamma_centred(f0, N0));
            sfor<R>([&](auto k_) {
                constexpr int k = decltype(k_)::value;
                u[k] = cmul_i(u[k], r0 + di * double(gamma_centred(ka + in_ax.RA * k, in_ax.n)));
            });
        }
    });
    __syncthreads();
    if (in_ax.RA > 1) {
        step_a<NT, MAXR, 1>(in_ax, tid, pl, in_ax.estr, in_ax.lstr, pl, in_ax.estr, in_ax.lstr);
        __syncthreads();
    }
    if (both) {
        if (x0.RB > 1) {
            step_b<NT, MAXR, 1>(x0, tid, pl, [](int, int, auto&) {});
            __syncthreads();
        }
        step_a<NT, MAXR, 1>(x0, tid, pl, N1P, 1, out, N1, 1);
    } else {
        for (int i = tid; i < Nk; i += NT) {
            const int r = fast_div(i, a.inv_N1);
            out[i] = pl[r * N1P + (i - r * N1)];
        }
    }
}

// Both axes' one-dimensional derivatives, their line groups side by side in one
// launch: work-groups [0, nb0) take columns, the others rows, L lines each, and
// the two results stay apart (the commutator adds them; either may be left
// out).  On small grids, where
// a launch costs what it computes, this saves the second launch and its wait
// for the first.  Bound by latency there: three barriers and the launch.  On
// large ones by memory and the lanes at work (axes_best_shape): 120 x 120, 196
// planes 31.8 us by itself and 36.3 in the step, 5.7 and 5.0 TB/s of its two
// reads and two writes, both reads of the planes from memory.
template <int MAXR>
__global__ void __launch_bounds__(kAxesMaxThreads, MAXR <= 12 ? 4 : 3) axes_kernel(PlaneArgs a, int nb0, int L0, int L1)
{
    extern __shared__ double2 lds[];
    const int N0 = a.N0, N1 = a.N1, Nk = N0 * N1, tid = threadIdx.x;
    const bool col = int(blockIdx.x) < nb0;
    const int n = col ? N0 : N1, RA = col ? a.RA0 : a.RA1, RB = col ? a.RB0 : a.RB1;
    const int gs = col ? N1 : 1, gl = col ? 1 : N1;  // element and line strides in memory
    long base;  // first element of the group's first line
    int lines, plane0;
    if (col) {
        const int per = (N1 + L0 - 1) / L0;
        plane0 = int(blockIdx.x) / per;
        const int c = (int(blockIdx.x) - plane0 * per) * L0;
        lines = min(L0, N1 - c);
        base = long(plane0) * Nk + c;
    } else {
        const long row = long(blockIdx.x - nb0) * L1;
        lines = int(min(long(L1), long(a.P) * N0 - row));
        plane0 = int(row / N0);
        base = row * N1;
    }
    const int row_in_plane = col ? 0 : int((base / N1) % N0);
    const double2* src = a.in + base;
    double2* dst = a.out[col ? 0 : 1] + base;
    auto coef = [&](int line) {
        if (!a.coef_tab) return col ? a.coef[0] : a.coef[1];
        const int plane = col ? plane0 : plane0 + (row_in_plane + line) / N0;
        return a.coef_tab[long(plane / a.ppi) * a.coef_stride + (col ? 0 : 1)];
    };
    if (RB == 1) {  // the whole line in one thread
        with_radix<MAXR>(RA, [&](auto r_) {
            constexpr int R = decltype(r_)::value;
            for (int line = tid; line < lines; line += blockDim.x) {
                const double2* p = src + line * gl;
                double2* q = dst + line * gl;
                const double c = coef(line);
                double2 v[R];
                sfor<R>([&](auto j_) {
                    constexpr int j = decltype(j_)::value;
                    v[j] = p[j * gs];
                });
                reg::rdft<R, -1>(v);
                sfor<R>([&](auto j_) {
                    constexpr int j = decltype(j_)::value;
                    v[j] = cmul_i(v[j], c * double(gamma_centred(j, R)));
                });
                reg::rdft<R, 1>(v);
                sfor<R>([&](auto j_) {
                    constexpr int j = decltype(j_)::value;
                    q[j * gs] = v[j];
                });
            }
        });
        return;
    }
    double2* tw = lds;
    double2* buf = lds + n;
    const double2* twg = col ? a.tw0 : a.tw1;
    for (int i = tid; i < n; i += blockDim.x) tw[i] = twg[i];
    const int es = col ? L0 : 1, ls = col ? 1 : (n | 1);  // strides in LDS
    const PlaneAxis ax{n, RA, RB, lines, es, ls, 1.0f / float(lines), 1.0f / float(RB), tw};
    __syncthreads();
    if (col)
        step_a<0, MAXR, -1>(ax, tid, src, gs, gl, buf, es, ls);
    else
        step_a<0, MAXR, -1, true>(ax, tid, src, gs, gl, buf, es, ls);
    __syncthreads();
    step_b<0, MAXR, 0>(ax, tid, buf, [&](int line, int ka, auto& u) {
        constexpr int R = sizeof(u) / sizeof(double2);
        const double c = coef(line);
        sfor<R>([&](auto k_) {
            constexpr int k = decltype(k_)::value;
            u[k] = cmul_i(u[k], c * double(gamma_centred(ka + RA * k, n)));
        });
    });
    __syncthreads();
    if (col)
        step_a<0, MAXR, 1>(ax, tid, buf, es, ls, dst, gs, gl);
    else
        step_a<0, MAXR, 1, true>(ax, tid, buf, es, ls, dst, gs, gl);
}

// W[f0 * N1 + f1] of every plane into the order the convolution reads it:
// Wp[p1 * N0 + p0], the frequencies at positions p0, p1 of the two axes
__global__ void plane_permute_kernel(const double* __restrict__ W, double* __restrict__ Wp, long total, int N0, int N1,
                                     int RA0, int RB0, int RA1, int RB1)
{
    const long i = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int Nk = N0 * N1;
    const long p = i / Nk;
    const int e = int(i - p * Nk), p1 = e / N0, p0 = e - p1 * N0;
    const int f0 = p0 / RB0 + RA0 * (p0 % RB0), f1 = p1 / RB1 + RA1 * (p1 % RB1);
    Wp[i] = W[p * Nk + long(f0) * N1 + f1];
}

// n = RA * RB with both at most 16, the larger factor as small as possible;
// lines of at most 16 are one step
bool split_line(int n, int& big, int& small)
{
    if (n < 2) return false;
    if (n <= 16) {
        big = n;
        small = 1;
        return true;
    }
    for (big = 2; big <= 16; ++big)
        if (n % big == 0 && n / big <= big) {
            small = n / big;
            return true;
        }
    return false;
}

template <int NT, int MAXR, bool PHASE>
void launch_plane_nt(const PlaneArgs& a, int blocks, size_t lds, hipStream_t s)
{
    auto kern = &plane_kernel<NT, MAXR, PHASE>;
    static std::once_flag raised;  // contexts may be created from several host threads
    std::call_once(raised, [&] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(kPlaneLds));
    });
    if (g_attributes_only) return;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(NT), lds, s, a);
}

bool wide_radix(const PlaneArgs& a)
{
    for (int r : {a.RA0, a.RB0, a.RA1, a.RB1})
        if (r > 12 || r == 11) return true;
    return false;
}

size_t plane_lds(int N0, int N1, bool phase)
{
    return size_t(N0 * (N1 | 1) + (phase ? 2 : 1) * (N0 + N1)) * sizeof(double2);
}

}  // namespace

bool plane_available(int N0, int N1)
{
    int b, c;
    return split_line(N0, b, c) && split_line(N1, b, c) && plane_lds(N0, N1, true) <= kPlaneLds;
}

PlaneArgs plane_args(int N0, int N1)
{
    PlaneArgs a{};
    a.N0 = N0;
    a.N1 = N1;
    split_line(N0, a.RA0, a.RB0);
    // the inner axis keeps the multiplier in its B step
    if (N1 <= 16) {
        a.RA1 = 1;
        a.RB1 = N1;
    } else {
        split_line(N1, a.RA1, a.RB1);
    }
    a.inv_N0 = 1.0f / float(N0);
    a.inv_N1 = 1.0f / float(N1);
    a.inv_RB0 = 1.0f / float(a.RB0);
    return a;
}

template <bool PHASE>
void launch_plane_shape(const PlaneArgs& a, hipStream_t s)
{
    const int blocks = a.P * (PHASE ? 1 : (a.out[0] ? 1 : 0) + (a.conv ? 1 : 0));
    const size_t lds = plane_lds(a.N0, a.N1, PHASE);
    // 11 and radices above 12 need more than 128 registers.  The others run with
    // as many threads as give a step about one round of tasks (us for 256, 512,
    // 1024 threads: 30 x 30, 4 planes 6.2, 6.2, 6.5; 60 x 66, 25 planes 13.7,
    // 11.9, 12.2; 90 x 90 with exchange, 64 planes 25.0, 22.1, 18.9)
    const bool wide = wide_radix(a);
    const int Nk = a.N0 * a.N1;
    if (wide)
        launch_plane_nt<512, 16, PHASE>(a, blocks, lds, s);
    else if (Nk <= 1024)
        launch_plane_nt<256, 12, PHASE>(a, blocks, lds, s);
    else if (Nk <= 6000)
        launch_plane_nt<512, 12, PHASE>(a, blocks, lds, s);
    else
        launch_plane_nt<1024, 12, PHASE>(a, blocks, lds, s);
}

void launch_plane(const PlaneArgs& a, hipStream_t s)
{
    if (a.phase)
        launch_plane_shape<true>(a, s);
    else
        launch_plane_shape<false>(a, s);
}

bool axes_available(int N0, int N1)
{
    int b, c;
    return split_line(N0, b, c) && split_line(N1, b, c);
}

bool axes_wide(int N0, int N1) { return wide_radix(axes_args(N0, N1)); }

PlaneArgs axes_args(int N0, int N1)
{
    PlaneArgs a{};
    a.N0 = N0;
    a.N1 = N1;
    split_line(N0, a.RA0, a.RB0);
    split_line(N1, a.RA1, a.RB1);
    return a;
}

namespace {

// Threads and lines of an axes_kernel launch
struct AxesShape {
    int nt, L0, L1;
    size_t lds;
};

AxesShape axes_shape(const PlaneArgs& a, int nt)
{
    // about one task per thread and step, columns in whole 128-byte runs, within
    // the 64 KB of LDS that need no raised limit
    auto lines = [&](int n, int RA, int RB) {
        if (RB == 1) return nt;
        const int most = (64 * 1024 / int(sizeof(double2)) - n) / (n | 1);
        return std::max(1, std::min(nt / std::max(RA, RB), most));
    };
    AxesShape s{nt, std::min(lines(a.N0, a.RA0, a.RB0), a.N1), lines(a.N1, a.RA1, a.RB1), 0};
    if (s.L0 > 8 && s.L0 < a.N1) s.L0 = s.L0 / 8 * 8;
    s.lds = sizeof(double2) * std::max(a.RB0 > 1 ? a.N0 + a.N0 * s.L0 : 0, a.RB1 > 1 ? a.N1 + (a.N1 | 1) * s.L1 : 0);
    return s;
}

// Work-group size.  With at most kAxesFewGroups work-groups of one wave the
// launch is latency and they are spread widest (us for 64, 128, 192, 256 threads:
// 30 x 30, 4 planes 3.8, 4.1, 4.2, 4.3; 45 x 63, 21 planes 4.8, 5.0, 5.3, 5.6).
// Otherwise the size that keeps most threads of a CU at work, given the waves its
// registers allow, the LDS of the lines and the tasks these make, ties to the
// smaller (120 x 120, 196 planes -, 30.6, 31.8, 33.5; 90 x 90, 64 planes -, 10.6,
// 10.2, 9.4; 48 x 48, 2352 planes 44.5, 45.6, 47.1, 49.3), of those whose columns
// fill 128-byte runs (one wave at 120 x 120: 5 columns, 44.9).
constexpr long kAxesFewGroups = 1024;

AxesShape axes_best_shape(const PlaneArgs& a)
{
    const AxesShape s1 = axes_shape(a, 64);
    const long groups = long(a.P) * ((a.N1 + s1.L0 - 1) / s1.L0) + (long(a.P) * a.N0 + s1.L1 - 1) / s1.L1;
    if (groups <= kAxesFewGroups) return s1;
    const int waves = wide_radix(a) ? 12 : 16;  // of a CU
    AxesShape best{};
    long most = -1;
    for (int nt = 64; nt <= kAxesMaxThreads; nt += 64) {
        const AxesShape s = axes_shape(a, nt);
        if (s.L0 < std::min(8, a.N1) && nt < kAxesMaxThreads) continue;
        const long per_cu = std::min(waves * 64 / nt, s.lds ? int(kPlaneLds / s.lds) : 16);
        const long busy = per_cu * (s.L0 * (a.RA0 + a.RB0) + s.L1 * (a.RA1 + a.RB1));
        if (busy > most) {
            most = busy;
            best = s;
        }
    }
    return best;
}

}  // namespace

void launch_axes(const PlaneArgs& a, hipStream_t s)
{
    const AxesShape q = axes_best_shape(a);
    const int nb0 = a.out[0] ? a.P * ((a.N1 + q.L0 - 1) / q.L0) : 0;
    const int nb1 = a.out[1] ? int((long(a.P) * a.N0 + q.L1 - 1) / q.L1) : 0;
    if (wide_radix(a))
        hipLaunchKernelGGL(axes_kernel<16>, dim3(nb0 + nb1), dim3(q.nt), q.lds, s, a, nb0, q.L0, q.L1);
    else
        hipLaunchKernelGGL(axes_kernel<12>, dim3(nb0 + nb1), dim3(q.nt), q.lds, s, a, nb0, q.L0, q.L1);
}

void launch_plane_permute(const double* W, double* Wp, int P, int N0, int N1, hipStream_t s)
{
    const PlaneArgs a = plane_args(N0, N1);
    const long n = long(P) * N0 * N1;
    hipLaunchKernelGGL(plane_permute_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, W, Wp, n, N0, N1, a.RA0,
                       a.RB0, a.RA1, a.RB1);
}

}  // namespace edus
