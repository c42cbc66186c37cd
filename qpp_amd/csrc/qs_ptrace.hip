// qs_ptrace.hip -- partial trace of kets and density matrices.
//
//   k_gram, k_gram_pair   kets: tr_B |psi><psi| = M M^dagger with M(i, t) =
//                 psi(i, t), i the kept digits and t the traced ones, as FP64
//                 matrix products on tiles of M read straight from the state.
//   k_gram_out    sums their partial tiles into the output matrix.
//   k_ptrace      direct sums, one output entry by a few threads: density
//                 matrices, and kets too small for the matrix products to pay.
//
// All sums run in FP64, for complex64 states too.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "qs_digits.hpp"
#include "qs_internal.hpp"

namespace {

using namespace qs_digits;

typedef double doublex4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// kets: M M^dagger on the FP64 matrix cores
// ---------------------------------------------------------------------------
// A "row" is a kept index together with, where the kept space has fewer than
// 16 states, as many of the fastest traced digits as fill 16 rows (`grp` of
// them per kept index): the product of two rows counts only where their
// traced digits agree, and k_gram_out picks those.  So M has R = Dbar * grp
// rows, and a wave step multiplies 16 x 4 pieces of it with
// v_mfma_f64_16x16x4f64 (D[16x16] += A[16x4] B[4x16]; lane l holds
// A[l%16][l/16], B[l/16][l%16] and D[4v + l/16][l%16], v = 0..3): a lane's
// amplitude M(16 b + l%16, t + l/16) is the A operand of row block b and the
// B operand of column block b at once.  Re(M M^d) = Mr Mr^T + Mi Mi^T and
// Im = Mi Mr^T - Mr Mi^T take four of them per 16 x 16 tile.
//
// The traced index is (th, tl): tl runs over the fastest digits, whose
// offsets sit in LDS, th over the others; a workgroup takes a slice of th.
//
// Measured against one wave per entry with its offsets by 64-bit division
// (k_ptrace as it was), complex128: 24 qubits with 8 kept 54.6 -> 0.42 ms (46
// TFLOP/s; 12 kept 58 TFLOP/s), with 4 kept 62 -> 0.084 ms, 26 qubits with 1
// kept 2600 -> 0.34 ms (3.2 TB/s), 14 qutrits with 4 kept 4.4 -> 0.15 ms.
template <int TB>
struct Acc {
    doublex4 re[TB][TB], im[TB][TB];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int x = 0; x < TB; ++x)
#pragma unroll
            for (int y = 0; y < TB; ++y) {
                re[x][y] = doublex4{0, 0, 0, 0};
                im[x][y] = doublex4{0, 0, 0, 0};
            }
    }
    template <typename T>
    __device__ __forceinline__ void add(const T (&a)[TB], const T (&b)[TB]) {
#pragma unroll
        for (int x = 0; x < TB; ++x) {
            const double ar = a[x].x, ai = a[x].y;
#pragma unroll
            for (int y = 0; y < TB; ++y) {
                const double br = b[y].x, bi = b[y].y;
                re[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, re[x][y], 0, 0, 0);
                im[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, br, im[x][y], 0, 0, 0);
                re[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, bi, re[x][y], 0, 0, 0);
                im[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ar, bi, im[x][y], 0, 0, 0);
            }
        }
    }
};

// R <= 16 TB rows: all of them in one wave's tile, the loads straight from
// the state (each amplitude once), so HBM bounds it.  The four waves take
// every fourth step of the slice and add their tiles up in LDS.
template <typename T, int TB>
__global__ __launch_bounds__(256) void k_gram(const T* __restrict__ a, Digits rows, Digits lo,
                                              Digits hi, uint32_t R, uint32_t TL, uint32_t nth,
                                              uint32_t per, double2* __restrict__ part) {
    constexpr int W = 16 * TB;
    extern __shared__ unsigned char smem_raw[];
    double2* tile = reinterpret_cast<double2*>(smem_raw);                // W x W, column-major
    uint64_t* lo_off = reinterpret_cast<uint64_t*>(smem_raw + sizeof(double2) * W * W);  // TL
    for (uint32_t i = threadIdx.x; i < TL; i += 256) lo_off[i] = offset_of(lo, i);
    const uint32_t lane = threadIdx.x & 63, lr = lane & 15, lt = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const T* row[TB];
    // rows past the last one repeat it; their products are never read
#pragma unroll
    for (int b = 0; b < TB; ++b) row[b] = a + offset_of(rows, min(16 * b + lr, R - 1));
    __syncthreads();
    Acc<TB> acc;
    acc.clear();
    constexpr int U = 4 / TB;  // steps loaded together: 64 U contiguous traced bytes a row
    const uint32_t th1 = min((blockIdx.x + 1) * per, nth), nsteps = (TL + 4 * U - 1) / (4 * U);
    // the wave's steps (th, s): s = wave, wave + 4, ... of every th
    uint32_t th = blockIdx.x * per, s = wave;
    if (s >= nsteps) th = th1;
    uint64_t base = offset_of(hi, th);
    T cur[U][TB], next[U][TB];
    auto fetch = [&](uint32_t step, T (&x)[U][TB]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t t = (step * U + u) * 4 + lt;
            const bool ok = t < TL;
            const uint64_t off = base + lo_off[ok ? t : 0];
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                x[u][b] = row[b][off];
                if (!ok) x[u][b].x = 0, x[u][b].y = 0;
            }
        }
    };
    if (th < th1) fetch(s, cur);
    while (th < th1) {
        s += 4;
        if (s >= nsteps) {
            s = wave;
            base = offset_of(hi, ++th);
        }
        if (th < th1) fetch(s, next);
#pragma unroll
        for (int u = 0; u < U; ++u) acc.add(cur[u], cur[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int b = 0; b < TB; ++b) cur[u][b] = next[u][b];
    }
    for (uint32_t w = 0; w < 4; ++w) {
        if (wave == w) {
#pragma unroll
            for (int x = 0; x < TB; ++x)
#pragma unroll
                for (int y = 0; y < TB; ++y)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        double2& d = tile[(16 * y + lr) * W + 16 * x + 4 * v + lt];
                        double2 z = make_double2(acc.re[x][y][v], acc.im[x][y][v]);
                        if (w) z.x += d.x, z.y += d.y;
                        d = z;
                    }
        }
        __syncthreads();
    }
    double2* o = part + uint64_t(blockIdx.x) * (W * W);
    for (uint32_t e = threadIdx.x; e < W * W; e += 256) o[e] = tile[e];
}

// More rows: a workgroup takes one pair of 64-row blocks I <= J (the rest
// follows from hermiticity), each wave one 32 x 32 quarter of it, and stages
// 8 traced values of both blocks at a time in LDS while the next ones are on
// their way to registers.  The matrix rate bounds it: 32 matrix instructions
// (2048 cycles) per wave and 16 KiB staged.  Loads run along
// the rows (ROWFAST) or along the traced index, whichever has the smaller
// stride.  Eight slices or more go round the 8 XCDs by workgroup number, all
// pairs of a slice on the same one, so that a slice comes from HBM into one
// L2; fewer would leave XCDs idle, and all pairs go round them.
constexpr int kGramW = 64, kGramK = 8;

template <typename T, bool ROWFAST>
__global__ __launch_bounds__(256) void k_gram_pair(const T* __restrict__ a, Digits rows, Digits lo,
                                                   Digits hi, uint32_t R, uint32_t TL, uint32_t nth,
                                                   uint32_t npairs, uint32_t nslices, uint32_t per,
                                                   double2* __restrict__ part, T* __restrict__ out) {
    constexpr int W = kGramW, K = kGramK, LD = W + 1;  // LD: spreads a row's values over the banks
    extern __shared__ unsigned char smem_raw[];
    T* lds = reinterpret_cast<T*>(smem_raw);  // [buffer][side][t][row]
    uint64_t* lo_off = reinterpret_cast<uint64_t*>(smem_raw + sizeof(T) * 4 * K * LD);  // TL
    for (uint32_t i = threadIdx.x; i < TL; i += 256) lo_off[i] = offset_of(lo, i);
    uint32_t pair = blockIdx.x % npairs, slice = blockIdx.x / npairs;
    if (nslices >= 8) {
        const uint32_t xcd = blockIdx.x & 7, r8 = blockIdx.x >> 3;
        pair = r8 % npairs;
        slice = (r8 / npairs) * 8 + xcd;
    }
    if (slice >= nslices) return;  // the whole workgroup
    uint32_t J = uint32_t((sqrt(8.0 * pair + 1.0) - 1.0) * 0.5);
    while ((J + 1) * (J + 2) / 2 <= pair) ++J;
    while (J * (J + 1) / 2 > pair) --J;
    const uint32_t I = pair - J * (J + 1) / 2;
    const bool diag = I == J;
    const uint32_t lane = threadIdx.x & 63, lr = lane & 15, lt = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wi = wave & 1, wj = wave >> 1;  // the wave's quarter
    // the elements a thread stages per side: rows and traced values
    constexpr int E = W * K / 256, NR = ROWFAST ? 1 : E;
    const uint32_t er = ROWFAST ? threadIdx.x % W : threadIdx.x / K;
    const uint32_t et = ROWFAST ? threadIdx.x / W : threadIdx.x % K;
    auto row_of = [&](int e) { return ROWFAST ? er : er + (256u / K) * e; };
    auto t_of = [&](int e) { return ROWFAST ? et + (256u / W) * e : et; };
    const T* src[2][NR];
#pragma unroll
    for (int e = 0; e < NR; ++e) {
        // rows past the last one repeat it; their products are never read
        src[0][e] = a + offset_of(rows, min(I * W + row_of(e), R - 1));
        src[1][e] = a + offset_of(rows, min(J * W + row_of(e), R - 1));
    }
    __syncthreads();
    T st[2][E];
    uint64_t base = 0;
    auto fetch = [&](uint32_t c) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const uint32_t t = c * K + t_of(e);
            const bool ok = t < TL;
            const uint64_t off = base + lo_off[ok ? t : 0];
            st[0][e] = src[0][ROWFAST ? 0 : e][off];
            if (!diag) st[1][e] = src[1][ROWFAST ? 0 : e][off];
            if (!ok) st[0][e].x = 0, st[0][e].y = 0, st[1][e].x = 0, st[1][e].y = 0;
        }
    };
    auto stage = [&](uint32_t buf) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            lds[((buf * 2) * K + t_of(e)) * LD + row_of(e)] = st[0][e];
            if (!diag) lds[((buf * 2 + 1) * K + t_of(e)) * LD + row_of(e)] = st[1][e];
        }
    };
    Acc<2> acc;
    acc.clear();
    const uint32_t th1 = min((slice + 1) * per, nth), nchunks = (TL + K - 1) / K;
    // every pair starts elsewhere in the slice: rows are often a power of two
    // apart, and pairs in step would all read the same few memory channels
    const uint32_t th0 = slice * per;
    uint32_t th = th0 + pair % (th1 - th0), left = th1 - th0, c = 0, buf = 0;
    base = offset_of(hi, th);
    fetch(0);
    stage(0);
    __syncthreads();
    while (left) {
        if (++c == nchunks) {
            c = 0;
            --left;
            if (++th == th1) th = th0;
            base = offset_of(hi, th);
        }
        if (left) fetch(c);
        if (!diag || wi <= wj) {  // the quarter below the diagonal is not read
            const T* A = lds + (buf * 2) * K * LD + 32 * wi + lr;
            const T* B = lds + (buf * 2 + (diag ? 0 : 1)) * K * LD + 32 * wj + lr;
#pragma unroll
            for (int s = 0; s < K / 4; ++s) {
                T x[2], y[2];
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    x[b] = A[(4 * s + lt) * LD + 16 * b];
                    y[b] = B[(4 * s + lt) * LD + 16 * b];
                }
                acc.add(x, y);
            }
        }
        buf ^= 1;
        if (left) stage(buf);
        __syncthreads();
    }
    if (diag && wi > wj) return;
    if (out) {  // the only slice: the result itself
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const uint32_t i = I * W + 32 * wi + 16 * x + 4 * v + lt;
                    const uint32_t j = J * W + 32 * wj + 16 * y + lr;
                    if (i >= R || j >= R || i > j) continue;
                    T z;
                    z.x = acc.re[x][y][v];
                    z.y = i == j ? acc.im[x][y][v] * 0 : acc.im[x][y][v];  // (NaN stays NaN)
                    out[uint64_t(j) * R + i] = z;
                    z.y = -z.y;
                    if (i != j) out[uint64_t(i) * R + j] = z;
                }
        return;
    }
    double2* o = part + (uint64_t(pair) * nslices + slice) * (W * W);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                o[(32 * wj + 16 * y + lr) * W + 32 * wi + 16 * x + 4 * v + lt] =
                    make_double2(acc.re[x][y][v], acc.im[x][y][v]);
}

// out(i, j) = sum over slices (and over the `grp` traced values shared by a
// row pair) of the tiles of W x W; entries below the diagonal are the conjugates
// of those above, the diagonal is real.  A workgroup makes 256 / sl entries,
// sl threads each.
template <typename T, uint32_t W>
__global__ __launch_bounds__(256) void k_gram_out(const double2* __restrict__ part, uint32_t Dbar,
                                                  uint32_t grp, uint32_t nslices, uint32_t sl,
                                                  T* __restrict__ out) {
    __shared__ double2 red[256];
    const uint32_t E = 256 / sl, e = threadIdx.x % E, l = threadIdx.x / E;
    const uint64_t o = uint64_t(blockIdx.x) * E + e;
    const uint32_t i = uint32_t(o % Dbar), j = uint32_t(o / Dbar);
    double2 v = make_double2(0, 0);
    if (j < Dbar) {
        const uint32_t p = min(i, j) * grp, q = max(i, j) * grp;  // first rows of the two
        const uint32_t I = p / W, J = q / W;
        const double2* t = part + (uint64_t(J) * (J + 1) / 2 + I) * nslices * (W * W);
        const uint32_t at = (q % W) * W + p % W;
        for (uint32_t s = l; s < nslices; s += sl)
            for (uint32_t g = 0; g < grp; ++g) {
                const double2 x = t[uint64_t(s) * (W * W) + at + g * (W + 1)];
                v.x += x.x;
                v.y += x.y;
            }
    }
    red[threadIdx.x] = v;
    __syncthreads();
    if (l == 0 && j < Dbar) {
        for (uint32_t k = 1; k < sl; ++k) {
            v.x += red[k * E + e].x;
            v.y += red[k * E + e].y;
        }
        T r;
        r.x = v.x;
        r.y = i < j ? v.y : i > j ? -v.y : v.y * 0;  // (NaN and infinity stay NaN)
        out[o] = r;
    }
}

// ---------------------------------------------------------------------------
// direct sums
// ---------------------------------------------------------------------------
// A workgroup makes E = 256 / sl consecutive rows i of one output column j,
// sl threads each over the traced index; consecutive threads take
// consecutive rows (kept digits), which are consecutive in memory where the
// lowest subsystem is kept.
template <typename T, typename DG>
__global__ __launch_bounds__(256) void k_ptrace(const T* __restrict__ a, T* __restrict__ out,
                                                DG keep, DG tr, uint64_t Dbar, uint64_t Dsub,
                                                uint64_t D, uint32_t sl, int rho) {
    __shared__ double2 red[256];
    const uint32_t E = 256 / sl, e = threadIdx.x % E, l = threadIdx.x / E;
    using Ix = typename DG::Index;
    const uint64_t i = uint64_t(blockIdx.x) * E + e;
    const uint64_t rb = offset_of(keep, Ix(min(i, Dbar - 1)));
    for (uint64_t j = blockIdx.y; j < Dbar; j += gridDim.y) {
        const uint64_t cb = offset_of(keep, Ix(j));
        // a ket's entry below the diagonal is the conjugate of the one above
        const bool above = i <= j;
        const uint64_t pb = above ? rb : cb, qb = above ? cb : rb;
        double sr = 0, si = 0;
        for (uint64_t t = l; t < Dsub; t += sl) {
            const uint64_t off = offset_of(tr, Ix(t));
            if (rho) {
                const T v = a[(rb + off) + (cb + off) * D];
                sr += v.x;
                si += v.y;
            } else {
                const T x = a[pb + off], y = a[qb + off];
                // x * conj(y)
                const double xr = x.x, xi = x.y, yr = y.x, yi = y.y;
                sr += xr * yr + xi * yi;
                si += xi * yr - xr * yi;
            }
        }
        if (sl > 1) {
            red[threadIdx.x] = make_double2(sr, si);
            __syncthreads();
            if (l == 0)
                for (uint32_t k = 1; k < sl; ++k) {
                    sr += red[k * E + e].x;
                    si += red[k * E + e].y;
                }
            __syncthreads();
        }
        if (l == 0 && i < Dbar) {
            T v;
            v.x = sr;
            v.y = rho ? si : i == j ? si * 0 : above ? si : -si;  // (NaN and infinity stay NaN)
            out[i + j * Dbar] = v;
        }
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
uint64_t count_of(const DigitList& list) {
    uint64_t c = 1;
    for (const auto& d : list) c *= d.first;
    return c;
}

// How the matrix products of W-row tiles are cut: slices of `per` values of
// the outer traced index, and an estimate of the time.
struct GramPlan {
    uint32_t npairs, nslices, per;
    bool whole;  // one slice of k_gram_pair writes the result itself
    double us;
};

GramPlan gram_plan(uint32_t W, uint32_t R, uint32_t TL, uint32_t nth) {
    const uint32_t nb = (R + W - 1) / W;
    GramPlan g{};
    g.npairs = nb * (nb + 1) / 2;
    // One round of resident workgroups: k_gram_pair's three per CU are 96 on
    // each XCD, which takes whole slices (one workgroup too many on an XCD is
    // a second round: 24 qubits with 8 kept, 10 pairs, take 465 us with 94
    // slices, 524 with 74, 420 with 69).  Each has at least 64 traced values
    // (below that writing the tiles shows).
    uint32_t want = (W == 16 ? 2048 : 1024) / std::min<uint32_t>(g.npairs, 1024);
    if (W == kGramW && g.npairs <= 96) want = 8 * (96 / g.npairs);
    const uint32_t most = std::max<uint32_t>(1, static_cast<uint32_t>(uint64_t(TL) * nth / 64));
    g.nslices = std::min({want, most, std::max<uint32_t>(nth, 1)});
    g.per = (nth + g.nslices - 1) / g.nslices;
    g.nslices = (nth + g.per - 1) / g.per;
    g.whole = W == kGramW && g.nslices == 1;
    // a slice is serial: 0.14 us a traced value (k_gram 0.04), 81 rows of
    // 1000 values of one digit 165 us, 30 of 3000 142
    const double rounds = std::max(1.0, double(g.npairs) * g.nslices / 768);
    g.us = (g.whole ? 17 : 28) + rounds * g.per * TL * (W == kGramW ? 0.14 : 0.04);
    return g;
}

// Threads per entry of k_ptrace: as many as leave each a few terms, and more
// where there are few entries.
uint32_t direct_threads(uint64_t Dbar, uint64_t Dsub) {
    uint32_t sl = 1;
    while (sl < 256 && sl * 8 <= Dsub && Dbar * Dbar * sl < (uint64_t{1} << 18)) sl *= 2;
    while (sl < 256 && sl < Dsub && Dbar * Dbar * sl < (uint64_t{1} << 14)) sl *= 2;
    return sl;
}

// An estimate of k_ptrace's time on a ket.  Calls of one MI355X, either dtype
// (matrix products / direct sums): kept 2 of 13, 14, 16 qubits 26/25, 28/42,
// 28/158 us; 16 of 12, 16, 18 qubits 26/21, 28/26, 28/82; 64 of 12, 16, 18
// 19/21, 29/26, 30/92; 512 of 14, 16 18/31, 35/123; 9 qutrits with 4 kept
// 34/20, 11 with 5 40/114; one digit of 1000 kept and one traced 169/4000.
double direct_us(uint64_t Dbar, uint64_t Dsub) {
    const double terms = std::ceil(double(Dsub) / direct_threads(Dbar, Dsub));
    return 19 + std::max(1.1 * (terms - 12), 2.2e-6 * double(Dbar) * double(Dbar) * double(Dsub));
}

// launch_gram: no memory for the partial tiles
constexpr int kNoRoom = -1;

template <typename T, uint32_t W>
int launch_gram(const qs_state* in, qs_state* out, const Digits& rows, const Digits& lo,
                const Digits& hi, uint32_t Dbar, uint32_t grp, uint32_t TL, uint32_t nth,
                bool rowfast) {
    constexpr const char* where = "qpp::ptrace()";
    const uint32_t R = Dbar * grp;
    const GramPlan plan = gram_plan(W, R, TL, nth);
    const uint32_t npairs = plan.npairs, nslices = plan.nslices, per = plan.per;
    const bool direct = plan.whole;
    double2* part = nullptr;  // at most 2048 tiles
    if (!direct) {
        const hipError_t e = hipMallocAsync(reinterpret_cast<void**>(&part),
                                            sizeof(double2) * W * W * uint64_t(npairs) * nslices, in->stream);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();  // handled: not the next call's
            return kNoRoom;
        }
        if (e != hipSuccess) return qs::fail_hip(e, where);
    }
    const T* src = static_cast<const T*>(in->d);
    T* dst = static_cast<T*>(out->d);
    if constexpr (W == kGramW) {
        const dim3 g(npairs * (nslices < 8 ? nslices : (nslices + 7) / 8 * 8));
        const size_t shmem = sizeof(T) * 4 * kGramK * (W + 1) + sizeof(uint64_t) * TL;
        T* whole = direct ? dst : nullptr;
        if (rowfast)
            hipLaunchKernelGGL((k_gram_pair<T, true>), g, dim3(256), shmem, in->stream, src, rows, lo,
                               hi, R, TL, nth, npairs, nslices, per, part, whole);
        else
            hipLaunchKernelGGL((k_gram_pair<T, false>), g, dim3(256), shmem, in->stream, src, rows, lo,
                               hi, R, TL, nth, npairs, nslices, per, part, whole);
    } else {
        const size_t shmem = sizeof(double2) * W * W + sizeof(uint64_t) * TL;
        hipLaunchKernelGGL((k_gram<T, W / 16>), dim3(nslices), dim3(256), shmem, in->stream, src, rows,
                           lo, hi, R, TL, nth, per, part);
    }
    if (!direct) {
        uint32_t sl = 1;  // threads per output entry
        while (sl < 64 && sl * 4 <= nslices) sl *= 2;
        const uint64_t no = uint64_t(Dbar) * Dbar, E = 256 / sl;
        hipLaunchKernelGGL((k_gram_out<T, W>), dim3(static_cast<uint32_t>((no + E - 1) / E)), dim3(256),
                           0, in->stream, part, Dbar, grp, nslices, sl, dst);
    }
    const hipError_t e = hipGetLastError();
    if (part) (void)hipFreeAsync(part, in->stream);
    if (e != hipSuccess) return qs::fail_hip(e, where);
    return QS_OK;
}

template <typename T>
int ptrace_impl(const qs_state* in, qs_state* out, const DigitList& keep, const DigitList& tr) {
    constexpr const char* W = "qpp::ptrace()";
    const bool rho = in->kind == QS_RHO;
    const uint64_t Dbar = count_of(keep), Dsub = count_of(tr);
    // the smallest stride last, so that consecutive traced values are near
    DigitList ts = tr;
    std::stable_sort(ts.begin(), ts.end(), [](auto& x, auto& y) { return x.second > y.second; });
    if (!rho && Dbar * Dbar * Dsub >= (uint64_t{1} << 16) && Dsub >= 16 && Dbar <= (uint64_t{1} << 18)) {
        DigitList rows = keep;
        uint64_t grp = 1, TL = 1;
        while (!ts.empty() && Dbar * grp * ts.back().first <= 16) {
            grp *= ts.back().first;
            rows.push_back(ts.back());  // a row's traced digits: its fastest ones
            ts.pop_back();
        }
        // rows lists the traced digits fastest first: put the fastest last
        std::reverse(rows.begin() + static_cast<std::ptrdiff_t>(keep.size()), rows.end());
        DigitList lo;
        const uint64_t cap = Dbar > 32 || Dsub < (uint64_t{1} << 17) ? 64 : 256;
        while (!ts.empty() && (TL * ts.back().first <= cap || (lo.empty() && ts.back().first <= 4096))) {
            TL *= ts.back().first;
            lo.push_back(ts.back());
            ts.pop_back();
        }
        std::reverse(lo.begin(), lo.end());
        const uint64_t nth = count_of(ts);
        Digits drows, dlo, dhi;
        if (digits_fit(rows, &drows) && digits_fit(lo, &dlo) && digits_fit(ts, &dhi) &&
            (!lo.empty() || ts.empty())) {
            const auto D32 = static_cast<uint32_t>(Dbar), G32 = static_cast<uint32_t>(grp);
            const auto T32 = static_cast<uint32_t>(TL), H32 = static_cast<uint32_t>(nth);
            // along the rows where the fastest kept digit is below the traced ones
            const bool rowfast = dlo.n == 0 || (drows.n && drows.str[drows.n - 1] < dlo.str[dlo.n - 1]);
            // the matrix products where they are expected to take less time
            // than the direct sums (their slices cut whole digits, so one
            // large traced digit leaves most of the chip idle)
            const uint32_t w = Dbar * grp <= 16 ? 16 : Dbar <= 32 ? 32 : kGramW;
            int rc = kNoRoom;
            if (gram_plan(w, D32 * G32, T32, H32).us < direct_us(Dbar, Dsub))
                rc = w == 16   ? launch_gram<T, 16>(in, out, drows, dlo, dhi, D32, G32, T32, H32, rowfast)
                     : w == 32 ? launch_gram<T, 32>(in, out, drows, dlo, dhi, D32, G32, T32, H32, rowfast)
                               : launch_gram<T, kGramW>(in, out, drows, dlo, dhi, D32, G32, T32, H32, rowfast);
            if (rc != kNoRoom) return rc;
        }
        ts = tr;
    }
    const uint32_t sl = direct_threads(Dbar, Dsub);
    const uint64_t gx = (Dbar + 256 / sl - 1) / (256 / sl);
    const uint64_t gy = std::min<uint64_t>(Dbar, std::max<uint64_t>(1, 16384 / gx));
    const dim3 g(static_cast<uint32_t>(gx), static_cast<uint32_t>(gy));
    const T* src = static_cast<const T*>(in->d);
    T* dst = static_cast<T*>(out->d);
    Digits dk, dt;
    if (digits_fit(keep, &dk) && digits_fit(ts, &dt)) {
        hipLaunchKernelGGL((k_ptrace<T, Digits>), g, dim3(256), 0, in->stream, src, dst, dk, dt, Dbar,
                           Dsub, in->D, sl, int(rho));
    } else {
        hipLaunchKernelGGL((k_ptrace<T, WideDigits>), g, dim3(256), 0, in->stream, src, dst,
                           wide_digits(keep), wide_digits(ts), Dbar, Dsub, in->D, sl, int(rho));
    }
    QS_HIP(hipGetLastError(), W);
    return QS_OK;
}

}  // namespace

namespace qs {

int launch_ptrace(const qs_state* in, qs_state* out, const std::vector<std::pair<uint64_t, uint64_t>>& keep,
                  const std::vector<std::pair<uint64_t, uint64_t>>& traced) {
    return in->dtype == QS_C128 ? ptrace_impl<double2>(in, out, keep, traced)
                                : ptrace_impl<float2>(in, out, keep, traced);
}

}  // namespace qs
