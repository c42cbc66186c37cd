// qs_gates.hip -- gate-application kernels for gfx950 (CDNA4, wave64).
//
// Kernels operate on a bit-addressed array of complex elements (see
// qs_internal.hpp): kets, and density matrices as vec(rho) over 2n bits.
//
//   k_gate1_hi  1-bit gate, target bit >= 6: each work item is one amplitude
//               pair (i0, i0 | 2^bit); control bits and the target bit are
//               squeezed out of the work index, so only pairs whose controls
//               are met are read or written (2*s*2^(nb-c) bytes) and lanes of
//               a wave touch consecutive addresses in both halves.
//   k_gate1_lo  1-bit gate, target bit < 6: the partner of an element lies in
//               the same 64-element aligned chunk, i.e. in another lane of
//               the same wave; lanes load consecutive elements (fully
//               coalesced) and exchange partners with a lane shuffle.
//   k_gate_reg  2- to 4-bit dense gates (complex64: 2 and 3 bits), and 1- and
//               2-qubit gates on both sides of a density matrix in one pass:
//               a thread's group of amplitudes in registers.
//   k_gatek     wider dense gates (k <= 10) through LDS: a workgroup stages a
//               batch of amplitude groups, each thread then forms outputs
//               from the staged group and the gate matrix.
//   k_gatek_mfma  5-bit dense gates on complex64 states with FP32 MFMA: Y = U X over the state's amplitude groups as a real
//               GEMM (2^(k+1) x 2^(k+1) times 16 groups per wave step).
//   k_qudit     mixed-radix gate for qudit states (multi-index strides).
//
// Arithmetic: complex128 in double, complex64 in float; gate matrices are
// converted to the state's precision on the host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "qs_digits.hpp"
#include "qs_internal.hpp"

namespace {

using namespace qs_digits;

template <typename R>
struct cx;
template <>
struct cx<double> {
    using T = double2;
};
template <>
struct cx<float> {
    using T = float2;
};
template <typename R>
using cxt = typename cx<R>::T;

template <typename R>
__device__ __forceinline__ cxt<R> cmul(cxt<R> a, cxt<R> b) {
    cxt<R> r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    return r;
}

template <typename R>
__device__ __forceinline__ cxt<R> conj_c(cxt<R> a) {
    a.y = -a.y;
    return a;
}

template <typename R>
__device__ __forceinline__ cxt<R> cfma(cxt<R> a, cxt<R> b, cxt<R> c) {
    // a * b + c
    cxt<R> r;
    r.x = c.x + a.x * b.x - a.y * b.y;
    r.y = c.y + a.x * b.y + a.y * b.x;
    return r;
}

// 2x2 gate, row-major entries u00 u01 u10 u11 in the state's precision
template <typename R>
struct M2 {
    cxt<R> u00, u01, u10, u11;
};

// Insert zero bits at the sorted positions pos[0..np-1] (ascending) into x.
// The positions (bytes of a kernel argument) are read four to a 32-bit
// word: a uniform word load is a scalar load, where a byte load would be a
// vector load whose wait also waits for every other load and store the
// wave has in flight (the prefetched amplitudes among them).
__device__ __forceinline__ uint64_t insert_zeros(uint64_t x, const uint8_t* pos,
                                                 int np) {
    const uint32_t* w = reinterpret_cast<const uint32_t*>(pos);
    for (int i = 0; i < np; ++i) {
        const uint32_t p = (w[i >> 2] >> (8 * (i & 3))) & 0xFFu;
        const uint64_t lo = x & ((uint64_t{1} << p) - 1);
        x = ((x >> p) << (p + 1)) | lo;
    }
    return x;
}

struct Fixed {
    uint8_t pos[64];  // sorted ascending bit positions to squeeze out
    int np;
};

constexpr int kBlock = 256;

// ---------------------------------------------------------------------------
// 1-bit gate, target bit >= 6
// ---------------------------------------------------------------------------
template <typename R, int PPT>
__global__ __launch_bounds__(kBlock) void k_gate1_hi(cxt<R>* __restrict__ a,
                                                      uint64_t npairs,
                                                      uint64_t step, M2<R> u,
                                                      Fixed fx, uint64_t cval) {
    const uint64_t nthreads = uint64_t(gridDim.x) * kBlock;
    uint64_t p = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    // PPT independent pairs per thread, strided by the grid for coalescing
    cxt<R> x0[PPT], x1[PPT];
    uint64_t i0[PPT];
    for (; p < npairs; p += nthreads * PPT) {
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            const uint64_t q = p + j * nthreads;
            i0[j] = q < npairs ? (insert_zeros(q, fx.pos, fx.np) | cval) : 0;
            if (q < npairs) {
                x0[j] = a[i0[j]];
                x1[j] = a[i0[j] + step];
            }
        }
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            const uint64_t q = p + j * nthreads;
            if (q < npairs) {
                const cxt<R> y0 = cfma<R>(u.u00, x0[j], cmul<R>(u.u01, x1[j]));
                const cxt<R> y1 = cfma<R>(u.u10, x0[j], cmul<R>(u.u11, x1[j]));
                a[i0[j]] = y0;
                a[i0[j] + step] = y1;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// 1-bit gate, target bit < 6 (partner in the same wave)
// ---------------------------------------------------------------------------
template <typename R>
__device__ __forceinline__ cxt<R> shfl_xor_c(cxt<R> v, int m) {
    cxt<R> r;
    r.x = __shfl_xor(v.x, m, 64);
    r.y = __shfl_xor(v.y, m, 64);
    return r;
}

// Work index w covers all elements with the high control bits squeezed out
// (fx holds only control bits >= 6, so the low 6 bits of w are the lane's
// element offset inside an aligned 64-element chunk).  Low control bits are
// tested per element.
template <typename R, int EPT>
__global__ __launch_bounds__(kBlock) void k_gate1_lo(cxt<R>* __restrict__ a,
                                                      uint64_t nwork, int bit,
                                                      M2<R> u, Fixed fx,
                                                      uint64_t cval,
                                                      uint64_t lmask,
                                                      uint64_t lval) {
    const uint64_t nthreads = uint64_t(gridDim.x) * kBlock;
    const uint64_t tbit = uint64_t{1} << bit;
    // nwork is a multiple of 64 and every wave's indices are a full aligned
    // chunk, so all 64 lanes take part in each shuffle.
    for (uint64_t w0 = uint64_t(blockIdx.x) * kBlock + threadIdx.x; w0 < nwork;
         w0 += nthreads * EPT) {
        cxt<R> x[EPT];
        uint64_t e[EPT];
        bool ok[EPT];
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
            const uint64_t w = w0 + j * nthreads;
            ok[j] = w < nwork;
            e[j] = ok[j] ? (insert_zeros(w, fx.pos, fx.np) | cval) : 0;
            x[j].x = 0;
            x[j].y = 0;
            if (ok[j]) x[j] = a[e[j]];
        }
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
            // every lane joins the shuffle; a lane's partner (lane ^ tbit) is
            // in range whenever the lane is (nwork is a power of two > tbit)
            const cxt<R> y = shfl_xor_c<R>(x[j], int(tbit));
            if (ok[j]) {
                const bool one = (e[j] & tbit) != 0;
                const bool act = (e[j] & lmask) == lval;
                cxt<R> r;
                if (!one)
                    r = cfma<R>(u.u00, x[j], cmul<R>(u.u01, y));
                else
                    r = cfma<R>(u.u10, y, cmul<R>(u.u11, x[j]));
                if (act) a[e[j]] = r;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// 2- to 4-bit dense gates in registers
// ---------------------------------------------------------------------------
// A thread holds the 2^K amplitudes of one group in registers, multiplies
// them by the gate and stores them; HBM bounds it (16 FP64 FMA per amplitude
// at K = 2, 64 at K = 4, against 32 bytes).  Every load and store runs over
// 64 consecutive amplitudes: a target bit below 6 is one of the lane bits
// there, so its place among the register bits is taken by the lowest free
// bit above, and after the loads the two are exchanged (half of the
// registers with the lane across that bit), and back before the stores.
// Loading the groups of a low target directly instead would touch every
// line 2^K times.
//
// RHO: a density matrix's U rho U^dagger in one pass: the register bits are
// the K/2 column targets, then the K/2 row targets; U goes to the row bits
// where the row controls hold and conj(U) to the column bits where the
// column controls hold.  11 qubits complex128: 37 -> 18 us for one qubit (two
// passes before), 94-125 -> 20 us for two.
struct RegGate {
    Fixed fx;            // squeezed out of the group index: register bits, high controls
    uint64_t cval;       // the high controls' values
    uint64_t off[16];    // offset of register c (before the exchange)
    uint64_t mask[2], val[2];  // RHO: row and column controls; else mask[0]: low controls
    int8_t lane_bit[4];  // lane bit to exchange with register bit j, or -1
};

// N matrix entries, as a kernel's argument or behind a pointer
template <typename R, int N, bool BYVAL>
struct GateMatN {
    cxt<R> m[N];
    __device__ __forceinline__ cxt<R> at(int i) const { return m[i]; }
};
template <typename R, int N>
struct GateMatN<R, N, false> {
    const cxt<R>* m;
    __device__ __forceinline__ cxt<R> at(int i) const { return m[i]; }
};
template <typename R, int DIM, bool BYVAL>
using GateMat = GateMatN<R, DIM * DIM, BYVAL>;
// a matrix of up to 1 KiB travels in the kernel's arguments
template <typename R, int K, bool RHO>
using RegMat = GateMat<R, RHO ? (1 << (K / 2)) : (1 << K), RHO || K <= 3>;

template <typename R, int K>
__device__ __forceinline__ void exchange(cxt<R> (&x)[1 << K], const int8_t (&lane_bit)[4]) {
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const int b = lane_bit[j];
        if (b < 0) continue;
        const bool one = (threadIdx.x >> b) & 1;
#pragma unroll
        for (int c = 0; c < (1 << K); ++c) {
            if ((c >> j) & 1) continue;
            const cxt<R> lo = x[c], hi = x[c | (1 << j)];
            cxt<R> give;
            give.x = one ? lo.x : hi.x;
            give.y = one ? lo.y : hi.y;
            const cxt<R> got = shfl_xor_c<R>(give, 1 << b);
            x[c].x = one ? got.x : lo.x;
            x[c].y = one ? got.y : lo.y;
            x[c | (1 << j)].x = one ? hi.x : got.x;
            x[c | (1 << j)].y = one ? hi.y : got.y;
        }
    }
}

template <typename R, int K, bool RHO, int NG>
__global__ __launch_bounds__(kBlock) void k_gate_reg(cxt<R>* __restrict__ a, uint64_t ngroups, RegGate g,
                                                     RegMat<R, K, RHO> m) {
    constexpr int DIM = 1 << K;
    const uint64_t nthreads = uint64_t(gridDim.x) * kBlock;
    const uint64_t p = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    cxt<R> x[NG][DIM];
    uint64_t base[NG];
    bool act[NG], rows[NG], cols[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const uint64_t q = p + i * nthreads;
        base[i] = insert_zeros(q, g.fx.pos, g.fx.np) | g.cval;
        rows[i] = (base[i] & g.mask[0]) == g.val[0];
        cols[i] = RHO && (base[i] & g.mask[1]) == g.val[1];
        act[i] = q < ngroups && (rows[i] || cols[i]);
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
            x[i][c].x = 0;
            x[i][c].y = 0;
            if (act[i]) x[i][c] = a[base[i] + g.off[c]];
        }
    }
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        // (a lane and those it exchanges with have the same controls)
        exchange<R, K>(x[i], g.lane_bit);
        if constexpr (RHO) {
            constexpr int D = 1 << (K / 2);
            if (rows[i]) {
#pragma unroll
                for (int h = 0; h < D; ++h) {
                    cxt<R> in[D];
#pragma unroll
                    for (int c = 0; c < D; ++c) in[c] = x[i][h * D + c];
#pragma unroll
                    for (int r = 0; r < D; ++r) {
                        cxt<R> acc = cmul<R>(m.at(r), in[0]);
#pragma unroll
                        for (int c = 1; c < D; ++c) acc = cfma<R>(m.at(r + c * D), in[c], acc);
                        x[i][h * D + r] = acc;
                    }
                }
            }
            if (cols[i]) {
#pragma unroll
                for (int h = 0; h < D; ++h) {
                    cxt<R> in[D];
#pragma unroll
                    for (int c = 0; c < D; ++c) in[c] = x[i][c * D + h];
#pragma unroll
                    for (int r = 0; r < D; ++r) {
                        cxt<R> acc = cmul<R>(conj_c<R>(m.at(r)), in[0]);
#pragma unroll
                        for (int c = 1; c < D; ++c) acc = cfma<R>(conj_c<R>(m.at(r + c * D)), in[c], acc);
                        x[i][r * D + h] = acc;
                    }
                }
            }
        } else {
            cxt<R> y[DIM];
#pragma unroll
            for (int r = 0; r < DIM; ++r) y[r] = cmul<R>(m.at(r), x[i][0]);
#pragma unroll
            for (int c = 1; c < DIM; ++c)
#pragma unroll
                for (int r = 0; r < DIM; ++r) y[r] = cfma<R>(m.at(r + c * DIM), x[i][c], y[r]);
#pragma unroll
            for (int r = 0; r < DIM; ++r) x[i][r] = y[r];
        }
        exchange<R, K>(x[i], g.lane_bit);
#pragma unroll
        for (int c = 0; c < DIM; ++c)
            if (act[i]) a[base[i] + g.off[c]] = x[i][c];
    }
}

// ---------------------------------------------------------------------------
// k-bit dense gate through LDS
// ---------------------------------------------------------------------------
// Groups: the 2^k elements sharing all non-target bits.  The group index g
// enumerates spectator bits (targets and high controls squeezed out, control
// value OR-ed in); `inner[c]` is the offset of gate digit c (bits[0] = MSB).
// A block stages G = kBlock*EPT / 2^k groups.  Thread t loads element
// (c = t / G, g = t % G) so consecutive lanes read consecutive groups.
template <typename R, int EPT>
__global__ __launch_bounds__(kBlock) void k_gatek(
    cxt<R>* __restrict__ a, uint64_t ngroups, int k,
    const uint64_t* __restrict__ inner, const cxt<R>* __restrict__ m,
    Fixed fx, uint64_t cval, uint64_t lmask, uint64_t lval) {
    extern __shared__ unsigned char smem_raw[];
    cxt<R>* s = reinterpret_cast<cxt<R>*>(smem_raw);
    const int dim = 1 << k;
    const int G = (kBlock * EPT) >> k;  // groups per block (>= 1)
    for (uint64_t gb = uint64_t(blockIdx.x) * G; gb < ngroups;
         gb += uint64_t(gridDim.x) * G) {
        // stage
        for (int t = threadIdx.x; t < G * dim; t += kBlock) {
            const int c = t / G, gl = t % G;
            const uint64_t g = gb + gl;
            if (g < ngroups) {
                const uint64_t base = insert_zeros(g, fx.pos, fx.np) | cval;
                s[gl * dim + c] = a[base + inner[c]];
            }
        }
        __syncthreads();
        for (int t = threadIdx.x; t < G * dim; t += kBlock) {
            const int r = t / G, gl = t % G;
            const uint64_t g = gb + gl;
            if (g < ngroups) {
                const uint64_t base = insert_zeros(g, fx.pos, fx.np) | cval;
                if ((base & lmask) == lval) {
                    cxt<R> acc;
                    acc.x = 0;
                    acc.y = 0;
                    const cxt<R>* in = s + gl * dim;
                    // m is column-major: m[r + c*dim]
                    for (int c = 0; c < dim; ++c) acc = cfma<R>(m[r + c * dim], in[c], acc);
                    a[base + inner[r]] = acc;
                }
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// 5-bit dense gate with MFMA (complex64)
// ---------------------------------------------------------------------------
// The groups (columns) are as in k_gatek.  Over the real and imaginary parts
// the gate is one real GEMM, [Yr; Yi] = W [Xr; Xi] with W = [[Ur, -Ui],
// [Ui, Ur]] (2 DIM x 2 DIM, DIM = 2^K), and every wave step multiplies W by
// 16 groups with v_mfma_f32_16x16x4f32 (D[16x16] += A[16x4] B[4x16]; lane l
// holds A[l%16][l/16], B[l/16][l%16] and D[4(l/16)+v][l%16], v = 0..3):
//   B: lane (g = l/16, j = l%16) holds real row 4s+g of group j for slice
//      s; it loads the complex amplitudes 4q+g of its group, whose real
//      parts are slices q and whose imaginary parts are slices DIM/4+q;
//   A: W in 16-row blocks mb and 4-column slices s, each lane's entries
//      packed by the host in that order and read from LDS;
//   D: row block mb < NB/2 holds real parts and mb + NB/2 the imaginary
//      parts of the same complex rows 16 mb + 4 g + v, so each lane writes
//      whole complex amplitudes.
// Arithmetic per amplitude: 4 DIM FP32 FMA, as many as the complex product
// takes on VALU, at twice the VALU FP32 rate (packed FP32 aside).
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr uint32_t kMfmaGrid = 2048;

template <int K>
__global__ __launch_bounds__(kBlock) void k_gatek_mfma(float2* __restrict__ a, uint64_t ncols,
                                                       const uint64_t* __restrict__ inner,
                                                       const float* __restrict__ wpack, Fixed fx,
                                                       uint64_t cval) {
    constexpr int DIM = 1 << K;
    constexpr int NX = DIM / 4;       // complex inputs per lane
    constexpr int NS = 2 * NX;        // slices of 4 real columns of W
    constexpr int NB = 2 * DIM / 16;  // blocks of 16 real rows of W
    constexpr int NO = NB / 2;        // output row blocks (complex)
    const int lane = threadIdx.x & 63;
    const int j = lane & 15, g = lane >> 4;
    // the packed matrix in LDS, shared by the workgroup's waves (registers
    // go to the amplitudes in flight instead)
    __shared__ float wl[NB * NS * 64];
    for (int i = threadIdx.x; i < NB * NS * 64; i += kBlock) wl[i] = wpack[i];
    __syncthreads();
    uint64_t in_off[NX], out_off[NO][4];
#pragma unroll
    for (int q = 0; q < NX; ++q) in_off[q] = inner[4 * q + g];
#pragma unroll
    for (int mh = 0; mh < NO; ++mh)
#pragma unroll
        for (int v = 0; v < 4; ++v) out_off[mh][v] = inner[16 * mh + 4 * g + v];
    constexpr int kWaves = kBlock / 64;
    const uint64_t nwaves = uint64_t(gridDim.x) * kWaves;
    // a wave's group `grp` covers columns 16 grp .. 16 grp + 15.  The
    // groups after the current one are loaded before its products, into
    // register buffers taken in turn (the loop unrolled, so no buffer is
    // copied and no load has to land before its own group's turn)
    struct Buf {
        float xr[NX], xi[NX];
        uint64_t base;
        bool ok;
    };
    // a lane past the last column loads column 0's amplitudes (in bounds,
    // no branch around the loads) and stores nothing
    auto fetch = [&](uint64_t grp, Buf& b) {
        const uint64_t col = grp * 16 + j;
        b.ok = col < ncols;
        b.base = insert_zeros(b.ok ? col : 0, fx.pos, fx.np) | cval;
#pragma unroll
        for (int q = 0; q < NX; ++q) {
            const float2 v = a[b.base + in_off[q]];
            b.xr[q] = v.x;
            b.xi[q] = v.y;
        }
    };
    auto process = [&](const Buf& b) {
        floatx4 acc[NB];
#pragma unroll
        for (int mb = 0; mb < NB; ++mb) acc[mb] = floatx4{0.f, 0.f, 0.f, 0.f};
        // slice s's matrix entries are read while slice s-1's products run.
        // The matrix is read again at every group: an offset the compiler
        // cannot see through (zero, from an instruction it must keep) stops
        // it from hoisting all 2 DIM^2 / 16 entries into registers, and the
        // scheduling barrier from issuing every slice's reads at once.
        int z;
        asm volatile("s_mov_b32 %0, 0" : "=s"(z));
        const float* wv = wl + z;
        float wc[NB], wn[NB];
#pragma unroll
        for (int mb = 0; mb < NB; ++mb) wc[mb] = wv[mb * NS * 64 + lane];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (s + 1 < NS) {
#pragma unroll
                for (int mb = 0; mb < NB; ++mb) wn[mb] = wv[(mb * NS + s + 1) * 64 + lane];
            }
            const float bx = s < NX ? b.xr[s] : b.xi[s - NX];
#pragma unroll
            for (int mb = 0; mb < NB; ++mb)
                acc[mb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[mb], bx, acc[mb], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int mb = 0; mb < NB; ++mb) wc[mb] = wn[mb];
        }
        if (b.ok) {
#pragma unroll
            for (int mh = 0; mh < NO; ++mh)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    a[b.base + out_off[mh][v]] = make_float2(acc[mh][v], acc[mh + NO][v]);
        }
    };
    uint64_t grp = uint64_t(blockIdx.x) * kWaves + threadIdx.x / 64;
    if (grp * 16 >= ncols) return;
    // every fetch is issued, past the wave's last group on its current
    // group again (in bounds, never used): with no load under a branch the
    // waits before each group's products count exactly the loads and
    // stores issued after its own loads
    // 8 amplitudes per lane and group, 4 waves per SIMD: the next two
    // groups in flight (three buffers in turn)
    Buf b0, b1, b2;
    fetch(grp, b0);
    bool has1 = (grp + nwaves) * 16 < ncols;
    fetch(has1 ? grp + nwaves : grp, b1);
    // `cur` holds group grp, the next buffer group grp + nwaves (when
    // has1), and `far` receives group grp + 2 nwaves; false once grp was
    // the last
    auto step = [&](const Buf& cur, Buf& far) {
        const bool has2 = (grp + 2 * nwaves) * 16 < ncols;
        fetch(has2 ? grp + 2 * nwaves : grp, far);
        process(cur);
        if (!has1) return false;
        grp += nwaves;
        has1 = has2;
        return true;
    };
    for (;;) {
        if (!step(b0, b2)) break;
        if (!step(b1, b0)) break;
        if (!step(b2, b1)) break;
    }
}

// ---------------------------------------------------------------------------
// qudit (mixed-radix) gate
// ---------------------------------------------------------------------------
struct QG {
    uint32_t ntg, nsp, nctrl;
    uint64_t tg_stride[16], tg_dim[16];
    uint64_t sp_stride[40], sp_dim[40];
    uint64_t c_stride[40], c_shift[40];
    uint64_t c_dim;
    uint64_t DA;
};

// One thread per spectator index: gather DA elements (<= 64) from the
// target-digit offsets, apply A^r, scatter.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_qudit(cxt<R>* __restrict__ a,
                                                   uint64_t nspec, QG q,
                                                   const cxt<R>* __restrict__ mats,
                                                   const uint64_t* __restrict__ off) {
    const uint64_t nthreads = uint64_t(gridDim.x) * kBlock;
    for (uint64_t s = uint64_t(blockIdx.x) * kBlock + threadIdx.x; s < nspec;
         s += nthreads) {
        uint64_t base = 0, rem = s;
        for (int j = int(q.nsp) - 1; j >= 0; --j) {
            base += (rem % q.sp_dim[j]) * q.sp_stride[j];
            rem /= q.sp_dim[j];
        }
        uint64_t r = 1;  // exponent of A (1 when uncontrolled)
        if (q.nctrl) {
            r = ((base / q.c_stride[0]) % q.c_dim + q.c_shift[0]) % q.c_dim;
            for (uint32_t c = 1; c < q.nctrl; ++c)
                if (((base / q.c_stride[c]) % q.c_dim + q.c_shift[c]) % q.c_dim != r)
                    r = 0;
        }
        if (r == 0) continue;  // A^0 = identity
        const cxt<R>* m = mats + (q.nctrl ? r : 0) * q.DA * q.DA;
        cxt<R> in[64];
        for (uint64_t c = 0; c < q.DA; ++c) in[c] = a[base + off[c]];
        for (uint64_t rr = 0; rr < q.DA; ++rr) {
            cxt<R> acc;
            acc.x = 0;
            acc.y = 0;
            for (uint64_t c = 0; c < q.DA; ++c) acc = cfma<R>(m[rr + c * q.DA], in[c], acc);
            a[base + off[rr]] = acc;
        }
    }
}

// The same with the group in registers and the spectator digits by 32-bit
// reciprocals, for the gate dimensions of one and two qudits (2 to 5 states
// each).  cshift[k] is digit k's control shift, or -1 for a spectator that
// controls nothing.  Threads of a wave with different powers of A take them
// in turn, so that the matrix is always uniform (scalar loads).  14 qutrits
// complex128: 100 -> 27 us a gate on one, 48 on two; HBM bounds it.  Wider
// gates, on two qudits of different dimensions or three of any, stay with
// k_qudit: a group of 27 and more complex128 amplitudes leaves few waves to a
// SIMD, and those widths have not been measured here.
struct QGFast {
    Digits sp;
    int32_t cshift[kMaxDigits];
    uint32_t nctrl, c_dim;
    uint64_t off[25];  // offsets of the gate's digits
};

// the matrices in the kernel's arguments where they fit 2 KiB (GateMat)
constexpr int kQuditMats = 128;

template <typename R, int DA, bool BYVAL>
__global__ __launch_bounds__(kBlock) void k_qudit_reg(cxt<R>* __restrict__ a, uint32_t nspec, QGFast q,
                                                      GateMatN<R, kQuditMats, BYVAL> mats) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    uint64_t base = 0;
    int r = -1;  // the controls' common value (the power of A)
    uint32_t v = s;
    for (int k = int(q.sp.n) - 1; k >= 0; --k) {
        const uint32_t up = __umulhi(v, q.sp.mag[k]);
        const uint32_t dig = v - up * q.sp.dim[k];
        base += uint64_t(dig) * q.sp.str[k];
        v = up;
        if (q.cshift[k] >= 0) {
            const int c = int((dig + uint32_t(q.cshift[k])) % q.c_dim);
            r = r < 0 || r == c ? c : 0;
            if (r == 0) break;  // A^0, or controls that differ
        }
    }
    const bool act = s < nspec && r != 0;
    cxt<R> x[DA];
#pragma unroll
    for (int c = 0; c < DA; ++c)
        if (act) x[c] = a[base + q.off[c]];
    const uint32_t top = q.nctrl ? q.c_dim : 1;
    for (uint32_t w = q.nctrl ? 1 : 0; w < top; ++w) {
        if (!act || (q.nctrl && uint32_t(r) != w)) continue;
        const int m = int(w) * DA * DA;
#pragma unroll 1
        for (int rr = 0; rr < DA; ++rr) {
            cxt<R> acc = cmul<R>(mats.at(m + rr), x[0]);
#pragma unroll
            for (int c = 1; c < DA; ++c) acc = cfma<R>(mats.at(m + rr + c * DA), x[c], acc);
            a[base + q.off[rr]] = acc;
        }
    }
}

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------
uint32_t grid_for(uint64_t work, uint64_t per_block) {
    uint64_t b = (work + per_block - 1) / per_block;
    if (b < 1) b = 1;
    if (b > (uint64_t{1} << 30)) b = uint64_t{1} << 30;
    return static_cast<uint32_t>(b);
}

template <typename R>
cxt<R> to_c(const double* m, uint64_t idx, bool conj) {
    cxt<R> v;
    v.x = static_cast<R>(m[2 * idx]);
    v.y = static_cast<R>(conj ? -m[2 * idx + 1] : m[2 * idx + 1]);
    return v;
}

template <typename R>
M2<R> make_m2(const double* m, bool conj) {
    // column-major input: m[r + 2c]
    M2<R> u;
    u.u00 = to_c<R>(m, 0, conj);
    u.u10 = to_c<R>(m, 1, conj);
    u.u01 = to_c<R>(m, 2, conj);
    u.u11 = to_c<R>(m, 3, conj);
    return u;
}

Fixed make_fixed(std::vector<uint32_t> pos) {
    std::sort(pos.begin(), pos.end());
    Fixed f;
    f.np = static_cast<int>(pos.size());
    for (size_t i = 0; i < pos.size(); ++i) f.pos[i] = static_cast<uint8_t>(pos[i]);
    return f;
}

std::vector<uint32_t> bits_of(uint64_t mask) {
    std::vector<uint32_t> v;
    for (uint32_t b = 0; b < 64; ++b)
        if ((mask >> b) & 1) v.push_back(b);
    return v;
}

template <typename R>
int gate1_impl(qs_state* st, uint32_t bit, const double* m, uint64_t cmask,
               uint64_t cval, bool conj) {
    const M2<R> u = make_m2<R>(m, conj);
    auto* a = static_cast<cxt<R>*>(st->d);
    const uint32_t nb = st->nbits;
    if (bit >= 6) {
        std::vector<uint32_t> fixed = bits_of(cmask);
        fixed.push_back(bit);
        const Fixed fx = make_fixed(fixed);
        const uint64_t npairs = uint64_t{1} << (nb - fx.np);
        constexpr int PPT = 4;
        const uint32_t grid = grid_for(npairs, uint64_t(kBlock) * PPT);
        hipLaunchKernelGGL((k_gate1_hi<R, PPT>), dim3(grid), dim3(kBlock), 0,
                           st->stream, a, npairs, uint64_t{1} << bit, u, fx,
                           cval & ~(uint64_t{1} << bit));
    } else {
        // controls above bit 5 are squeezed out, the others tested in-lane
        const uint64_t hmask = cmask & ~uint64_t{63};
        const uint64_t lmask = cmask & uint64_t{63};
        const Fixed fx = make_fixed(bits_of(hmask));
        const uint64_t nwork = uint64_t{1} << (nb - fx.np);
        constexpr int EPT = 4;
        const uint32_t grid = grid_for(nwork, uint64_t(kBlock) * EPT);
        hipLaunchKernelGGL((k_gate1_lo<R, EPT>), dim3(grid), dim3(kBlock), 0,
                           st->stream, a, nwork, int(bit), u, fx, cval & hmask,
                           lmask, cval & lmask);
    }
    return QS_OK;
}

// Up to 3 KiB of a host table, carried in a kernel's arguments to device
// memory: ordered on the stream without the host waiting for a copy.
struct PutChunk {
    uint32_t w[768];
};
__global__ __launch_bounds__(256) void k_put(uint32_t* __restrict__ d, PutChunk c, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += 256) d[i] = c.w[i];
}

// Device copy of a host table of one call (matrices, offsets), a multiple of
// 4 bytes.  Up to kTabBytes it goes into the state's own table memory, which
// its next call overwrites in stream order (the caller holds tab_mutex until
// the kernel that reads it is launched): a few launches, where an
// allocation, a pageable copy, its wait and the free took 25 us (16 KiB: six
// launches).  Larger tables are copied into memory of their own (*owned),
// freed stream-ordered after the kernel.
constexpr size_t kTabBytes = 24576;

int upload(qs_state* st, const void* host, size_t bytes, void** dptr, void** owned) {
    constexpr const char* W = "qpp_amd::upload";
    *owned = nullptr;
    if (bytes <= kTabBytes) {
        if (!st->tab) QS_HIP(hipMallocAsync(&st->tab, kTabBytes, st->stream), W);
        *dptr = st->tab;
        PutChunk c;
        for (size_t at = 0; at < bytes; at += sizeof(c)) {
            const size_t part = std::min(sizeof(c), bytes - at);
            std::memcpy(c.w, static_cast<const char*>(host) + at, part);
            hipLaunchKernelGGL(k_put, dim3(1), dim3(256), 0, st->stream,
                               reinterpret_cast<uint32_t*>(static_cast<char*>(st->tab) + at), c,
                               static_cast<uint32_t>(part / 4));
        }
        QS_HIP(hipGetLastError(), W);
        return QS_OK;
    }
    QS_HIP(hipMallocAsync(owned, bytes, st->stream), W);
    *dptr = *owned;
    hipError_t e = hipMemcpyAsync(*owned, host, bytes, hipMemcpyHostToDevice, st->stream);
    // pageable source: make sure the copy has consumed `host` before return
    if (e == hipSuccess) e = hipStreamSynchronize(st->stream);
    if (e != hipSuccess) {
        (void)hipFreeAsync(*owned, st->stream);
        return qs::fail_hip(e, W);
    }
    return QS_OK;
}

// Descriptor of k_gate_reg: `regs` the bits of register bits K-1 .. 0, the
// controls as masks of the index (RHO: rows then columns).
RegGate reg_gate(uint32_t nb, const uint32_t* regs, uint32_t K, bool rho, const uint64_t (&cmask)[2],
                 const uint64_t (&cval)[2], uint64_t* ngroups) {
    RegGate g{};
    const uint64_t ctrl = cmask[0] | cmask[1];
    uint64_t used = ctrl;
    uint32_t low = 0;
    for (uint32_t j = 0; j < K; ++j) {
        used |= uint64_t{1} << regs[j];
        low += regs[j] < 6;
    }
    std::vector<uint32_t> free_bits;
    for (uint32_t b = 6; b < nb && free_bits.size() < low; ++b)
        if (!((used >> b) & 1)) free_bits.push_back(b);
    // a register too small for whole waves of groups takes one group a lane
    // with the targets where they are
    const bool lanes = free_bits.size() == low && nb >= 6;
    const uint64_t squeezed = rho ? 0 : lanes ? ctrl & ~uint64_t{63} : ctrl;
    std::vector<uint32_t> fixed = bits_of(squeezed);
    uint32_t next = 0;
    for (uint32_t j = 0; j < 4; ++j) g.lane_bit[j] = -1;
    uint64_t bit_off[4] = {};
    for (uint32_t j = 0; j < K; ++j) {
        uint32_t b = regs[K - 1 - j];  // register bit j
        if (lanes && b < 6) {
            g.lane_bit[j] = static_cast<int8_t>(b);
            b = free_bits[next++];
        }
        fixed.push_back(b);
        bit_off[j] = uint64_t{1} << b;
    }
    for (uint32_t c = 0; c < (1u << K); ++c)
        for (uint32_t j = 0; j < K; ++j)
            if ((c >> j) & 1) g.off[c] |= bit_off[j];
    g.fx = make_fixed(fixed);
    g.cval = cval[0] & squeezed;
    for (int i = 0; i < 2; ++i) {
        g.mask[i] = cmask[i] & ~squeezed;
        g.val[i] = cval[i] & g.mask[i];
    }
    *ngroups = uint64_t{1} << (nb - g.fx.np);
    return g;
}

template <typename R, int K, bool RHO>
int gate_reg(qs_state* st, const uint32_t* regs, const double* m, bool conj, const uint64_t (&cmask)[2],
             const uint64_t (&cval)[2]) {
    constexpr int DIM = RHO ? 1 << (K / 2) : 1 << K;
    uint64_t ngroups = 0;
    const RegGate g = reg_gate(st->nbits, regs, K, RHO, cmask, cval, &ngroups);
    // small groups: 128 bytes of loads in flight per thread
    constexpr int NG = K >= 4 ? 1 : (sizeof(R) == 8 ? 8 : 16) >> K;
    const uint32_t grid = grid_for(ngroups, uint64_t(kBlock) * NG);
    auto* a = static_cast<cxt<R>*>(st->d);
    RegMat<R, K, RHO> mat;
    if constexpr (RHO || K <= 3) {
        for (int i = 0; i < DIM * DIM; ++i) mat.m[i] = to_c<R>(m, i, conj);
        hipLaunchKernelGGL((k_gate_reg<R, K, RHO, NG>), dim3(grid), dim3(kBlock), 0, st->stream, a, ngroups, g,
                           mat);
        return QS_OK;
    } else {
        cxt<R> mm[DIM * DIM];
        for (int i = 0; i < DIM * DIM; ++i) mm[i] = to_c<R>(m, i, conj);
        const std::lock_guard<std::mutex> hold(st->tab_mutex);
        void *d = nullptr, *owned = nullptr;
        static_assert(sizeof(mm) <= kTabBytes, "in the state's table memory");
        if (int rc = upload(st, mm, sizeof(mm), &d, &owned)) return rc;
        mat.m = static_cast<const cxt<R>*>(d);
        hipLaunchKernelGGL((k_gate_reg<R, K, RHO, NG>), dim3(grid), dim3(kBlock), 0, st->stream, a, ngroups, g,
                           mat);
        return QS_OK;
    }
}

int gatek_mfma(qs_state* st, uint32_t k, const std::vector<uint64_t>& inner, const double* m,
               bool conj, const Fixed& fx, uint64_t cval, uint64_t ncols);

template <typename R>
int gatek_impl(qs_state* st, const uint32_t* bits, uint32_t k, const double* m,
               uint64_t cmask, uint64_t cval, bool conj) {
    constexpr bool f64 = std::is_same<R, double>::value;
    const uint64_t cm[2] = {cmask, 0}, cv[2] = {cval, 0};
    if (k == 2) return gate_reg<R, 2, false>(st, bits, m, conj, cm, cv);
    if (k == 3) return gate_reg<R, 3, false>(st, bits, m, conj, cm, cv);
    if (k == 4 && (f64 || !qs::gatek_valu_forced())) return gate_reg<R, 4, false>(st, bits, m, conj, cm, cv);
    const uint32_t dim = 1u << k;
    std::vector<uint64_t> inner(dim);
    for (uint32_t c = 0; c < dim; ++c) {
        uint64_t v = 0;
        for (uint32_t j = 0; j < k; ++j)
            if ((c >> j) & 1) v |= uint64_t{1} << bits[k - 1 - j];
        inner[c] = v;
    }
    std::vector<cxt<R>> mm(uint64_t(dim) * dim);
    for (uint64_t i = 0; i < mm.size(); ++i) mm[i] = to_c<R>(m, i, conj);
    // squeeze targets and control bits that are not targets
    std::vector<uint32_t> fixed(bits, bits + k);
    for (uint32_t b : bits_of(cmask)) fixed.push_back(b);
    const Fixed fx = make_fixed(fixed);
    const uint64_t ngroups = uint64_t{1} << (st->nbits - fx.np);
    if constexpr (!f64)
        if (k == 5 && !qs::gatek_valu_forced())
            return gatek_mfma(st, k, inner, m, conj, fx, cval, ngroups);
    const size_t inner_bytes = inner.size() * sizeof(uint64_t);
    const size_t mat_bytes = mm.size() * sizeof(cxt<R>);
    std::vector<unsigned char> blob(inner_bytes + mat_bytes);
    std::memcpy(blob.data(), inner.data(), inner_bytes);
    std::memcpy(blob.data() + inner_bytes, mm.data(), mat_bytes);
    const std::lock_guard<std::mutex> hold(st->tab_mutex);
    void *dblob = nullptr, *owned = nullptr;
    if (int rc = upload(st, blob.data(), blob.size(), &dblob, &owned)) return rc;
    constexpr int EPT = 4;
    // groups per block must be >= 1: for dim > kBlock*EPT use larger EPT
    int G = (kBlock * EPT) >> k;
    if (G < 1) return qs::fail(QS_ERR_NOT_IMPLEMENTED, "qpp::apply()",
                               "gate wider than 10 qubits");
    const uint32_t grid = grid_for(ngroups, uint64_t(G));
    const size_t shmem = size_t(G) * dim * sizeof(cxt<R>);
    hipLaunchKernelGGL((k_gatek<R, EPT>), dim3(grid), dim3(kBlock), shmem,
                       st->stream, static_cast<cxt<R>*>(st->d), ngroups, int(k),
                       static_cast<const uint64_t*>(dblob),
                       reinterpret_cast<const cxt<R>*>(
                           static_cast<unsigned char*>(dblob) + inner_bytes),
                       fx, cval, uint64_t{0}, uint64_t{0});
    if (owned) QS_HIP(hipFreeAsync(owned, st->stream), "qpp_amd::apply");
    return QS_OK;
}

// W = [[Ur, -Ui], [Ui, Ur]] (m column-major complex, conj: conj(U)) packed
// in k_gatek_mfma's A-operand order: entry (mb, s, lane) = W[16 mb + lane %
// 16][4 s + lane / 16].
int gatek_mfma(qs_state* st, uint32_t k, const std::vector<uint64_t>& inner, const double* m,
               bool conj, const Fixed& fx, uint64_t cval, uint64_t ncols) {
    const int dim = 1 << k, nr = 2 * dim, ns = nr / 4, nb = nr / 16;
    auto W = [&](int r, int c) -> float {
        const int rr = r % dim, cc = c % dim;
        const double re = m[2 * (rr + cc * dim)];
        const double im = conj ? -m[2 * (rr + cc * dim) + 1] : m[2 * (rr + cc * dim) + 1];
        if ((r < dim) == (c < dim)) return static_cast<float>(re);
        return static_cast<float>(r < dim ? -im : im);
    };
    std::vector<float> wp(size_t(nb) * ns * 64);
    for (int mb = 0; mb < nb; ++mb)
        for (int s = 0; s < ns; ++s)
            for (int l = 0; l < 64; ++l) wp[(size_t(mb) * ns + s) * 64 + l] = W(16 * mb + l % 16, 4 * s + l / 16);
    const size_t inner_bytes = inner.size() * sizeof(uint64_t);
    std::vector<unsigned char> blob(inner_bytes + wp.size() * sizeof(float));
    std::memcpy(blob.data(), inner.data(), inner_bytes);
    std::memcpy(blob.data() + inner_bytes, wp.data(), wp.size() * sizeof(float));
    // persistent waves (each walks many groups, two ahead in flight): no
    // more workgroups than are resident at once, so none starts late
    const uint64_t groups16 = (ncols + 15) / 16;
    int per_cu = 0, dev = 0, ncu = 0;
    QS_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_gatek_mfma<5>,
                                                        kBlock, 0),
           "qpp::apply()");
    QS_HIP(hipGetDevice(&dev), "qpp::apply()");
    QS_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev), "qpp::apply()");
    const uint32_t resident = static_cast<uint32_t>(std::max(1, per_cu) * std::max(1, ncu));
    const uint32_t grid = std::min<uint32_t>(grid_for(groups16, kBlock / 64), std::min(kMfmaGrid, resident));
    const std::lock_guard<std::mutex> hold(st->tab_mutex);
    void *dblob = nullptr, *owned = nullptr;
    if (int rc = upload(st, blob.data(), blob.size(), &dblob, &owned)) return rc;
    auto* inn = static_cast<const uint64_t*>(dblob);
    auto* wpk = reinterpret_cast<const float*>(static_cast<unsigned char*>(dblob) + inner_bytes);
    hipLaunchKernelGGL(k_gatek_mfma<5>, dim3(grid), dim3(kBlock), 0, st->stream,
                       static_cast<float2*>(st->d), ncols, inn, wpk, fx, cval);
    QS_HIP(hipGetLastError(), "qpp::apply()");
    if (owned) QS_HIP(hipFreeAsync(owned, st->stream), "qpp_amd::apply");
    return QS_OK;
}

// *took: whether k_qudit_reg took the gate
template <typename R>
int qudit_reg(qs_state* st, const qs::QuditGate& g, const std::vector<uint64_t>& off, uint64_t DA,
              uint64_t nspec, const std::vector<cxt<R>>& mm, bool* took) {
    QGFast f{};
    *took = false;
    DigitList sp;
    for (uint32_t i = 0; i < g.nsp; ++i) sp.emplace_back(g.sp_dim[i], g.sp_stride[i]);
    if (!digits_fit(sp, &f.sp) || DA > 25) return QS_OK;
    for (uint32_t k = 0; k < f.sp.n; ++k) {
        f.cshift[k] = -1;
        for (uint32_t c = 0; c < g.nctrl; ++c)
            if (f.sp.str[k] == g.c_stride[c]) f.cshift[k] = static_cast<int32_t>(g.c_shift[c]);
    }
    // controls of dimension 1 are no digit (their power is A^0): not here
    if (g.nctrl && g.c_dim < 2) return QS_OK;
    f.nctrl = g.nctrl;
    f.c_dim = static_cast<uint32_t>(g.c_dim);
    std::copy(off.begin(), off.end(), f.off);
    auto* a = static_cast<cxt<R>*>(st->d);
    const dim3 grid(grid_for(nspec, kBlock));
    const auto ns = static_cast<uint32_t>(nspec);
    auto go = [&](auto by_value, auto by_pointer) -> int {
        *took = true;
        if (mm.size() <= kQuditMats) {
            GateMatN<R, kQuditMats, true> m;
            std::copy(mm.begin(), mm.end(), m.m);
            hipLaunchKernelGGL(by_value, grid, dim3(kBlock), 0, st->stream, a, ns, f, m);
            return QS_OK;
        }
        const std::lock_guard<std::mutex> hold(st->tab_mutex);
        void *d = nullptr, *owned = nullptr;
        if (int rc = upload(st, mm.data(), mm.size() * sizeof(cxt<R>), &d, &owned)) return rc;
        GateMatN<R, kQuditMats, false> m;
        m.m = static_cast<const cxt<R>*>(d);
        hipLaunchKernelGGL(by_pointer, grid, dim3(kBlock), 0, st->stream, a, ns, f, m);
        if (owned) (void)hipFreeAsync(owned, st->stream);
        return QS_OK;
    };
    switch (DA) {
        case 2: return go(k_qudit_reg<R, 2, true>, k_qudit_reg<R, 2, false>);
        case 3: return go(k_qudit_reg<R, 3, true>, k_qudit_reg<R, 3, false>);
        case 4: return go(k_qudit_reg<R, 4, true>, k_qudit_reg<R, 4, false>);
        case 5: return go(k_qudit_reg<R, 5, true>, k_qudit_reg<R, 5, false>);
        case 6: return go(k_qudit_reg<R, 6, true>, k_qudit_reg<R, 6, false>);
        case 9: return go(k_qudit_reg<R, 9, true>, k_qudit_reg<R, 9, false>);
        case 16: return go(k_qudit_reg<R, 16, true>, k_qudit_reg<R, 16, false>);
        case 25: return go(k_qudit_reg<R, 25, true>, k_qudit_reg<R, 25, false>);
        default: return QS_OK;
    }
}

template <typename R>
int qudit_impl(qs_state* st, const qs::QuditGate& g, const double* mats,
               uint32_t nmats, uint64_t DA, bool conj) {
    if (DA > 64)
        return qs::fail(QS_ERR_NOT_IMPLEMENTED, "qpp::apply()",
                        "qudit gate dimension above 64");
    QG q{};
    q.ntg = g.ntg;
    q.nsp = g.nsp;
    q.nctrl = g.nctrl;
    for (uint32_t i = 0; i < g.ntg; ++i) q.tg_stride[i] = g.tg_stride[i], q.tg_dim[i] = g.tg_dim[i];
    if (g.nsp > 40 || g.nctrl > 40)
        return qs::fail(QS_ERR_NOT_IMPLEMENTED, "qpp::apply()", "too many subsystems");
    uint64_t nspec = 1;
    for (uint32_t i = 0; i < g.nsp; ++i) {
        q.sp_stride[i] = g.sp_stride[i];
        q.sp_dim[i] = g.sp_dim[i];
        nspec *= g.sp_dim[i];
    }
    for (uint32_t i = 0; i < g.nctrl; ++i) q.c_stride[i] = g.c_stride[i], q.c_shift[i] = g.c_shift[i];
    q.c_dim = g.c_dim;
    q.DA = DA;
    // offsets of the gate digits (target[0] most significant)
    std::vector<uint64_t> off(DA);
    for (uint64_t mi = 0; mi < DA; ++mi) {
        uint64_t rem = mi, v = 0;
        for (int j = int(g.ntg) - 1; j >= 0; --j) {
            v += (rem % g.tg_dim[j]) * g.tg_stride[j];
            rem /= g.tg_dim[j];
        }
        off[mi] = v;
    }
    std::vector<cxt<R>> mm(uint64_t(nmats) * DA * DA);
    for (uint64_t i = 0; i < mm.size(); ++i) mm[i] = to_c<R>(mats, i, conj);
    bool took = false;
    if (int rc = qudit_reg<R>(st, g, off, DA, nspec, mm, &took)) return rc;
    if (took) return QS_OK;
    const size_t off_bytes = off.size() * sizeof(uint64_t);
    const size_t mat_bytes = mm.size() * sizeof(cxt<R>);
    std::vector<unsigned char> blob(off_bytes + mat_bytes);
    std::memcpy(blob.data(), off.data(), off_bytes);
    std::memcpy(blob.data() + off_bytes, mm.data(), mat_bytes);
    const std::lock_guard<std::mutex> hold(st->tab_mutex);
    void *dblob = nullptr, *owned = nullptr;
    if (int rc = upload(st, blob.data(), blob.size(), &dblob, &owned)) return rc;
    const auto* dmats = reinterpret_cast<const cxt<R>*>(static_cast<unsigned char*>(dblob) + off_bytes);
    const uint32_t grid = grid_for(nspec, kBlock);
    hipLaunchKernelGGL((k_qudit<R>), dim3(grid), dim3(kBlock), 0, st->stream,
                       static_cast<cxt<R>*>(st->d), nspec, q, dmats, static_cast<const uint64_t*>(dblob));
    if (owned) QS_HIP(hipFreeAsync(owned, st->stream), "qpp_amd::apply");
    return QS_OK;
}

}  // namespace

namespace qs {

int launch_gate1(qs_state* st, uint32_t bit, const double* m, uint64_t cmask,
                 uint64_t cval, bool conj) {
    int rc = st->dtype == QS_C128
                 ? gate1_impl<double>(st, bit, m, cmask, cval, conj)
                 : gate1_impl<float>(st, bit, m, cmask, cval, conj);
    if (rc) return rc;
    QS_HIP(hipGetLastError(), "qpp::apply()");
    return QS_OK;
}

int launch_gatek(qs_state* st, const uint32_t* bits, uint32_t k,
                 const double* m, uint64_t cmask, uint64_t cval, bool conj) {
    if (k == 1) return launch_gate1(st, bits[0], m, cmask, cval, conj);
    int rc = st->dtype == QS_C128
                 ? gatek_impl<double>(st, bits, k, m, cmask, cval, conj)
                 : gatek_impl<float>(st, bits, k, m, cmask, cval, conj);
    if (rc) return rc;
    QS_HIP(hipGetLastError(), "qpp::apply()");
    return QS_OK;
}

int launch_gate_rho(qs_state* st, const uint32_t* bits, uint32_t k, const double* m,
                    const uint64_t (&cmask)[2], const uint64_t (&cval)[2]) {
    int rc = QS_OK;
    if (k == 1)
        rc = st->dtype == QS_C128 ? gate_reg<double, 2, true>(st, bits, m, false, cmask, cval)
                                  : gate_reg<float, 2, true>(st, bits, m, false, cmask, cval);
    else
        rc = st->dtype == QS_C128 ? gate_reg<double, 4, true>(st, bits, m, false, cmask, cval)
                                  : gate_reg<float, 4, true>(st, bits, m, false, cmask, cval);
    if (rc) return rc;
    QS_HIP(hipGetLastError(), "qpp::apply()");
    return QS_OK;
}

int launch_qudit_gate(qs_state* st, const QuditGate& g, const double* mats,
                      uint32_t nmats, uint64_t DA, bool conj) {
    int rc = st->dtype == QS_C128 ? qudit_impl<double>(st, g, mats, nmats, DA, conj)
                                  : qudit_impl<float>(st, g, mats, nmats, DA, conj);
    if (rc) return rc;
    QS_HIP(hipGetLastError(), "qpp::apply()");
    return QS_OK;
}

}  // namespace qs
