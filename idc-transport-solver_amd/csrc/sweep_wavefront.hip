// "hip-wavefront" traversal: one workgroup per ordinate walking the diagonals (k_sweep_rows), or, for meshes with more
// rows than it takes, one launch per spatial diagonal, all four quadrants in the same launch (k_sweep_diag).
//
// Mirrors SweepPatternUniCartWavefront::Sweep (SweepPatternUniCartWavefront.cpp:253-296): for
// diag = 1 .. nx+ny-1, every (cell on the diagonal, ordinate) pair is independent; the quadrant of
// the ordinate flips the cell index so each quadrant walks the mesh from its own inflow corner.
// Thread t of a launch of the latter handles cell c = t / nq of the diagonal and ordinate q = t % nq, so the
// lanes of a wavefront cover consecutive ordinates of a quadrant, whose N coefficients are
// contiguous in the [i][j][q][d][e] layout.  Upwind values are the neighbours written by the
// previous launch (L2 resident); the source of the cell is read before it is overwritten.
#include "cell_solve.hpp"
#include "tsw_internal.hpp"

namespace tsw {

// The cell matrix from sigma_t, its cell mean sig or (not null) its tensor tc.
template <typename T, int P>
__device__ __forceinline__ void cell_matrix(T (&A)[P * P * P * P], const SweepParams<T> &sp, T xi, T eta, T sig,
                                            const T *__restrict__ tc) {
    constexpr int N = P * P;
    if (!tc) {
        assemble_matrix<T, P>(A, xi, eta, sp.dx, sp.dy, (sig + sp.inv_dt) * sp.dx * sp.dy);
    } else {
        // degree-p sigma_t (SweepLinearSolveSpec.cpp:300-321): dx dy / dt on the diagonal, then
        // dx dy / 4 (2d+1)(2e+1) sigma(i,j,d,e,u,v) in row (d,e), column (u,v)
        assemble_matrix<T, P>(A, xi, eta, sp.dx, sp.dy, sp.dx * sp.dy * sp.inv_dt);
        const T quarter = sp.dx * sp.dy / T(4);
#pragma unroll
        for (int uv = 0; uv < N; ++uv)
#pragma unroll
            for (int de = 0; de < N; ++de) {
                const int d = de / P, e = de - P * d;
                A[de + N * uv] += quarter * T((2 * d + 1) * (2 * e + 1)) * tc[uv * N + de];
            }
    }
}

// Most rows of a workgroup of k_sweep_rows: 8 waves, two a SIMD (with more, the SIMDs of the one CU that an ordinate has
// would take longer than a launch per diagonal spread over the chip), 4 at degree 2 for 512 registers a lane; none at
// degree 3, whose 16 x 16 matrix spills either way and where one CU an ordinate loses (40 x 40 S4 FP64: 2.59 against
// 2.12 ms).
template <int P>
constexpr int sweep_rows_most() {
    return P == 4 ? 0 : P == 3 ? 256 : 512;
}

// All diagonals of an ordinate by one workgroup, thread r the cells of row r (counted from the inflow edge): column
// t - r at step t.  The x-neighbour's solution stays in the thread's registers, the y-neighbour's comes from the row
// below through LDS; the source (and for N <= 4 the cross section) of the next step is loaded during this one.  Bound
// by the chain of steps (elimination with its divisions, then a barrier): see launch_sweep_wavefront.
template <typename T, int P>
__global__ __launch_bounds__(sweep_rows_most<P>() ? sweep_rows_most<P>() : 64) void k_sweep_rows(SweepParams<T> sp) {
    constexpr int N = P * P;
    constexpr bool AHEAD = P <= 2;  // the tensor of the next cell fits the registers too
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T *last = reinterpret_cast<T *>(smem_raw);  // [2][N][rows] solutions of the last two steps
    const int R = (int)blockDim.x, r = threadIdx.x, q = blockIdx.x, nx = sp.nx, ny = sp.ny;
    const bool row = r < ny, irev = q >= sp.qo2, jrev = (q >= sp.qo1 && q < sp.qo2) || q >= sp.qo3;
    const T xi = sp.xi[q], eta = sp.eta[q];
    const int xo = xi <= T(0) ? 1 : -1, yo = eta <= T(0) ? 1 : -1;
    const ptrdiff_t stride_j = (ptrdiff_t)sp.nq * N, stride_i = (ny + 2) * stride_j;
    const ptrdiff_t cstep = irev ? -1 : 1;  // one column on
    const int j = row ? (jrev ? ny - r : r + 1) : 1;
    T *const psi0 = sp.psi + (ptrdiff_t)(irev ? nx : 1) * stride_i + j * stride_j + (ptrdiff_t)q * N;  // column 0
    const ptrdiff_t cell0 = (ptrdiff_t)(irev ? nx : 1) * (ny + 2) + j;
    const bool first = r == 0;
    T src[N], halo[N], sig = T(0), tc[AHEAD ? N * N : 1];
    auto load = [&](int c) {  // the cell of column c (clamped into the mesh): its source, row 0's y-inflow, sigma_t
        const int cc = c < 0 ? 0 : (c >= nx ? nx - 1 : c);
        const T *p = psi0 + cc * cstep * stride_i;
#pragma unroll
        for (int k = 0; k < N; ++k) src[k] = p[k];
        if (first) {
#pragma unroll
            for (int k = 0; k < N; ++k) halo[k] = p[yo * stride_j + k];
        }
        const ptrdiff_t cell = cell0 + cc * cstep * (ny + 2);
        if (!sp.xs) {
            sig = sp.sigma[cell];
        } else if constexpr (AHEAD) {
#pragma unroll
            for (int k = 0; k < N * N; ++k) tc[k] = sp.xs[cell * N * N + k];
        }
    };
    T x[N];  // this row's last solution: first the x-inflow
#pragma unroll
    for (int k = 0; k < N; ++k) x[k] = psi0[xo * stride_i + k];
#pragma unroll
    for (int k = 0; k < N; ++k) halo[k] = T(0);
    load(-r);
    const int steps = nx + ny - 1;
    for (int t = 0; t < steps; ++t) {
        const int c = t - r;
        const bool now = row && c >= 0 && c < nx;
        T B[N], up[N], A[N * N];
        // (a wave without a cell on this diagonal only passes the barrier)
        if (__ballot(now) != 0) {
            const T *tcell = sp.xs + (cell0 + (ptrdiff_t)(c < 0 ? 0 : (c >= nx ? nx - 1 : c)) * cstep * (ny + 2)) * N * N;
            cell_matrix<T, P>(A, sp, xi, eta, sig, sp.xs ? (AHEAD ? tc : tcell) : nullptr);
#pragma unroll
            for (int k = 0; k < N; ++k) up[k] = first ? halo[k] : last[(((t + 1) & 1) * N + k) * R + r - 1];
            assemble_rhs<T, P>(B, src, x, up, xi, eta, sp.dx, sp.dy);
            load(c + 1);
            ge_solve<T, N>(A, B);
            if (now) {
                T *self = psi0 + c * cstep * stride_i;
#pragma unroll
                for (int k = 0; k < N; ++k) {
                    self[k] = B[k];
                    x[k] = B[k];
                    last[((t & 1) * N + k) * R + r] = B[k];
                }
            }
        }
        lds_barrier();
    }
}

template <typename T, int P>
__global__ __launch_bounds__(256) void k_sweep_diag(SweepParams<T> sp, int diag, int i_hi, int len) {
    constexpr int N = P * P;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= len * sp.nq) return;
    const int c = t / sp.nq;
    const int q = t - c * sp.nq;
    int i = i_hi - c;
    int j = diag - i + 1;
    if (q >= sp.qo2) i = sp.nx - i + 1;                     // quadrants 2,3: xi < 0
    if ((q >= sp.qo1 && q < sp.qo2) || q >= sp.qo3) j = sp.ny - j + 1;  // quadrants 1,3: eta < 0

    const T xi = sp.xi[q], eta = sp.eta[q];
    const int xo = xi <= T(0) ? 1 : -1;
    const int yo = eta <= T(0) ? 1 : -1;
    const size_t stride_j = (size_t)sp.nq * N;
    const size_t stride_i = (size_t)(sp.ny + 2) * stride_j;
    T *self = sp.psi + (size_t)i * stride_i + (size_t)j * stride_j + (size_t)q * N;
    const T *upx = self + xo * (ptrdiff_t)stride_i;
    const T *upy = self + yo * (ptrdiff_t)stride_j;

    T B[N];
    assemble_rhs<T, P>(B, self, upx, upy, xi, eta, sp.dx, sp.dy);
    T A[N * N];
    const size_t cell = (size_t)i * (sp.ny + 2) + j;
    cell_matrix<T, P>(A, sp, xi, eta, sp.xs ? T(0) : sp.sigma[cell], sp.xs ? sp.xs + cell * N * N : nullptr);
    ge_solve<T, N>(A, B);
#pragma unroll
    for (int k = 0; k < N; ++k) self[k] = B[k];
}

// Most workgroups of k_sweep_rows a CU, by the waves of one: with more, a step waits for the other workgroups of its SIMD
// or they run one after the other, and a launch per diagonal, spread over the chip, is the faster.  One launch against a
// launch per diagonal, us, FP64, at and past the line: Q0 100 x 256 768 ordinates 658 and 849, 1024 930 and 846; Q1 100 x
// 128 737 and 870, 1024 1206 and 1013, 100 x 256 512 1010 and 1270, 640 1731 and 1320, 60 x 512 256 869 and 1640, 320 1960
// and 1880; Q2 100 x 128 512 878 and 1520, with degree-2 cross sections 640 2340 and 2080, 100 x 256 256 1776 and 3040, 320
// 3341 and 3210.  FP32 differs at Q2 with one wave: 100 x 16 512 ordinates 355 and 543, 640 565 and 554.
template <typename T, int P>
constexpr int sweep_rows_per_cu(int waves) {
    if (P == 1) return waves <= 2 ? 4 : 3;
    if (P == 2) return waves == 1 ? 4 : waves == 2 ? 3 : waves <= 4 ? 2 : 1;
    return waves == 1 ? (sizeof(T) == 8 ? 4 : 2) : waves == 2 ? 2 : 1;
}

template <typename T, int P>
static void sweep_wavefront_p(const SweepParams<T> &sp, hipStream_t s) {
    // One workgroup per ordinate while its rows fit one and a CU has few of them, in place of nx + ny - 1 launches of about
    // 3 us each.  Before and after, FP64: Q1 64 x 64 S8 324 -> 171 us, with degree-1 cross sections 450 -> 127, 200 x 200
    // 1.10 -> 0.58 ms, 150 x 500 S4 1.84 -> 0.94; Q2 64 x 64 S8 621 -> 400 us, with degree-2 cross sections 961 -> 493,
    // 200 x 250 2.33 -> 1.49 ms.
    if constexpr (sweep_rows_most<P>() > 0) {
        const int waves = (sp.ny + 63) / 64;
        if (sp.ny <= sweep_rows_most<P>() && sp.nq <= kCus * sweep_rows_per_cu<T, P>(waves)) {
            const int threads = 64 * waves;
            const size_t lds = (size_t)2 * P * P * threads * sizeof(T);  // 36 KB at most
            hipLaunchKernelGGL((k_sweep_rows<T, P>), dim3(sp.nq), dim3(threads), lds, s, sp);
            TSW_HIP(hipGetLastError());
            return;
        }
    }
    const int num_diags = sp.nx + sp.ny - 1;
    for (int diag = 1; diag <= num_diags; ++diag) {
        const int i_hi = diag < sp.nx ? diag : sp.nx;
        const int i_lo = diag - sp.ny + 1 > 1 ? diag - sp.ny + 1 : 1;
        const int len = i_hi - i_lo + 1;
        const int threads = len * sp.nq;
        const int blocks = (threads + 255) / 256;
        hipLaunchKernelGGL((k_sweep_diag<T, P>), dim3(blocks), dim3(256), 0, s, sp, diag, i_hi, len);
    }
    TSW_HIP(hipGetLastError());
}

template <typename T>
void launch_sweep_wavefront(const SweepParams<T> &sp, int p, hipStream_t s) {
    switch (p) {
        case 0: sweep_wavefront_p<T, 1>(sp, s); break;
        case 1: sweep_wavefront_p<T, 2>(sp, s); break;
        case 2: sweep_wavefront_p<T, 3>(sp, s); break;
        case 3: sweep_wavefront_p<T, 4>(sp, s); break;
        default: throw Error(TSW_E_UNSUPPORTED, "DG degree " + std::to_string(p) + " not built (0..3)");
    }
}

template void launch_sweep_wavefront<double>(const SweepParams<double> &, int, hipStream_t);
template void launch_sweep_wavefront<float>(const SweepParams<float> &, int, hipStream_t);

}  // namespace tsw
