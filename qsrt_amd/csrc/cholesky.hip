// Diagonal-block step of a blocked float64 Cholesky factorisation.
//
// block_ldl (reference qsrt/exl3_encoder_backend.py:323-393) factors the damped
// Hessian H = C C^T before forming L = C blockdiag(C_ii)^-1; here that
// factorisation runs in float64.  A right-looking blocked Cholesky spends its
// flops in the trailing updates A22 -= L21 L21^T, which are plain DGEMMs on
// the matrix cores; what a library factorisation of one matrix loses time on
// is the chain of small diagonal-block factorisations between them.  This
// kernel does one diagonal block in a single workgroup (registers and LDS), and
// also returns the block's inverse so that the panel solve
// L21 = A21 L11^-T becomes one more DGEMM.
//
// Block of nb <= 128 rows, 16 waves.  In the factorisation wave w keeps columns 8 w .. 8 w + 7 of the block in
// registers, a lane two rows (l and l + 64); in the inverse X = L11^-1 it keeps rows 8 w .. 8 w + 7, a lane two
// columns.  A panel of eight columns then belongs to one wave, and so do eight rows of X:
//   factor    step k: the pivot a_kk is read from its lane, d = sqrt(a_kk), l_ik = a_ik * (1 / d) (the reciprocal
//             multiply of LAPACK's dpotf2) and a_ij -= l_ik l_jk (fma) for the panel's later columns, l_jk read from
//             lane j: no barrier inside a panel.  The panel goes to LDS.
//   update    every later wave: a_ij -= l_ik l_jk for the panel's eight k, ascending.
//   solve     the panel's wave, one panel later: its rows of X, x_kc / l_kk and x_ic -= l_ik x_kc, no barrier either.
// One round p is [wave p factors, wave p - 1 solves], barrier, [later waves update from both]: one barrier per eight
// columns, the solve in the shadow of the factor, and each element meets its fmas in the order k = 0, 1, ... of the
// plain right-looking algorithm.
//
// What bounds it is the chain of pivots, 128 square roots and reciprocals one after the other: 560 cycles a column,
// so 4500 of the 6600 (late) to 8400 (early) cycles of a round, the rest being the update that the next panel's wave
// has to finish first, among the LDS reads of the others.  That wave therefore runs at raised priority and leaves its
// rows of X for the round after (66 us without, 60 us with).  With one barrier per column, all 16 waves in each, and
// each evaluating the root, a block of 128 rows took 237 us between two events, of 64 rows 128 us and of 16 rows
// 40 us; it takes 60, 37 and 19 us, with the same bits.  One workgroup per matrix of a batch.

#include "common.h"
#include "qsrt_amd.h"

namespace {

constexpr int kMaxNb = 128;
constexpr int kPanel = 8;                           // columns of a panel, rows of X of a wave
constexpr int kPanels = kMaxNb / kPanel;            // 16
constexpr int kThreadsChol = 64 * kPanels;          // a wave per panel
constexpr int kLdL = kMaxNb + 2;                    // doubles per column of L in LDS: 16-byte aligned, and the final
                                                    // transposed read meets a bank 4 times instead of 64

struct CholShared {
    double L[kMaxNb * kLdL];         // column-major: l_ik at k * kLdL + i
    double X[2][kPanel * kMaxNb];    // eight rows of X, two panels in turn
    int failed[kPanels];             // 1 + the step whose pivot is not positive, per panel
};

__device__ __forceinline__ double lane_value(double v, int lane) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}

// Factors panel p from its wave's registers; R is the register row that holds rows 8 p .. (rows l for p < 8, l + 64
// from there on, where the rows l lie above the panel and are left out).
template <int R>
__device__ __forceinline__ void factor_panel(double (&a)[2][kPanel], int p, int nb, CholShared& sh) {
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int k0 = kPanel * p, lane0 = k0 & 63;
#pragma unroll
    for (int c = 0; c < kPanel; ++c) {
        const int k = k0 + c;
        if (k >= nb) break;
        const double piv = lane_value(a[R][c], lane0 + c);
        if (!(piv > 0.0)) {
            if (lane == 0) sh.failed[p] = k + 1;
            return;
        }
        const double d = sqrt(piv), rd = 1.0 / d;
#pragma unroll
        for (int r = R; r < 2; ++r) a[r][c] *= rd;
#pragma unroll
        for (int j = c + 1; j < kPanel; ++j) {
            const double lj = lane_value(a[R][c], lane0 + j);
#pragma unroll
            for (int r = R; r < 2; ++r) a[r][j] = fma(-a[r][c], lj, a[r][j]);
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int i = lane + 64 * r;
            sh.L[k * kLdL + i] = i > k ? a[r][c] : i == k ? d : 0.0;
        }
    }
}

// The nb x nb diagonal block at (j0, j0) of matrix blockIdx.x (leading dimension n, batch stride
// `stride`): its lower triangle is read, the factor L11 is written over it with zeros above the
// diagonal, and L11^-1 goes to inv (nb x nb row-major per matrix, zeros above the diagonal).  A pivot
// k that is not positive (or NaN) stops the factorisation; info[b] then receives j0 + k + 1 unless it
// already holds an earlier failure, and the block and its inverse are left undefined.
__global__ __launch_bounds__(kThreadsChol) void chol_diag_block_f64_kernel(double* __restrict__ A, int64_t n,
                                                                           int64_t stride, int64_t j0, int nb,
                                                                           double* __restrict__ inv,
                                                                           int32_t* __restrict__ info) {
    __shared__ __attribute__((aligned(16))) CholShared sh;
    const int t = static_cast<int>(threadIdx.x);
    const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int panels = (nb + kPanel - 1) / kPanel;
    double* M = A + static_cast<int64_t>(blockIdx.x) * stride + j0 * n + j0;
    double* Xo = inv + static_cast<int64_t>(blockIdx.x) * nb * nb;

    // Row-major lines in, columns out: through LDS, as the other way a load would touch 64 lines.
    double in[kMaxNb * kMaxNb / kThreadsChol];
#pragma unroll
    for (int e = 0; e < kMaxNb * kMaxNb / kThreadsChol; ++e) {
        const int i = w + kPanels * (e >> 1), j = lane + 64 * (e & 1);
        in[e] = i < nb && j <= i ? M[static_cast<int64_t>(i) * n + j] : 0.0;
    }
#pragma unroll
    for (int e = 0; e < kMaxNb * kMaxNb / kThreadsChol; ++e)
        sh.L[(lane + 64 * (e & 1)) * kLdL + w + kPanels * (e >> 1)] = in[e];
    if (t < kPanels) sh.failed[t] = 0;
    __syncthreads();
    double a[2][kPanel], x[kPanel][2];
#pragma unroll
    for (int c = 0; c < kPanel; ++c)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            a[r][c] = sh.L[(kPanel * w + c) * kLdL + lane + 64 * r];
            x[c][r] = kPanel * w + c == lane + 64 * r ? 1.0 : 0.0;
        }

    // Nothing is overwritten early: a wave writes only columns of L that it alone has read before, and the rows of X
    // of panel p (written in round p + 1) make room for those of panel p + 2 in round p + 3, after the barrier of round
    // p + 2, which their readers reach last, or by the one wave that is later than that, p + 2 itself.
    for (int p = 0; p <= panels; ++p) {
        int own = w;  // the compiler knows p == w inside and would keep every predicate of the panel over the loop
        asm volatile("" : "+s"(own));
        if (w == p && p < panels) {
            if (p < kPanels / 2)
                factor_panel<0>(a, own, nb, sh);
            else
                factor_panel<1>(a, own, nb, sh);
        }
        if (w == p - 1) {  // rows 8 w ..: their columns of L are this wave's own, written in the round before
            const int k0 = kPanel * own;
            double* row = sh.X[own & 1];
#pragma unroll
            for (int c = 0; c < kPanel; ++c) {
                if (k0 + c >= nb) break;
                const double lkk = sh.L[(k0 + c) * kLdL + k0 + c];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    x[c][q] = x[c][q] / lkk;
                    row[c * kMaxNb + lane + 64 * q] = x[c][q];
                }
#pragma unroll
                for (int i = c + 1; i < kPanel; ++i) {
                    const double li = sh.L[(k0 + c) * kLdL + k0 + i];
#pragma unroll
                    for (int q = 0; q < 2; ++q) x[i][q] = fma(-li, x[c][q], x[i][q]);
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();
        if (p < panels) {
            if (const int failed = sh.failed[p]) {  // the same word for every thread: uniform
                if (t == 0) atomicCAS(info + blockIdx.x, 0, static_cast<int32_t>(j0 + failed));
                return;
            }
            if (w == p + 1) __builtin_amdgcn_s_setprio(3);  // the chain goes through this wave
            if (w > p) {
#pragma unroll 2
                for (int k = 0; k < kPanel; ++k) {
                    const double* l = sh.L + (kPanel * p + k) * kLdL;
                    double lj[kPanel];
#pragma unroll
                    for (int c = 0; c < kPanel; ++c) lj[c] = l[kPanel * w + c];
                    if (w < kPanels / 2) {  // rows l reach below the diagonal of these columns
                        const double li = l[lane];
#pragma unroll
                        for (int c = 0; c < kPanel; ++c) a[0][c] = fma(-li, lj[c], a[0][c]);
                    }
                    const double li = l[lane + 64];
#pragma unroll
                    for (int c = 0; c < kPanel; ++c) a[1][c] = fma(-li, lj[c], a[1][c]);
                }
            }
        }
        // Rows of X of the panels before p; the wave that factors next has its factor to get on with and takes the
        // last two together a round later (rows p - 2 are overwritten by its own solve at the earliest).
        const int first = w == p + 1 ? p : w == p && p > 1 ? p - 2 : p - 1;
        for (int s = first < 0 ? 0 : first; s < p && w >= p; ++s) {
            const double* row = sh.X[s & 1];
#pragma unroll 2
            for (int k = 0; k < kPanel; ++k) {
                const double* l = sh.L + (kPanel * s + k) * kLdL + kPanel * w;
                const double x0 = row[k * kMaxNb + lane], x1 = row[k * kMaxNb + lane + 64];
#pragma unroll
                for (int i = 0; i < kPanel; ++i) {
                    const double li = l[i];
                    x[i][0] = fma(-li, x0, x[i][0]);
                    x[i][1] = fma(-li, x1, x[i][1]);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < kPanel; ++c)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int i = kPanel * w + c, j = lane + 64 * q;
            if (i < nb && j < nb) Xo[i * nb + j] = j <= i ? x[c][q] : 0.0;
        }
#pragma unroll
    for (int e = 0; e < kMaxNb * kMaxNb / kThreadsChol; ++e) {
        const int i = w + kPanels * (e >> 1), j = lane + 64 * (e & 1);
        if (i < nb && j < nb) M[static_cast<int64_t>(i) * n + j] = sh.L[j * kLdL + i];
    }
}

}  // namespace

// Unit block-lower factor from a lower Cholesky factor, in place: row i of column block j (i past the block's
// diagonal) becomes C[i, 16 j : 16 j + 16] inv_j, the diagonal 16 x 16 blocks become the identity, and the zero
// blocks above the diagonal are not touched.  One workgroup per (row chunk, column block, matrix); inv_j is
// staged in LDS and each thread owns one row: sixteen doubles read, sixteen 16-term products, sixteen written.
// Element (i, c) sits at i * ld + c (row-major, 16-byte loads along the row) or at c * ld + i (column-major, the
// layout torch's batched Cholesky returns: a wave's 64 rows are then 512 contiguous bytes per column).
constexpr int kUnitRows = 256;

template <bool kRowMajor>
__global__ __launch_bounds__(kUnitRows) void block_unit_lower_f64_kernel(double* __restrict__ C,
                                                                         const double* __restrict__ inv, int64_t n,
                                                                         int64_t ld, int64_t batch_stride) {
    const int64_t j = blockIdx.y, mat = blockIdx.z;
    const int64_t col0 = 16 * j;
    const int64_t row0 = col0 + static_cast<int64_t>(blockIdx.x) * kUnitRows;
    if (row0 >= n) return;  // the whole workgroup is past the last row
    __shared__ double iv[16][17];
    const double* ij = inv + (mat * (n / 16) + j) * 256;
    for (int e = threadIdx.x; e < 256; e += kUnitRows) iv[e >> 4][e & 15] = ij[e];
    __syncthreads();
    const int64_t row = row0 + threadIdx.x;
    if (row >= n) return;
    double* base = C + mat * batch_stride;
    const int64_t rs = kRowMajor ? ld : 1, cs = kRowMajor ? 1 : ld;
    double* r = base + row * rs + col0 * cs;
    if (row < col0 + 16) {  // the diagonal block
#pragma unroll
        for (int l = 0; l < 16; ++l) r[l * cs] = (row - col0 == l) ? 1.0 : 0.0;
        return;
    }
    double x[16];
    if constexpr (kRowMajor) {
#pragma unroll
        for (int k = 0; k < 16; k += 2) {
            const double2 v = *reinterpret_cast<const double2*>(r + k);
            x[k] = v.x;
            x[k + 1] = v.y;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) x[k] = r[k * cs];
    }
#pragma unroll
    for (int l = 0; l < 16; l += 2) {
        double a0 = 0.0, a1 = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            a0 = __builtin_fma(x[k], iv[k][l], a0);
            a1 = __builtin_fma(x[k], iv[k][l + 1], a1);
        }
        if constexpr (kRowMajor) {
            *reinterpret_cast<double2*>(r + l) = make_double2(a0, a1);
        } else {
            r[l * cs] = a0;
            r[(l + 1) * cs] = a1;
        }
    }
}

extern "C" {

int qsrt_block_unit_lower_f64(double* C, const double* inv, int64_t batch, int64_t n, int64_t row_stride,
                              int64_t col_stride, int64_t batch_stride, void* stream_handle) {
    hipStream_t stream = static_cast<hipStream_t>(stream_handle);
    if (!C || !inv) return qsrt::fail(qsrt::kBadArgument, "null pointer argument");
    if (n <= 0 || batch <= 0) return qsrt::fail(qsrt::kBadArgument, "n and batch must be positive");
    if (n % 16) return qsrt::fail(qsrt::kBadArgument, "n must be a multiple of 16");
    const bool row_major = col_stride == 1;
    if (!row_major && row_stride != 1)
        return qsrt::fail(qsrt::kBadArgument, "one of row_stride and col_stride must be 1");
    const int64_t ld = row_major ? row_stride : col_stride;
    if (ld < n) return qsrt::fail(qsrt::kBadArgument, "the leading dimension must be at least n");
    if (row_major && (ld % 2 || reinterpret_cast<uintptr_t>(C) % 16 || (batch > 1 && batch_stride % 2)))
        return qsrt::fail(qsrt::kBadArgument, "row-major matrices need 16-byte aligned rows");
    if (batch > 1 && batch_stride < (n - 1) * ld + n)
        return qsrt::fail(qsrt::kBadArgument, "the batch stride must keep the matrices apart");
    if (batch > 65535 || n / 16 > 65535) return qsrt::fail(qsrt::kBadArgument, "batch or n too large for one launch");
    const dim3 grid(static_cast<unsigned>((n + kUnitRows - 1) / kUnitRows), static_cast<unsigned>(n / 16),
                    static_cast<unsigned>(batch));
    const int64_t bs = batch > 1 ? batch_stride : 0;
    if (row_major)
        hipLaunchKernelGGL(block_unit_lower_f64_kernel<true>, grid, dim3(kUnitRows), 0, stream, C, inv, n, ld, bs);
    else
        hipLaunchKernelGGL(block_unit_lower_f64_kernel<false>, grid, dim3(kUnitRows), 0, stream, C, inv, n, ld, bs);
    QSRT_HIP_TRY(hipGetLastError());
    return qsrt::kOk;
}

int qsrt_chol_diag_block_f64(double* A, int64_t n, int64_t batch, int64_t batch_stride, int64_t j0, int nb,
                             double* inv, int32_t* info, void* stream_handle) {
    hipStream_t stream = static_cast<hipStream_t>(stream_handle);
    if (!A || !inv || !info) return qsrt::fail(qsrt::kBadArgument, "null pointer argument");
    if (n <= 0 || batch <= 0) return qsrt::fail(qsrt::kBadArgument, "n and batch must be positive");
    if (nb < 1 || nb > kMaxNb) return qsrt::fail(qsrt::kBadArgument, "nb must be in 1..%d", kMaxNb);
    if (j0 < 0 || j0 + nb > n) return qsrt::fail(qsrt::kBadArgument, "block [j0, j0 + nb) outside the matrix");
    if (batch > 1 && batch_stride < n * n) return qsrt::fail(qsrt::kBadArgument, "batch stride below n * n");
    if (batch > 0x7fffffff) return qsrt::fail(qsrt::kBadArgument, "batch too large for one launch");
    hipLaunchKernelGGL(chol_diag_block_f64_kernel, dim3(static_cast<unsigned>(batch)), dim3(kThreadsChol), 0, stream,
                       A, n, batch_stride, j0, nb, inv, info);
    QSRT_HIP_TRY(hipGetLastError());
    return qsrt::kOk;
}

}  // extern "C"
