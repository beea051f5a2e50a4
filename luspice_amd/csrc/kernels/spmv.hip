// spmv.hip -- SpMV kernels (gfx950).
//
// sell_spmv_kernel: SELL-C-sigma with C = 64.  One wave per slice, one lane
//   per row; slot j of row r of slice s sits at off[s] + j*64 + r, so each
//   step of the row loop is one fully coalesced 64-lane load of values and
//   column ids.  Lanes stop at their own row length, so padding is never
//   read.  Each row is summed sequentially in CSR order, hence with
//   contraction off the fp64 result is bitwise equal to a CPU CSR loop
//   (src/spmv.cu:154-171 of the reference is that loop, one thread per row).
//   Reference layout: src/sellc_spmv.cu:170-257 (C = 32, one warp per slice,
//   y returned in slice order and permuted on the host at
//   bench/test_lu_gpu_f32.cu:196-199); here y is written straight to the
//   original row through perm.  Value type V = double or float (the products of
//   GMRES, sell_block_kernel, also __half),
//   accumulation always fp64 (src/mp/fp16_spmv.cu:50-59 pattern).
//   Batched: tasks are (matrix, slice) pairs over any number of matrices;
//   vectors of matrix m start at voff[m] in the shared arenas.
//
// csr_spmv_kernel: the reference's spmv_launch contract (one thread per row,
//   256-thread blocks, y = A x in CSR order).
#include "common.hpp"
#include "launch.hpp"

namespace lsp {

constexpr int kSpmvBatch = 8;           // slots of a row loaded per round

template <typename V>
__global__ void __launch_bounds__(256)
sell_spmv_kernel(const SellDesc<V> *mats, const int2 *tasks, int ntask,
                 const int64_t *voff, const double *x, double *y)
{
    // the task index is wave-uniform: readfirstlane lets the task and its
    // descriptor come through scalar loads
    const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    if (t >= ntask) return;
    const int2 tk = tasks[t];
    const SellDesc<V> M = mats[tk.x];
    const int lane = lane_id();
    const int k = tk.y * kWave + lane;
    if (k >= M.n) return;
    const int64_t vo = voff[tk.x];
    const double *xm = x + vo;
    const int len = M.rlen[k];
    const int64_t base = M.off[tk.y] + lane;
    const int row = M.perm[k];
    // kSpmvBatch slots per round: every value and column id of the round is
    // loaded, then every x entry, then the products are added in slot order
    // (the same sum as one slot at a time), so a row of up to kSpmvBatch
    // entries costs two dependent memory round trips instead of two per entry
    double s = 0.0;
    for (int j0 = 0; j0 < len; j0 += kSpmvBatch) {
        V v[kSpmvBatch];
        int c[kSpmvBatch];
#pragma unroll
        for (int u = 0; u < kSpmvBatch; u++) {
            const int64_t e = base + (int64_t)min(j0 + u, len - 1) * kWave;
            v[u] = M.val[e];
            c[u] = M.col[e];
        }
        double xv[kSpmvBatch];
#pragma unroll
        for (int u = 0; u < kSpmvBatch; u++) xv[u] = xm[c[u]];
#pragma unroll
        for (int u = 0; u < kSpmvBatch; u++)
            if (j0 + u < len) s += to_f64(v[u]) * xv[u];
    }
    y[vo + row] = s;
}

// The products of a GMRES cycle, one workgroup per four slices of one matrix;
// the sums over its rows that the next kernel needs go along with them, which
// saves a launch and a pass over the vectors each.  The row sums are those of
// sell_spmv_kernel.
template <typename V, int kMode>
__global__ void __launch_bounds__(256) sell_block_kernel(const SellDesc<V> *mats, SellArgs A)
{
    __shared__ double red[4][kSpmvDots];
    if (gated(A.gate)) return;
    if (A.zero_word && blockIdx.x == 0 && threadIdx.x == 0) *A.zero_word = 0;
    const int2 tk = A.blocks[blockIdx.x];
    if (A.mask[tk.x] != A.run) return;
    const SellDesc<V> M = mats[tk.x];
    const int lane = lane_id();
    const int wv = uniform((int)(threadIdx.x >> 6));
    const int sl = tk.y + wv;
    const int64_t vo = A.voff[tk.x];
    const int k = sl * kWave + lane;
    double sum[kSpmvDots] = {0.0, 0.0, 0.0, 0.0};
    if (sl < M.nslices && k < M.n) {
        const double *xm = A.x + vo;
        const int len = M.rlen[k];
        const int64_t base = M.off[sl] + lane;
        const int row = M.perm[k];
        const double bi = kMode == kSellDots ? 0.0 : A.b[vo + row];
        double s = 0.0;
        for (int j0 = 0; j0 < len; j0 += kSpmvBatch) {
            V v[kSpmvBatch];
            int c[kSpmvBatch];
#pragma unroll
            for (int u = 0; u < kSpmvBatch; u++) {
                const int64_t e = base + (int64_t)min(j0 + u, len - 1) * kWave;
                v[u] = M.val[e];
                c[u] = M.col[e];
            }
            double xv[kSpmvBatch];
#pragma unroll
            for (int u = 0; u < kSpmvBatch; u++) xv[u] = kMode == kSellResidual0 ? 0.0 : xm[c[u]];
#pragma unroll
            for (int u = 0; u < kSpmvBatch; u++)
                if (j0 + u < len) s += to_f64(v[u]) * xv[u];    // x = 0: a value that is not finite still shows
        }
        const double out = kMode == kSellDots ? s : bi - s;
        A.y[vo + row] = out;
        if constexpr (kMode == kSellResidual0) A.x[vo + row] = 0.0;
        if constexpr (kMode == kSellDots) {
#pragma unroll
            for (int i = 0; i < kSpmvDots; i++)
                if (i < A.nv) sum[i] = A.V[(long)i * A.ntot + vo + row] * out;
        } else {
            sum[0] = out * out;
            if (A.first) sum[1] = bi * bi;
        }
    }
    const int ns = kMode == kSellDots ? A.nv : 2;
#pragma unroll
    for (int i = 0; i < kSpmvDots; i++)
        if (i < ns) {
            const double t = wave_sum(sum[i]);
            if (lane == 0) red[wv][i] = t;
        }
    __syncthreads();
    const int i = threadIdx.x;
    constexpr int kStride = kMode == kSellDots ? kSpmvDots : 2;
    if (i < ns) A.partial[(long)blockIdx.x * kStride + i] = red[0][i] + red[1][i] + red[2][i] + red[3][i];
}

template <typename V>
hipError_t launch_sell_block(const SellDesc<V> *mats, const SellArgs &A, SellMode mode, hipStream_t st)
{
    if (A.nblocks <= 0) return hipSuccess;
    const dim3 g(A.nblocks), t(256);
    if (mode == kSellDots) {
        hipLaunchKernelGGL((sell_block_kernel<V, kSellDots>), g, t, 0, st, mats, A);
    } else if constexpr (sizeof(V) == 8) {              // residuals are taken with the fp64 values
        if (mode == kSellResidual) hipLaunchKernelGGL((sell_block_kernel<V, kSellResidual>), g, t, 0, st, mats, A);
        else hipLaunchKernelGGL((sell_block_kernel<V, kSellResidual0>), g, t, 0, st, mats, A);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
template hipError_t launch_sell_block<double>(const SellDesc<double> *, const SellArgs &, SellMode, hipStream_t);
template hipError_t launch_sell_block<float>(const SellDesc<float> *, const SellArgs &, SellMode, hipStream_t);
template hipError_t launch_sell_block<__half>(const SellDesc<__half> *, const SellArgs &, SellMode, hipStream_t);

__global__ void __launch_bounds__(256)
csr_spmv_kernel(int n, const int *__restrict__ rowptr, const int *__restrict__ colidx,
                const double *__restrict__ values, const double *__restrict__ x,
                double *__restrict__ y)
{
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row < n) {
        double s = 0.0;
        for (int e = rowptr[row]; e < rowptr[row + 1]; e++) s += values[e] * x[colidx[e]];
        y[row] = s;
    }
}

// CSR with fp32 values: the same loop reading float values, fp64 x and sum
// (the reference's k_csr32, src/mp/mp_spmv_bench.cu:80-88, keeps x and y in
// fp32; here only the stored values are narrowed).
__global__ void __launch_bounds__(256)
csr_spmv_f32_kernel(int n, const int *__restrict__ rowptr, const int *__restrict__ colidx,
                    const float *__restrict__ values, const double *__restrict__ x,
                    double *__restrict__ y)
{
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row < n) {
        double s = 0.0;
        for (int e = rowptr[row]; e < rowptr[row + 1]; e++) s += (double)values[e] * x[colidx[e]];
        y[row] = s;
    }
}

// out[i] = idx[i] >= 0 ? (Vout) in[idx[i]] : 0   (value repack per refactor)
template <typename Vout>
__global__ void gather_cast_kernel(long count, const int *idx, const double *in, Vout *out)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) {
        const int s = idx[i];
        out[i] = from_f64<Vout>(s >= 0 ? in[s] : 0.0);
    }
}

template <typename V>
hipError_t launch_sell_spmv(const SellDesc<V> *mats, const int2 *tasks, int ntask,
                            const int64_t *voff, const double *x, double *y, hipStream_t st)
{
    if (ntask <= 0) return hipSuccess;
    const int blocks = (ntask + 3) / 4;
    hipLaunchKernelGGL(sell_spmv_kernel<V>, dim3(blocks), dim3(256), 0, st, mats, tasks, ntask,
                       voff, x, y);
    return hipGetLastError();
}
template hipError_t launch_sell_spmv<double>(const SellDesc<double> *, const int2 *, int,
                                             const int64_t *, const double *, double *, hipStream_t);
template hipError_t launch_sell_spmv<float>(const SellDesc<float> *, const int2 *, int,
                                            const int64_t *, const double *, double *, hipStream_t);

hipError_t launch_csr_spmv(int n, const int *rowptr, const int *colidx, const double *values,
                           const double *x, double *y, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const int blocks = (n + 255) / 256;
    hipLaunchKernelGGL(csr_spmv_kernel, dim3(blocks), dim3(256), 0, st, n, rowptr, colidx,
                       values, x, y);
    return hipGetLastError();
}

hipError_t launch_csr_spmv_f32(int n, const int *rowptr, const int *colidx, const float *values,
                               const double *x, double *y, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const int blocks = (n + 255) / 256;
    hipLaunchKernelGGL(csr_spmv_f32_kernel, dim3(blocks), dim3(256), 0, st, n, rowptr, colidx,
                       values, x, y);
    return hipGetLastError();
}

template <typename Vout>
hipError_t launch_gather_cast(long count, const int *idx, const double *in, Vout *out,
                              hipStream_t st)
{
    if (count <= 0) return hipSuccess;
    const long blocks = (count + 255) / 256;
    hipLaunchKernelGGL(gather_cast_kernel<Vout>, dim3((unsigned)blocks), dim3(256), 0, st,
                       count, idx, in, out);
    return hipGetLastError();
}
template hipError_t launch_gather_cast<double>(long, const int *, const double *, double *, hipStream_t);
template hipError_t launch_gather_cast<float>(long, const int *, const double *, float *, hipStream_t);
template hipError_t launch_gather_cast<__half>(long, const int *, const double *, __half *, hipStream_t);

}  // namespace lsp
