// gmres.hip -- device-resident GMRES(m) pieces for fp64 GMRES-IR (gfx950).
//
// Reference behaviour: bench/test_lu_gpu_f32.cu:540-715 (right-preconditioned
// restarted GMRES, x0 = 0, Arnoldi with two orthogonalisation passes, Givens
// least squares, inner stop |g_{j+1}|/||b|| <= tol, outer stop on the true
// residual).  The reference runs all of it on the host with two PCIe
// crossings per inner iteration (:595-615); here every vector operation and
// the small Hessenberg/Givens work stay on the device.
//
// Orthogonalisation is classical Gram-Schmidt applied twice (CGS2); two passes
// give the same O(eps) loss of orthogonality as the reference's two-pass
// modified Gram-Schmidt.
//
// What bounds it: launches.  At n <= 1e5 every vector fits the caches and each
// kernel is near the cost of a launch (about 4 us), so the work is laid out for
// few of them.  Reductions are two-stage and deterministic; the second stage
// has no launch of its own while the parts are few (fold()): every workgroup
// that needs a sum adds its matrix's partial sums itself (in the same order, so
// all agree).  One inner iteration
// is the preconditioner's solves and four launches:
//   sell_block_kernel (spmv.hip)  w = A z, partial V^T w
//   orth_kernel<first>            h = V^T w, w -= V h, partial V^T w
//   orth_kernel<second>           h = V^T w, w -= V h, partial w^T w
//   basis_kernel                  V_{j+1} = w / ||w||, Givens step, and the
//                                 solves' work values of the next iteration set
//                                 to the unset marker
// and a cycle adds two (residual with its norm; start_kernel) and one at its
// end (update_kernel: back substitution and x += Z y).  With one launch per
// operation an iteration took thirteen beside the solves.  Whole Newton steps
// (refactor and solve): 200 unknowns 0.65 -> 0.38 ms, 1020 unknowns with fp32
// factors 0.97 -> 0.65 ms, 512 circuits with fp32 factors 7.77 -> 7.42 ms.
//
// Batch layout: vectors of matrix m live at voff[m] .. voff[m]+n_m in arenas
// of length ntot; basis vector i is V + i*ntot.  One workgroup per row chunk
// (matrix, r0, r1).  Matrices whose act[m] == 0 are skipped; a matrix's first
// workgroup (its lead) keeps its Hessenberg, rotations and state, and may clear
// act[m] in a launch whose other workgroups still read it: either value leaves
// a finished matrix's solution alone.
#include "common.hpp"
#include "launch.hpp"

namespace lsp {

constexpr int kKrT = 256;               // threads per workgroup
constexpr int kKrW = kKrT / kWave;

// Sum over the workgroup, in every thread.
__device__ __forceinline__ double block_sum(double v, double *red)
{
    v = wave_sum(v);
    if (lane_id() == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    const double s = red[0] + red[1] + red[2] + red[3];
    __syncthreads();
    return s;
}

// Sum of p[stride * c] over c in [c0, c1), by one wave, in every lane.
__device__ __forceinline__ double wave_partials(const double *p, long stride, int c0, int c1)
{
    double s = 0.0;
    for (int c = c0 + lane_id(); c < c1; c += kWave) s += p[stride * c];
    return wave_sum(s);
}

// Adds up each matrix's parts once, one wave per (matrix, sum), in the order in
// which the consumers would: out[nv * m + i] is sum i of in's parts of matrix m.
__global__ void __launch_bounds__(kWave) fold_kernel(const double *in, const int *pbeg, int pstride, int nv,
                                                     const int *mask, int run, const int *gate, double *out)
{
    if (gated(gate)) return;
    const int m = blockIdx.x / nv, i = blockIdx.x % nv;
    if (mask[m] != run) return;
    const double s = wave_partials(in + i, pstride, pbeg[m], pbeg[m + 1]);
    if (threadIdx.x == 0) out[(long)m * nv + i] = s;
}

// conv, abort word and active counts before a solve.
__global__ void __launch_bounds__(kKrT) solve_init_kernel(int *conv, int nmat, int *abort_word, int *nact)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nmat && conv) conv[i] = 0;
    if (i == 0 && abort_word) *abort_word = 0;
    if (i < kNact) nact[i] = 0;
}

// Sets the solves' work values of one row to the unset marker.
__device__ __forceinline__ void unset_row(const UnsetArgs &U, long i)
{
    const double u = Unset<double>::value();
    U.y[i] = u;
    U.yp[i] = u;
    U.z[i] = u;
    U.zp[i] = u;
}

// Cycle start: ||r|| (and on the first cycle ||b||) from the residual's
// partial sums, the outer convergence test, V_0 = r / ||r||.
__global__ void __launch_bounds__(kKrT) start_kernel(KrylovArgs K, const double *r, int cyc, double *hist,
                                                     const int *gate, UnsetArgs U, const double *pin,
                                                     const int *pbeg)
{
    __shared__ double s2[2];
    if (gated(gate)) return;
    const bool first = cyc == 0;
    const int4 ch = K.chunks[blockIdx.x];
    const int m = ch.x;
    const bool lead = ch.y == 0;
    if (K.conv[m]) {                            // skipped; the lead says so
        if (lead && threadIdx.x == 0) {
            K.act[m] = 0;
            K.cycled[m] = 0;
            if (first) K.jfin[m] = 0;
            if (m == 0) hist[cyc & 1] = K.nb[m] > 0 ? K.beta[m] / K.nb[m] : K.beta[m];   // its last residual
        }
        return;
    }
    const int wv = threadIdx.x >> 6;
    if (wv < 2) {
        const double s = wave_partials(pin + wv, 2, pbeg[m], pbeg[m + 1]);
        if (lane_id() == 0) s2[wv] = s;
    }
    __syncthreads();
    const double beta = sqrt(s2[0]);
    const double nb = first ? sqrt(s2[1]) : K.nb[m];
    const double rel = beta / nb;
    const bool done = rel <= K.outer_tol || !(beta > 0.0);
    if (lead && threadIdx.x == 0) {
        K.beta[m] = beta;
        if (first) K.nb[m] = nb;
        if (m == 0) hist[cyc & 1] = nb > 0 ? rel : beta;
        K.cycled[m] = 0;
        if (first) K.jfin[m] = 0;               // later cycles: basis_kernel's count, once it runs
        K.act[m] = done ? 0 : 1;
        if (done) K.conv[m] = 1;
        else {
            K.g[(long)m * (K.mmax + 1)] = beta;
            atomicAdd(&K.nact[nact_word(cyc, 0)], 1);
        }
    }
    if (done) return;
    const long vo = K.voff[m];
    for (int i = ch.y + threadIdx.x; i < ch.z; i += kKrT) {
        K.V[vo + i] = r[vo + i] / beta;
        unset_row(U, vo + i);
    }
}

// One orthogonalisation pass of column j: h_i = V_i^T w from the partial sums,
// w -= sum h_i V_i over the chunk, and the next partial sums: V_i^T w after the
// first pass, w^T w after the second.  pin holds `pstride` sums per part,
// parts pbeg[m] .. pbeg[m + 1).
constexpr int kOrthTile = 256;          // basis vectors whose coefficients are in LDS at a time
template <bool kFirst>
__global__ void __launch_bounds__(kKrT) orth_kernel(KrylovArgs K, int j, const double *pin, const int *pbeg,
                                                    int pstride)
{
    __shared__ double h[kOrthTile], red[kOrthTile * kKrW];
    const int4 ch = K.chunks[blockIdx.x];
    const int m = ch.x;
    // the next iteration's active count, read by nobody before basis_kernel adds to it
    if (kFirst && blockIdx.x == 0 && threadIdx.x == 0) K.nact[nact_word(0, j + 1)] = 0;
    if (!K.act[m]) return;
    const int nv = j + 1;
    const int wv = threadIdx.x >> 6;
    const int p0 = pbeg[m], p1 = pbeg[m + 1];
    const long vo = K.voff[m];
    double *w = K.w + vo;
    const double *V = K.V + vo;
    double *H = K.H + (long)m * (K.mmax + 1) * K.mmax;
    double *out = K.partial + (long)blockIdx.x * (K.mmax + 1);
    constexpr int kRows = 2;                    // rows per thread and pass (a chunk of 512 in one pass)
    double ww = 0.0;
    for (int r0 = ch.y; r0 < ch.z; r0 += kRows * kKrT) {
        double a[kRows];
        int r[kRows];
#pragma unroll
        for (int t = 0; t < kRows; t++) {
            r[t] = r0 + t * kKrT + (int)threadIdx.x;
            a[t] = r[t] < ch.z ? w[r[t]] : 0.0;
        }
        for (int t0 = 0; t0 < nv; t0 += kOrthTile) {
            const int nt = min(kOrthTile, nv - t0);
            __syncthreads();                    // the tile before has been read
            for (int i = wv; i < nt; i += kKrW) {
                const double s = wave_partials(pin + t0 + i, pstride, p0, p1);
                if (lane_id() == 0) h[i] = s;
            }
            __syncthreads();
            if (ch.y == 0 && r0 == 0)
                for (int i = threadIdx.x; i < nt; i += kKrT) {
                    if (kFirst) H[(long)(t0 + i) * K.mmax + j] = h[i];
                    else H[(long)(t0 + i) * K.mmax + j] += h[i];
                }
            for (int i = 0; i < nt; i++) {
                const double hi = h[i];
#pragma unroll
                for (int t = 0; t < kRows; t++)
                    if (r[t] < ch.z) a[t] -= hi * V[(long)(t0 + i) * K.ntot + r[t]];
            }
        }
#pragma unroll
        for (int t = 0; t < kRows; t++)
            if (r[t] < ch.z) w[r[t]] = a[t];
        if (kFirst) {
            for (int t0 = 0; t0 < nv; t0 += kOrthTile) {
                const int nt = min(kOrthTile, nv - t0);
                __syncthreads();
                for (int i = 0; i < nt; i++) {
                    double s = 0.0;
#pragma unroll
                    for (int t = 0; t < kRows; t++)
                        if (r[t] < ch.z) s += V[(long)(t0 + i) * K.ntot + r[t]] * a[t];
                    s = wave_sum(s);
                    if (lane_id() == 0) red[i * kKrW + wv] = s;
                }
                __syncthreads();
                for (int i = threadIdx.x; i < nt; i += kKrT) {
                    const double s = red[i * kKrW] + red[i * kKrW + 1] + red[i * kKrW + 2] + red[i * kKrW + 3];
                    out[t0 + i] = r0 == ch.y ? s : out[t0 + i] + s;
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < kRows; t++) ww += a[t] * a[t];
        }
    }
    if (!kFirst) {
        ww = block_sum(ww, red);
        if (threadIdx.x == 0) K.pnorm[blockIdx.x] = ww;
    }
}

// V_i^T w for i <= j over one chunk (more basis vectors than the product's
// kernel takes along).
__global__ void __launch_bounds__(kKrT) chunk_dots_kernel(KrylovArgs K, int nv)
{
    __shared__ double red[kKrW];
    const int4 ch = K.chunks[blockIdx.x];
    if (!K.act[ch.x]) return;
    const long vo = K.voff[ch.x];
    for (int i = 0; i < nv; i++) {
        const double *vi = K.V + (long)i * K.ntot + vo;
        double s = 0.0;
        for (int r = ch.y + threadIdx.x; r < ch.z; r += kKrT) s += vi[r] * K.w[vo + r];
        s = block_sum(s, red);
        if (threadIdx.x == 0) K.partial2[(long)blockIdx.x * (K.mmax + 1) + i] = s;
    }
}

// End of inner iteration j: V_{j+1} = w / ||w||, the work values of the next
// solves unset; the lead does the Givens step and ends the matrix's cycle when
// its residual estimate is small enough.
__global__ void __launch_bounds__(kKrT) basis_kernel(KrylovArgs K, int j, UnsetArgs U, const double *pin,
                                                     const int *pbeg)
{
    __shared__ double s_hn;
    const int4 ch = K.chunks[blockIdx.x];
    const int m = ch.x;
    if (!K.act[m]) return;
    if (threadIdx.x < kWave) {
        const double s = wave_partials(pin, 1, pbeg[m], pbeg[m + 1]);
        if (threadIdx.x == 0) s_hn = sqrt(s);
    }
    __syncthreads();
    const double hn = s_hn;
    const long vo = K.voff[m];
    const int mm = K.mmax;
    for (int i = ch.y + threadIdx.x; i < ch.z; i += kKrT) {
        K.V[(long)(j + 1) * K.ntot + vo + i] = K.w[vo + i] / hn;
        unset_row(U, vo + i);
    }
    if (ch.y != 0 || threadIdx.x != 0) return;
    double *H = K.H + (long)m * (mm + 1) * mm;
    double *cs = K.cs + (long)m * mm, *sn = K.sn + (long)m * mm;
    double *g = K.g + (long)m * (mm + 1);
    double a = H[j];                            // column j under the earlier rotations
    for (int i = 0; i < j; i++) {
        const double b = H[(long)(i + 1) * mm + j];
        H[(long)i * mm + j] = cs[i] * a + sn[i] * b;
        a = -sn[i] * a + cs[i] * b;
    }
    const double r = sqrt(a * a + hn * hn);
    const double c = r > 0 ? a / r : 1.0, s = r > 0 ? hn / r : 0.0;
    cs[j] = c;
    sn[j] = s;
    H[(long)j * mm + j] = r;
    const double gj = g[j];
    const double gn = -s * gj;
    g[j + 1] = gn;
    g[j] = c * gj;
    K.jfin[m] = j + 1;
    K.cycled[m] = 1;
    const bool done = fabs(gn) / K.nb[m] <= K.inner_tol || hn < 1e-14 || j + 1 >= mm;
    if (done) K.act[m] = 0;
    else atomicAdd(&K.nact[nact_word(0, j + 1)], 1);
}

// y = R^-1 g of the matrices whose cycle had more steps than a wave has lanes:
// once per matrix, one wave each, ahead of update_kernel.
__global__ void __launch_bounds__(kWave) long_backsolve_kernel(KrylovArgs K, const int *gate)
{
    if (gated(gate)) return;
    const int m = blockIdx.x;
    const int mm = K.mmax, jf = K.jfin[m];
    if (!K.cycled[m] || jf <= kWave) return;
    const double *H = K.H + (long)m * (mm + 1) * mm;
    const double *g = K.g + (long)m * (mm + 1);
    double *y = K.yv + (long)m * mm;
    for (int i = jf - 1; i >= 0; i--) {
        double s = 0.0;
        for (int t = i + 1 + (int)threadIdx.x; t < jf; t += kWave) s += H[(long)i * mm + t] * y[t];
        s = wave_sum(s);
        if (threadIdx.x == 0) y[i] = (g[i] - s) / H[(long)i * mm + i];
        __syncthreads();
    }
}

// End of a cycle: y = R^-1 g over the matrix's steps, x += sum y_i Z_i.
__global__ void __launch_bounds__(kKrT) update_kernel(KrylovArgs K, const double *Z, double *x, const int *gate)
{
    __shared__ double ylds[kWave];
    if (gated(gate)) return;
    const int4 ch = K.chunks[blockIdx.x];
    const int m = ch.x;
    if (!K.cycled[m]) return;
    const int mm = K.mmax, jf = K.jfin[m];
    const double *y = jf <= kWave ? ylds : K.yv + (long)m * mm;
    const double *H = K.H + (long)m * (mm + 1) * mm;
    const double *g = K.g + (long)m * (mm + 1);
    if (jf <= kWave) {
        // lane t holds row t: subtract column i once y_i is known
        if (threadIdx.x < kWave) {
            const int t = threadIdx.x;
            double s = t < jf ? g[t] : 0.0;
            for (int i = jf - 1; i >= 0; i--) {
                const double col = t <= i ? H[(long)t * mm + i] : 0.0;
                const double yi = bcast_f64(s, i) / bcast_f64(col, i);
                if (t == i) ylds[i] = yi;
                if (t < i) s -= col * yi;
            }
        }
    }
    __syncthreads();
    const long vo = K.voff[m];
    for (int r = ch.y + threadIdx.x; r < ch.z; r += kKrT) {
        double acc = 0.0;
        for (int i = 0; i < jf; i++) acc += y[i] * Z[(long)i * K.ntot + vo + r];
        x[vo + r] += acc;
    }
}

__global__ void zero_int_kernel(int *p, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void copy_kernel(const double *src, double *dst, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// ---------------------------------------------------------------------------
static inline int nb_for(long n, int t) { return (int)((n + t - 1) / t); }

hipError_t k_solve_init(int *conv, int nmat, int *abort_word, int *nact, hipStream_t s)
{
    hipLaunchKernelGGL(solve_init_kernel, dim3(nb_for(nmat > kNact ? nmat : kNact, kKrT)), dim3(kKrT), 0, s, conv,
                       nmat, abort_word, nact);
    return hipGetLastError();
}

// The sums a consumer is about to read: the parts as they are, or added up.
struct Parts {
    const double *p;
    const int *beg;
    int stride;
};
// Every workgroup of a consumer adds up all parts of its matrix (`reads` of them
// over the batch, for each of nv sums), which grows with the square of a
// circuit's size.  From kFoldLines cache lines on, a launch of its own adds them
// up first, to the same sums bit for bit.  An iteration beside its solves, as
// they are / added up first: n = 99 906 (196 chunks) 49 / 58 us over 3 iterations,
// 67 / 73 over 20, 146 / 142 over 60; n = 250 000 (489 chunks) 68 / 79 over 3,
// 209 / 180 over 60; chunks of 64 rows, n = 99 906 60 / 69 over 3, 136 / 97 over 20,
// 372 / 183 over 60.  A launch costs 3.3 us, a million lines 1 to 3 us.
constexpr double kFoldLines = 1.5e6;
static Parts fold(const KrylovArgs &K, Parts in, int nv, long reads, const int *mask, int run, const int *gate,
                  hipStream_t s)
{
    if ((double)reads * nv * (in.stride < 8 ? in.stride : 8) / 8 < kFoldLines) return in;
    hipLaunchKernelGGL(fold_kernel, dim3((unsigned)(K.nmat * nv)), dim3(kWave), 0, s, in.p, in.beg, in.stride, nv, mask,
                       run, gate, K.folded);
    return Parts{K.folded, K.each, nv};
}

hipError_t k_start(const KrylovArgs &K, const double *r, int cyc, double *hist, const int *gate,
                   const UnsetArgs &U, hipStream_t s)
{
    const Parts in = fold(K, Parts{K.spartial, K.sbeg, 2}, 2, K.sreads, K.conv, 0, gate, s);
    hipLaunchKernelGGL(start_kernel, dim3(K.nchunks), dim3(kKrT), 0, s, K, r, cyc, hist, gate, U, in.p, in.beg);
    return hipGetLastError();
}
hipError_t k_chunk_dots(const KrylovArgs &K, int nv, hipStream_t s)
{
    hipLaunchKernelGGL(chunk_dots_kernel, dim3(K.nchunks), dim3(kKrT), 0, s, K, nv);
    return hipGetLastError();
}
hipError_t k_orth(const KrylovArgs &K, int j, bool first, hipStream_t s)
{
    const bool prod = first && j < kSpmvDots;   // sums from the product's kernel
    Parts in = prod ? Parts{K.spartial, K.sbeg, kSpmvDots} : Parts{first ? K.partial2 : K.partial, K.cbeg, K.mmax + 1};
    in = fold(K, in, j + 1, prod ? K.sreads : K.creads, K.act, 1, nullptr, s);
    const dim3 g(K.nchunks), t(kKrT);
    if (first) hipLaunchKernelGGL(orth_kernel<true>, g, t, 0, s, K, j, in.p, in.beg, in.stride);
    else hipLaunchKernelGGL(orth_kernel<false>, g, t, 0, s, K, j, in.p, in.beg, in.stride);
    return hipGetLastError();
}
hipError_t k_basis(const KrylovArgs &K, int j, const UnsetArgs &U, hipStream_t s)
{
    const Parts in = fold(K, Parts{K.pnorm, K.cbeg, 1}, 1, K.creads, K.act, 1, nullptr, s);
    hipLaunchKernelGGL(basis_kernel, dim3(K.nchunks), dim3(kKrT), 0, s, K, j, U, in.p, in.beg);
    return hipGetLastError();
}
hipError_t k_update(const KrylovArgs &K, const double *Z, double *x, int steps, const int *gate, hipStream_t s)
{
    // (every workgroup repeating 150 steps' back substitution cost 3 ms on 1561 chunks)
    if (steps > kWave) hipLaunchKernelGGL(long_backsolve_kernel, dim3(K.nmat), dim3(kWave), 0, s, K, gate);
    hipLaunchKernelGGL(update_kernel, dim3(K.nchunks), dim3(kKrT), 0, s, K, Z, x, gate);
    return hipGetLastError();
}
hipError_t k_zero_int(int *p, long n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(zero_int_kernel, dim3(nb_for(n, 256)), dim3(256), 0, s, p, n);
    return hipGetLastError();
}
hipError_t k_copy(const double *src, double *dst, long n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(copy_kernel, dim3(nb_for(n, 256)), dim3(256), 0, s, src, dst, n);
    return hipGetLastError();
}

}  // namespace lsp
