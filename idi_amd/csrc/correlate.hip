// Correlators of photon images (reference: idi/reconstruction/cusimple.py:44-121
// and cucor.py:9-133).
//
// k_corr_accumulate: one streaming step of correlator2d.add (cusimple.py:80-107):
//   c = corr / maskcorr where maskcorr > 0.5, else 0;
//   count == 1: mean = c, m2 = 0;  else: d = c - mean; mean += d / count; m2 += d (c - mean)
// (Welford's running mean and sum of squared deviations), fused into one pass, in
// float32 with the reference's operation order and no contraction.
//
// k_qcorr_runs: q-corrected autocorrelation (cucor.py:54-91).  For a detector z pixels
// away, pixel (r, c) has zd = z / |(r - xc, c - yc, z)|; the pair (ref, target) with
// row offset 0 <= dr < qmax and column offset |dc| < qmax is binned at
//   dqx = round((tr - xc) zd_t - (rr - xc) zd_r),  dqy = round((tc - yc) zd_t - (rc - yc) zd_r),
//   dqz = round(z (zd_r - zd_t))
// (float32 arithmetic, no contraction, round half to even) and adds img_r img_t.
// Sums are FP64 atomics (the reference accumulates float32); bins outside the
// output are skipped (the reference does not check them).
// k_qcorr_assemble (cucor.py:93-96): out[i] and out[mirror(i)], mirror(i) = (-i) mod
// shape, both become their sum for every bin with dqx index < qmax (a bin that is
// its own mirror is doubled).  In the reference two threads update each pair of
// the dqx index 0 column at once; here that pair also gets the plain sum.
#include <algorithm>
#include <climits>

#include "device_util.hpp"

namespace idisim {

__global__ __launch_bounds__(256) void k_corr_accumulate(const float* __restrict__ corr,
                                                         const float* __restrict__ maskcorr, int64_t n,
                                                         int64_t count, float* __restrict__ mean,
                                                         float* __restrict__ m2)
{
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float mc = maskcorr[i];
    const float c = (mc > 0.5f) ? corr[i] / mc : 0.f;
    if (count <= 1) {
        mean[i] = c;
        m2[i] = 0.f;
    } else {
        const float m = mean[i];
        const float d = c - m;
        const float mn = m + d / (float)count;
        mean[i] = mn;
        m2[i] += d * (c - mn);
    }
}

__global__ __launch_bounds__(256) void k_fill_f64(double* __restrict__ p, int64_t n, double v)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// A lane keeps one column offset and walks along the reference columns: zd varies slowly along a row, so
// the bin stays the same for tens of pairs (51 on average at 256^2, z = 2000, offsets below 64).  It
// sums such a run in a register (the product of two floats is exact in FP64) and adds it to the bin when
// the bin changes; a closed run waits up to kQSteps pairs, so that the lanes of a wave add together.
// A workgroup takes one row offset, 64 column offsets, `rows` reference rows (one per wave at a time)
// and kQCols reference columns; its bins' range is read off the corners of that block and kept in LDS as
// far as it fits, any other bin is added to in global memory, so the sums do not depend on that range.
//
// Bound by latency and the vector instructions of the bins (three differences, roundings and compares a
// pair), no longer by the atomics: one LDS atomic a pair with a window per (row, row offset) ->
// this: 1623 -> 421 us at 256^2 (z 2000, offsets < 64, 4e8 pairs); where that window did not fit and every
// pair was a global atomic 131 -> 2.4 ms at 400^2 (z 1000, offsets < 96); 54 -> 36 us at 100^2.  Staging zd
// and y zd (12 bytes with the value) instead of 16 and 2048 bins of 3072 leave 6 workgroups a CU: 527 ->
// 421; reading a step ahead was slower (579).
constexpr float kQNone = -1e9f;        // no bin
constexpr int kQSteps = 8;
constexpr int kQCols = 64;             // reference columns of a workgroup
constexpr int kQSpan = kQCols + 63;    // and target columns
constexpr int kQBins = 2048;           // bins of its window, at most kQX and kQY of them along x and y
constexpr int kQX = 16, kQY = 96;
constexpr int kQFar = 1 << 20;         // beyond any bin

__global__ __launch_bounds__(256) void k_qcorr_runs(const float* __restrict__ zd, const float* __restrict__ img,
                                                    int nr, int nc, float xc, float yc, float cz, int qmax,
                                                    int maxdqz, int rows, double* __restrict__ out)
{
#pragma clang fp contract(off)
    __shared__ double hist[kQBins];
    __shared__ float2 s_ref[4][kQCols], s_tgt[4][kQSpan];  // (momentum y, zd) of a column
    __shared__ float s_rv[4][kQCols], s_tv[4][kQSpan];      // its value
    __shared__ int s_ext[6];
    const int chunk = blockIdx.z, offr = (int)blockIdx.x % qmax;
    const int g0 = (int)blockIdx.x / qmax * 64 - (qmax - 1);  // column offsets g0 .. g0 + 63
    const int r0 = (int)blockIdx.y * rows, r1 = min(r0 + rows, nr - offr);
    // reference columns with a target in the image for some lane
    const int c0 = max(chunk * kQCols, -(g0 + 63)), c1 = min(min((chunk + 1) * kQCols, nc), nc - g0);
    if (r0 >= r1 || c0 >= c1) return;  // whole workgroup: uniform
    const int sz = 2 * maxdqz, sq = 2 * qmax;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x < 3) {
        s_ext[threadIdx.x] = INT_MAX;
        s_ext[3 + threadIdx.x] = INT_MIN;
    }
    for (int b = threadIdx.x; b < kQBins; b += blockDim.x) hist[b] = 0.0;
    __syncthreads();
    if (threadIdx.x < 8) {
        // the bins of the pairs at the corners of the rows, columns and offsets
        const int refr = (threadIdx.x & 1) ? r1 - 1 : r0, tr = refr + offr;
        const int oc = max(min((threadIdx.x & 2) ? min(g0 + 63, qmax - 1) : g0, nc - 1), 1 - nc);
        const int rc = min(max((threadIdx.x & 4) ? c1 - 1 : c0, max(0, -oc)), min(nc, nc - oc) - 1), tc = rc + oc;
        const float rz = zd[(size_t)refr * nc + rc], tz = zd[(size_t)tr * nc + tc];
        const int q[3] = {(int)rintf(((float)tr - xc) * tz - ((float)refr - xc) * rz),
                          (int)rintf(((float)tc - yc) * tz - ((float)rc - yc) * rz), (int)rintf(cz * (rz - tz))};
        for (int d = 0; d < 3; ++d) {
            const int v = min(max(q[d], -kQFar), kQFar);
            atomicMin(&s_ext[d], v - 1);
            atomicMax(&s_ext[3 + d], v + 1);
        }
    }
    __syncthreads();
    // the window: all of x and y, as much of z as fits
    const int lox = s_ext[0], loy = s_ext[1], loz0 = s_ext[2];
    const int wx = min(s_ext[3] - lox + 1, kQX), wy = min(s_ext[4] - loy + 1, kQY);
    const int nz = s_ext[5] - loz0 + 1, wz = min(nz, kQBins / (wx * wy)), loz = loz0 + (nz - wz) / 2;

    for (int refr = r0 + w; refr < r1; refr += 4) {
        const int tr = refr + offr;
        const float tr2 = (float)tr - xc, rr2 = (float)refr - xc;
        for (int i = lane; i < c1 - c0; i += 64) {
            const int c = c0 + i;
            const float z = zd[(size_t)refr * nc + c];
            s_ref[w][i] = make_float2(((float)c - yc) * z, z);
            s_rv[w][i] = img[(size_t)refr * nc + c];
        }
        for (int i = lane; i < c1 - c0 + 63; i += 64) {
            const int c = c0 + g0 + i;
            if (c < 0 || c >= nc) continue;
            const float z = zd[(size_t)tr * nc + c];
            s_tgt[w][i] = make_float2(((float)c - yc) * z, z);
            s_tv[w][i] = img[(size_t)tr * nc + c];
        }
        wave_sync();
        float px = kQNone, py = 0.f, pz = 0.f, qx = kQNone, qy = 0.f, qz = 0.f;  // the open run's bin, the closed one's
        double acc = 0.0, closed = 0.0;
        auto add = [&]() {
            const int x = (int)qx, y = (int)qy, z = (int)qz;
            qx = kQNone;
            const unsigned ux = (unsigned)x - lox, uy = (unsigned)y - loy, uz = (unsigned)z - loz;
            if (ux < (unsigned)wx && uy < (unsigned)wy && uz < (unsigned)wz) {
                atomicAdd(&hist[(uz * wy + uy) * wx + ux], closed);
                return;
            }
            const unsigned dqx = (unsigned)qmax + x, dqy = (unsigned)qmax + y, dqz = (unsigned)maxdqz + z;
            if (dqx >= (unsigned)sq || dqy >= (unsigned)sq || dqz >= (unsigned)sz) return;
            unsafeAtomicAdd(out + ((size_t)dqz * sq + dqy) * sq + dqx, closed);
        };
        // the lane's columns: inside the image, and offsets below qmax
        const int tc0 = c0 + g0 + lane, i0 = max(0, -tc0);
        const unsigned ni = g0 + lane < qmax ? max(min(c1 - c0, nc - tc0) - i0, 0) : 0;
        for (int i = 0; i < c1 - c0; i += kQSteps) {
#pragma unroll 1
            for (int j = i; j < i + kQSteps; ++j) {
                if ((unsigned)(j - i0) >= ni) continue;
                const float2 r = s_ref[w][j], t = s_tgt[w][j + lane];
                const float x = rintf(tr2 * t.y - rr2 * r.y), y = rintf(t.x - r.x), z = rintf(cz * (r.y - t.y));
                const bool next = x != px || y != py || z != pz;
                if (next && qx != kQNone) add();
                qx = next ? px : qx;
                qy = next ? py : qy;
                qz = next ? pz : qz;
                closed = next ? acc : closed;
                acc = next ? 0.0 : acc;
                px = x;
                py = y;
                pz = z;
                acc = fma((double)s_rv[w][j], (double)s_tv[w][j + lane], acc);  // the product is exact
            }
            if (qx != kQNone) add();
        }
        qx = px;
        qy = py;
        qz = pz;
        closed = acc;
        if (qx != kQNone) add();
        wave_sync();
    }
    __syncthreads();
    for (int b = threadIdx.x; b < wx * wy * wz; b += blockDim.x) {
        const double v = hist[b];
        if (v != 0.0) {
            const int dqx = qmax + lox + b % wx, dqy = qmax + loy + b / wx % wy, dqz = maxdqz + loz + b / (wx * wy);
            if (dqx < 0 || dqx >= sq || dqy < 0 || dqy >= sq || dqz < 0 || dqz >= sz) continue;
            unsafeAtomicAdd(out + ((size_t)dqz * sq + dqy) * sq + dqx, v);
        }
    }
}

// One thread per bin with dqx index < qmax; the mirror has dqx index (sq - i2) mod sq,
// which is >= qmax except for i2 == 0 (its own column): there only the lower of the
// two flat indices writes, so every pair is updated exactly once.
__global__ __launch_bounds__(256) void k_qcorr_assemble(double* __restrict__ out, int maxdqz, int qmax)
{
    const int sz = 2 * maxdqz, sq = 2 * qmax;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nh = (int64_t)sz * sq * qmax;
    if (idx >= nh) return;
    const int i2 = (int)(idx % qmax);
    const int64_t r = idx / qmax;
    const int i1 = (int)(r % sq), i0 = (int)(r / sq);
    const int m0 = (sz - i0) % sz, m1 = (sq - i1) % sq, m2 = (sq - i2) % sq;
    const size_t a = ((size_t)i0 * sq + i1) * sq + i2;
    const size_t b = ((size_t)m0 * sq + m1) * sq + m2;
    if (a == b) {  // its own mirror (dqx index 0 only): added to itself, as in the reference
        out[a] = out[a] + out[a];
        return;
    }
    if (i2 == 0 && b < a) return;  // the pair is handled by its other member
    const double s = out[a] + out[b];
    out[a] = s;
    out[b] = s;
}

hipError_t launch_corr_accumulate(const float* corr, const float* maskcorr, int64_t n, int64_t count, float* mean,
                                  float* m2, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_corr_accumulate, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, corr, maskcorr, n,
                       count, mean, m2);
    return hipGetLastError();
}

hipError_t launch_qcorr(const float* zd, const float* img, int nr, int nc, float xc, float yc, float cz, int qmax,
                        int maxdqz, double* out, hipStream_t st)
{
    const int64_t nout = (int64_t)(2 * maxdqz) * (2 * qmax) * (2 * qmax);
    hipLaunchKernelGGL(k_fill_f64, dim3((unsigned)((nout + 255) / 256)), dim3(256), 0, st, out, nout, 0.0);
    // Rows of a workgroup: the most (fewer windows to add to global memory) that leave more than 16
    // workgroups a CU.  us with 4, 8, 16, 32 rows: 36, 37, 68, 123 at 100^2 (offsets < 32), 492, 438, 419,
    // 427 at 256^2 (64), 10120, 8781, 8108, 7790 at 600^2 (128).
    const unsigned chunks = (unsigned)((nc + kQCols - 1) / kQCols), groups = (unsigned)((2 * qmax + 62) / 64);
    int rows = 32;
    while (rows > 4 && (int64_t)((nr + rows - 1) / rows) * chunks * groups * qmax <= 4096) rows /= 2;
    hipLaunchKernelGGL(k_qcorr_runs, dim3((unsigned)qmax * groups, (unsigned)((nr + rows - 1) / rows), chunks), dim3(256),
                       0, st, zd, img, nr, nc, xc, yc, cz, qmax, maxdqz, rows, out);
    const int64_t nh = (int64_t)(2 * maxdqz) * (2 * qmax) * qmax;
    hipLaunchKernelGGL(k_qcorr_assemble, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, st, out, maxdqz, qmax);
    return hipGetLastError();
}

}  // namespace idisim
