// The adjoint's sums as matrix products over the pixels (the separable form of adjoint.hip; no
// reference counterpart).
//
// k_adjoint needs, per emitter and tile, S = sum_p Im(w'_p e^{2 pi i tau}) and V = sum_p Im(.) dq_p.
// Over a square of T x T pixels about (cx, cy) let a, b be half a side along the rows and columns over
// the distance, p the unit vector to the centre, and x = t / |p + t a|, t in [-1, 1] along the rows, y
// alike.  Then along each axis p's change is exact to third order in two powers, and
//   tau = A + gx(x) . r' + gy(y) . r' + m . r',   m = mu x y + nu1 x^2 y + nu2 x y^2 + ka x^2 y^2,
//   dq  = v1 x + v2 x^2 + w1 y + w2 y^2 + m,      v1 = -k (a - (p a) p), v2 = -k ((p a)^2 - a^2) p / 2,
// so with X = e^{2 pi i (A + gx . r')}, Y = e^{2 pi i gy . r'}, T_a(y) = sum_x x^a w'(x, y) X (a complex
// matrix product of the weights with the phasors of all emitters) and Z_ab = sum_y y^b Y T_a(y)
//   S = Im [Z00 + i (c Z11 + e1 Z21 + e2 Z12 + k2 Z22) - c^2 / 2 Z22 - c (e1 Z32 + e2 Z23)],
//   V = v1 Im [Z10 + i (c Z21 + e1 Z31 + e2 Z22) - c^2 / 2 Z32]
//     + w1 Im [Z01 + i (c Z12 + e1 Z22 + e2 Z13) - c^2 / 2 Z23]
//     + v2 Im [Z20 + i c Z31] + w2 Im [Z02 + i c Z13] + mu Im [Z11 + i c Z22] + nu1 Im Z21 + nu2 Im Z12,
// (c, e1, e2, k2) = 2 pi (mu, nu1, nu2, ka) . r', with an x^3 in Z as f x, f = <x^4> / <x^2> (its best
// linear part); mu holds x^3 y and x y^3 in the same way.  The planner bounds what is
// left out.  Measured against 64 bits over 9 geometries (64^2 to 2000^2 pixels, even and uneven weights) 1.7e-7 .. 3.0e-7
// of the gradients (k_adjoint 2.2e-7 .. 4.8e-7).  A square takes 2 T sincos per emitter where k_adjoint takes T^2.
//
// Weights and phasors are split into two FP16 parts (T_0, T_1: three products; T_2 and T_3, of second
// order, the high parts alone), the weights scaled per square by a power of two (kHalfTop).  A wave owns a square
// and keeps its weights (of 32 pixels T_2's and T_3's in LDS: they spilled, 812 against 766 us of a
// gradient at 512^2 x 20000) while the workgroup's 256 emitters pass, T at a time: lane l holds emitter
// l % T, forms the phasors X of 4 columns per instruction in the operand layout, and after the products
// its rows y of T_a for that emitter.  The sums over y, the moments and their fold are FP32 (as
// k_adjoint's sums over 256 pixels); workgroup tiles of 2 x 2 squares are then folded in FP64 as there.
//
// Bound by the vector instructions of the sums over y (about 40 per row and emitter: 0.40 of the cycles at
// least, the matrix cores 0.36, 0.35 of the wave cycles wait for an issue slot).  k_adjoint -> this: 1880 -> 430 us at
// 512^2 x 20000 with amplitudes (squares of 32), 68 -> 42 us at 256^2 x 4096 (of 16).
#include "mfma_util.hpp"
#include "adjoint.hpp"

namespace idisim {

namespace {
constexpr int kMats = 6;  // weight operands: w' high, low, x w' high, low, x^2 w' high, x^3 w' high

// The table of one square: gx and gy (rev per length) of its rows and columns (gy with y), the constants of the sums, the scale of its weights,
// and the weight operands of every instruction.
struct SqConst {
    double del[3];  // dq of the square's centre about the workgroup tile's
    float mu[3], n1[3], n2[3], ka[3], v1[3], w1[3], v2[3], w2[3];
    float scale, pad;
};
template <int T>
struct SqTab {
    static constexpr int kSteps = T * T / 256;  // 256 / T columns per instruction
    float4 gx[T], gy[T];
    SqConst c;
    half8_t f[kSteps][kMats][64];
};

// The axes of a square: a, b and p as above, and their products.
struct SqAxes {
    Frame f;
    double a[3], b[3], pa, pb, aa, bb;
};

__device__ inline SqAxes sq_axes(const Geom& g, double cx, double cy, int T)
{
    SqAxes s{pixel_frame(g, cx, cy), {g.pix, 0.0, 0.0}, {0.0, g.pix, 0.0}, 0.0, 0.0, 0.0, 0.0};
    const double h = 0.5 * T / s.f.R;
    for (int i = 0; i < 3; ++i) {
        if (g.rot) {
            s.a[i] = g.M[3 * i] * g.pix;
            s.b[i] = g.M[3 * i + 1] * g.pix;
        }
        s.a[i] *= h;
        s.b[i] *= h;
        s.pa += s.f.rh[i] * s.a[i];
        s.pb += s.f.rh[i] * s.b[i];
        s.aa += s.a[i] * s.a[i];
        s.bb += s.b[i] * s.b[i];
    }
    return s;
}

// t / |p + t a|
__device__ inline float sq_coord(float t, float pa, float aa)
{
    return t / sqrtf(fmaf(t, fmaf(t, aa, 2.f * pa), 1.f));
}

__device__ inline void sq_const(const Geom& g, double cx, double cy, const SqAxes& s, const Frame& super, int T,
                                SqConst& o)
{
    // mu and ka from differences at t = +-s with s^2 = <t^4> / <t^2>: (mu + (q1 + q3) s^2) s^2 and
    // ka s^4 are m's parts odd and even in both
    const double f = adj_x4(T), d = sqrt(f) * 0.5 * T, pa = s.pa, pb = s.pb, k = -g.krev;
    const Frame pp = pixel_frame(g, cx + d, cy + d), pm = pixel_frame(g, cx + d, cy - d),
                mp = pixel_frame(g, cx - d, cy + d), mm = pixel_frame(g, cx - d, cy - d),
                p0 = pixel_frame(g, cx + d, cy), m0 = pixel_frame(g, cx - d, cy),
                zp = pixel_frame(g, cx, cy + d), zm = pixel_frame(g, cx, cy - d);
    for (int i = 0; i < 3; ++i) {
        const double p = s.f.rh[i], a = s.a[i], b = s.b[i], u0 = s.f.u[i];
        const double mu = ((pp.u[i] - pm.u[i]) - (mp.u[i] - mm.u[i])) / (4.0 * f);
        const double n1 = (1.5 * s.aa * pb - 7.5 * pa * pa * pb) * p + 3.0 * pa * pb * a + (1.5 * pa * pa - 0.5 * s.aa) * b;
        const double n2 = (1.5 * s.bb * pa - 7.5 * pb * pb * pa) * p + 3.0 * pa * pb * b + (1.5 * pb * pb - 0.5 * s.bb) * a;
        const double ka = (((pp.u[i] - p0.u[i]) - (zp.u[i] - u0)) + ((mm.u[i] - m0.u[i]) - (zm.u[i] - u0)) +
                           ((pm.u[i] - p0.u[i]) - (zm.u[i] - u0)) + ((mp.u[i] - m0.u[i]) - (zp.u[i] - u0))) /
                          (4.0 * f * f);
        // powers of t to powers of x: t = x + (p a) x^2
        o.mu[i] = (float)(k * mu);
        o.n1[i] = (float)(k * (n1 + pa * mu));
        o.n2[i] = (float)(k * (n2 + pb * mu));
        o.ka[i] = (float)(k * (ka + pb * n1 + pa * n2 + pa * pb * mu));
        o.v1[i] = (float)(k * (a - pa * p));
        o.w1[i] = (float)(k * (b - pb * p));
        o.v2[i] = (float)(k * 0.5 * (pa * pa - s.aa) * p);
        o.w2[i] = (float)(k * 0.5 * (pb * pb - s.bb) * p);
        o.del[i] = k * (u0 - super.u[i]);
    }
}
}  // namespace

// The table of every square: one workgroup per T x T pixels.  SPLIT: the field is summed from the
// forward's split partials and stored when field_out is given (k_adj_pixels_split), else read.  The
// loss is summed per 16 x 16 tile as there (the same bits).
template <int T, bool SPLIT>
__global__ __launch_bounds__(kAdjTile) void k_adj_sep_pixels(Geom g, const float4* __restrict__ partial, int splits,
                                                             const float2* __restrict__ field, float2* field_out,
                                                             const float* __restrict__ dLdI,
                                                             const float* __restrict__ target, int sq_y,
                                                             SqTab<T>* __restrict__ tab, double* __restrict__ loss_tile)
{
    constexpr int NS = (T / 16) * (T / 16);
    __shared__ double red[kAdjTile];
    __shared__ float wmax[4];
    const int l = threadIdx.x;
    const int sx = (blockIdx.x / sq_y) * T, sy = (blockIdx.x % sq_y) * T;
    const size_t npix = (size_t)g.n0 * g.n1;
    const int tiles_y = (g.n1 + 15) / 16;
    SqTab<T>& tb = tab[blockIdx.x];

    float wr[NS], wi[NS], m = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int tx = sx + 16 * (s / (T / 16)), ty = sy + 16 * (s % (T / 16));
        const int x = tx + (l >> 4), y = ty + (l & 15);
        double dr = 0.0, di = 0.0, res2 = 0.0;
        if (x < g.n0 && y < g.n1) {
            const size_t idx = (size_t)x * g.n1 + y;
            const Frame f = pixel_frame(g, (double)x, (double)y);
            double cs = 1.0, sn = 0.0;
            if (g.nf) pixel_phasor(g, f, cs, sn);
            float2 E;
            if (SPLIT) {
                double re, im;
                split_sum(partial, splits, npix, idx, re, im);
                E = split_field(g, f, cs, sn, re, im);
                if (field_out != nullptr) field_out[idx] = E;
            } else {
                E = field[idx];
            }
            adj_pixel_weight(g, f, cs, sn, E, idx, dLdI, target, dr, di, res2);
        }
        wr[s] = (float)dr;
        wi[s] = (float)di;
        m = fmaxf(m, fmaxf(fabsf(wr[s]), fabsf(wi[s])));
        if (target != nullptr) {
            const bool tile = tx < g.n0 && ty < g.n1;  // uniform
            if (s > 0) __syncthreads();
            red[l] = res2;
            __syncthreads();
            for (int q = kAdjTile / 2; q > 0; q >>= 1) {
                if (l < q) red[l] += red[l + q];
                __syncthreads();
            }
            if (l == 0 && tile) loss_tile[(size_t)(tx / 16) * tiles_y + ty / 16] = red[0];
        }
    }
    // the power of two that brings the largest weight to [2^13, 2^14) (weights that are not finite or all
    // zero: no scale)
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
    if ((l & 63) == 0) wmax[l >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    float sc = 1.f, back = 1.f;
    if (m > 0.f && m < INFINITY) {
        const int ex = min(max(ilogbf(m) + 1 - kHalfTop, -120), 120);
        sc = ldexpf(1.f, -ex);
        back = ldexpf(1.f, ex);
    }
    // The matrix instruction truncates its sums downwards; from square to square the weights' sign changes
    // and that bias cancels (phase gradients of 2000 x 2000 pixels 9.2e-7 from 64 bits without it, 3.2e-7 of
    // k_adjoint).
    if ((sx / T + sy / T) & 1) {
        sc = -sc;
        back = -back;
    }
    constexpr float hw = 0.5f * (T - 1);
    const double cx = sx + (double)hw, cy = sy + (double)hw;
    const SqAxes ax = sq_axes(g, cx, cy, T);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int rx = 16 * (s / (T / 16)) + (l >> 4), ry = 16 * (s % (T / 16)) + (l & 15);
        const float xs = sq_coord(((float)rx - hw) * (2.f / T), (float)ax.pa, (float)ax.aa);
        // operand word of (x, y): instruction x / (4 * 64 / T), lane y + T * (x / 4 of it), slot x % 4
        constexpr int kx = 4 * (64 / T);  // columns per instruction
        const int step = rx / kx, lane = ry + T * ((rx % kx) / 4), slot = rx & 3;
        const float ar = wr[s] * sc, ai = -wi[s] * sc;
        half2_t h0, l0, h1, l1, h2, l2, h3, l3;
        split_half(ar, ai, h0, l0);
        split_half(ar * xs, ai * xs, h1, l1);
        split_half(ar * xs * xs, ai * xs * xs, h2, l2);
        split_half(ar * xs * xs * xs, ai * xs * xs * xs, h3, l3);
        half2_t* o = reinterpret_cast<half2_t*>(&tb.f[step][0][0]);
        o[(0 * 64 + lane) * 4 + slot] = h0;
        o[(1 * 64 + lane) * 4 + slot] = l0;
        o[(2 * 64 + lane) * 4 + slot] = h1;
        o[(3 * 64 + lane) * 4 + slot] = l1;
        o[(4 * 64 + lane) * 4 + slot] = h2;
        o[(5 * 64 + lane) * 4 + slot] = h3;
    }
    // rows, columns and constants: about the centre of the square and of its workgroup tile
    if (l <= 2 * T) {
        if (l == 2 * T) {
            const Frame fs = pixel_frame(g, sx / (2 * T) * (2 * T) + (T - 0.5), sy / (2 * T) * (2 * T) + (T - 0.5));
            SqConst c;
            sq_const(g, cx, cy, ax, fs, T, c);
            c.scale = back;
            c.pad = 0.f;
            tb.c = c;
        } else {
            const bool row = l < T;
            const Frame f = row ? pixel_frame(g, (double)(sx + l), cy) : pixel_frame(g, cx, (double)(sy + l - T));
            const float4 q = make_float4((float)(-g.krev * (f.u[0] - ax.f.u[0])), (float)(-g.krev * (f.u[1] - ax.f.u[1])),
                                         (float)(-g.krev * (f.u[2] - ax.f.u[2])),
                                         row ? 0.f : sq_coord(((float)(l - T) - hw) * (2.f / T), (float)ax.pb, (float)ax.bb));
            if (row)
                tb.gx[l] = q;
            else
                tb.gy[l - T] = q;
        }
    }
}

// blockIdx.x: 256 emitters, blockIdx.y: `per` workgroup tiles of 2 x 2 squares.
template <int T, bool AMP>
__global__ __launch_bounds__(kBlock, T == 16 ? 4 : 2) void k_adjoint_sep(Geom g, const double* __restrict__ emit,
                                                                         const double* __restrict__ amp, int64_t n,
                                                                         const SqTab<T>* __restrict__ tab, int sq_x,
                                                                         int sq_y, int wt_y, int nwt, int per,
                                                                         double* __restrict__ partial)
{
    using Tr = SepTraits<T>;
    using acc_t = typename Tr::acc_t;
    constexpr int R = Tr::kRegs, STEPS = SqTab<T>::kSteps, kx = 4 * (64 / T), kLds = T == 32 ? 2 : 0;
    __shared__ float4 s_rec[kBlock];
    __shared__ float s_A[4][kBlock];
    __shared__ float4 s_sv[4][kBlock];
    __shared__ float s_re[AMP ? 4 : 1][AMP ? kBlock : 1];
    __shared__ float4 s_g[4][2 * T];  // the square's rows and columns
    __shared__ half8_t s_a[T == 32 ? 4 : 1][T == 32 ? STEPS * kLds : 1][T == 32 ? 64 : 1];  // operands of T_2, T_3
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, grp = l / T;
    const int64_t e = (int64_t)blockIdx.x * kBlock + tid;
    const int t0 = blockIdx.y * per, t1 = min(t0 + per, nwt);
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const float f4 = (float)adj_x4(T);

    for (int t = t0; t < t1; ++t) {
        const int qx = 2 * (t / wt_y) + (w >> 1), qy = 2 * (t % wt_y) + (w & 1);  // the wave's square
        const bool active = qx < sq_x && qy < sq_y;
        const Frame c = pixel_frame(g, (t / wt_y) * (2 * T) + (T - 0.5), (t % wt_y) * (2 * T) + (T - 0.5));
        {
            float4 rec = make_float4(0.f, 0.f, 0.f, 0.f);
            if (e < n) {
                const double* a4 = emit + 4 * e;
                const SplitRec r = make_split_rec(g, c, a4[0], a4[1], a4[2], a4[3], 1.0);
                rec = make_float4(r.x, r.y, r.z, r.A);
            }
            s_rec[tid] = rec;
            // A about the centres of the squares, reduced to [-1/2, 1/2]
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int x = 2 * (t / wt_y) + (q >> 1), y = 2 * (t % wt_y) + (q & 1);
                if (x >= sq_x || y >= sq_y) continue;  // uniform
                const double* d = tab[(size_t)x * sq_y + y].c.del;
                const double A = fma(d[0], (double)rec.x, fma(d[1], (double)rec.y, fma(d[2], (double)rec.z, (double)rec.w)));
                s_A[q][tid] = (float)(A - rint(A));
            }
        }
        const SqTab<T>& tb = tab[active ? (size_t)qx * sq_y + qy : 0];
        if (l < 2 * T) s_g[w][l] = l < T ? tb.gx[l] : tb.gy[l - T];
        if constexpr (kLds > 0) {
#pragma unroll
            for (int q = 0; q < STEPS * kLds; ++q) s_a[w][q][l] = tb.f[q / kLds][kMats - kLds + q % kLds][l];
        }
        __syncthreads();
        if (active) {
            Frag a[STEPS][kMats];
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
#pragma unroll
                for (int q = 0; q < kMats - kLds; ++q) a[s][q].v = tb.f[s][q][l];
            const SqConst& k = tb.c;
#pragma unroll 1
            for (int eb = 0; eb < kBlock; eb += T) {
                if (kLds > 0) asm volatile("" ::: "memory");  // the operands in LDS stay there
                float4 r = s_rec[eb + l % T];
                r.w = s_A[w][eb + l % T];
                acc_t tr[4], ti[4];  // T_0..T_3; the imaginary parts negated
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int i = 0; i < R; ++i) tr[q][i] = ti[q][i] = 0.f;
#pragma unroll
                for (int s = 0; s < STEPS; ++s) {
                    Frag xh, xl, zh, zl;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float4 q = s_g[w][kx * s + 4 * grp + i];
                        float u = fmaf(q.x, r.x, r.w);
                        u = fmaf(q.y, r.y, u);
                        u = fmaf(q.z, r.z, u);
                        split_half(__builtin_amdgcn_cosf(u), __builtin_amdgcn_sinf(u), xh.p[i], xl.p[i]);
                        zh.p[i] = rot90(xh.p[i]);
                        zl.p[i] = rot90(xl.p[i]);
                    }
#pragma unroll
                    for (int q = 0; q < kLds; ++q) a[s][kMats - kLds + q].v = s_a[w][s * kLds + q][l];
                    Tr::mma(a[s][0], xh, tr[0]);
                    Tr::mma(a[s][0], zh, ti[0]);
                    Tr::mma(a[s][2], xh, tr[1]);
                    Tr::mma(a[s][2], zh, ti[1]);
                    Tr::mma(a[s][4], xh, tr[2]);
                    Tr::mma(a[s][4], zh, ti[2]);
                    Tr::mma(a[s][5], xh, tr[3]);
                    Tr::mma(a[s][5], zh, ti[3]);
                    Tr::mma(a[s][1], xh, tr[0]);
                    Tr::mma(a[s][1], zh, ti[0]);
                    Tr::mma(a[s][3], xh, tr[1]);
                    Tr::mma(a[s][3], zh, ti[1]);
                    Tr::mma(a[s][0], xl, tr[0]);
                    Tr::mma(a[s][0], zl, ti[0]);
                    Tr::mma(a[s][2], xl, tr[1]);
                    Tr::mma(a[s][2], zl, ti[1]);
                }
                // moments over this lane's rows y
                float i00 = 0.f, i01 = 0.f, i02 = 0.f, i10 = 0.f, i11 = 0.f, r11 = 0.f, r12 = 0.f, i20 = 0.f, i22 = 0.f,
                      r21 = 0.f, r22 = 0.f, r00 = 0.f, i12 = 0.f, i21 = 0.f, r31 = 0.f, r13 = 0.f;
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    const int row = Tr::row(i, 0);  // + 4 grp
                    const float4 q = s_g[w][T + row + 4 * grp];
                    float u = q.x * r.x;
                    u = fmaf(q.y, r.y, u);
                    u = fmaf(q.z, r.z, u);
                    const float cy = __builtin_amdgcn_cosf(u), sy = __builtin_amdgcn_sinf(u);
                    const float y = q.w, y2 = y * y;
                    const float p0i = fmaf(sy, tr[0][i], -cy * ti[0][i]);
                    const float p1r = fmaf(cy, tr[1][i], sy * ti[1][i]), p1i = fmaf(sy, tr[1][i], -cy * ti[1][i]);
                    const float p2r = fmaf(cy, tr[2][i], sy * ti[2][i]), p2i = fmaf(sy, tr[2][i], -cy * ti[2][i]);
                    i00 += p0i;
                    i01 = fmaf(y, p0i, i01);
                    i02 = fmaf(y2, p0i, i02);
                    i10 += p1i;
                    i11 = fmaf(y, p1i, i11);
                    r11 = fmaf(y, p1r, r11);
                    r12 = fmaf(y2, p1r, r12);
                    r13 = fmaf(y2 * y, p1r, r13);
                    r31 = fmaf(y, fmaf(cy, tr[3][i], sy * ti[3][i]), r31);
                    i20 += p2i;
                    i22 = fmaf(y2, p2i, i22);
                    r21 = fmaf(y, p2r, r21);
                    r22 = fmaf(y2, p2r, r22);
                    i12 = fmaf(y2, p1i, i12);
                    i21 = fmaf(y, p2i, i21);
                    if (AMP) r00 += fmaf(cy, tr[0][i], sy * ti[0][i]);
                }
                // the fold is linear in the moments: each lane folds its own rows
                const float tp = (float)kTwoPi;
                const float cc = tp * (k.mu[0] * r.x + k.mu[1] * r.y + k.mu[2] * r.z);
                const float e1 = tp * (k.n1[0] * r.x + k.n1[1] * r.y + k.n1[2] * r.z);
                const float e2 = tp * (k.n2[0] * r.x + k.n2[1] * r.y + k.n2[2] * r.z);
                const float k2 = tp * (k.ka[0] * r.x + k.ka[1] * r.y + k.ka[2] * r.z);
                const float h2 = -0.5f * cc * cc, fc = f4 * cc;
                const float s2 = fc * fmaf(e1, i12, e2 * i21);  // c (e1 Z32 + e2 Z23)
                float S = i00 + (cc * r11 + e1 * r21 + e2 * r12 + k2 * r22 + h2 * i22 - s2);
                const float zx = i10 + (cc * r21 + e1 * r31 + e2 * r22 + f4 * h2 * i12);
                const float zy = i01 + (cc * r12 + e1 * r22 + e2 * r13 + f4 * h2 * i21);
                const float zxx = fmaf(cc, r31, i20), zyy = fmaf(cc, r13, i02), zxy = fmaf(cc, r22, i11);
                float V[3], Re = 0.f;
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    V[d] = k.v1[d] * zx + k.w1[d] * zy + k.v2[d] * zxx + k.w2[d] * zyy + k.mu[d] * zxy +
                           k.n1[d] * i21 + k.n2[d] * i12 + (float)k.del[d] * S;
                if (AMP) Re = r00 - (cc * i11 + e1 * i21 + e2 * i12 + k2 * i22) + h2 * r22 - fc * fmaf(e1, r12, e2 * r21);
#pragma unroll
                for (int d = T; d < 64; d <<= 1) {  // over the lane groups
                    S += __shfl_xor(S, d);
#pragma unroll
                    for (int q = 0; q < 3; ++q) V[q] += __shfl_xor(V[q], d);
                    if (AMP) Re += __shfl_xor(Re, d);
                }
                if (l < T) {
                    s_sv[w][eb + l] = make_float4(S * k.scale, V[0] * k.scale, V[1] * k.scale, V[2] * k.scale);
                    if (AMP) s_re[w][eb + l] = Re * k.scale;
                }
            }
        } else {
            for (int q = l; q < kBlock; q += 64) {
                s_sv[w][q] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (AMP) s_re[w][q] = 0.f;
            }
        }
        __syncthreads();
        // the fold of k_adjoint, about the workgroup tile's centre
        if (e < n) {
            double S = 0.0, V[3] = {0.0, 0.0, 0.0}, Re = 0.0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 v = s_sv[q][tid];
                S += (double)v.x;
                V[0] += (double)v.y;
                V[1] += (double)v.z;
                V[2] += (double)v.w;
                if (AMP) Re += (double)s_re[q][tid];
            }
            const double* a4 = emit + 4 * e;
            const SplitRec r = make_split_rec(g, c, a4[0], a4[1], a4[2], a4[3], 1.0);
            const float b[3] = {(float)a4[0] * r.iD - (float)c.rh[0] * r.sigma,
                                (float)a4[1] * r.iD - (float)c.rh[1] * r.sigma,
                                (float)a4[2] * r.iD - (float)c.rh[2] * r.sigma};
            const double ma = (double)r.amp, ik = 1.0 / g.krev;
            S *= ma;
#pragma unroll
            for (int d = 0; d < 3; ++d) acc[d] += g.k * (((double)b[d] - c.u[d]) * S + ma * V[d] * ik);
            if (!g.nf && g.secondorder) {  // W is folded: lam ~ 1
                const double L = S * g.k / c.R;
                acc[0] += L * (double)r.x;
                acc[1] += L * (double)r.y;
            }
            acc[3] += S;
            if (AMP) acc[4] += ma * Re;
        }
        __syncthreads();  // s_rec and s_sv consumed
    }
    if (e < n) {
        const double a = (amp != nullptr) ? amp[e] : 1.0;
        double* o = partial + ((size_t)blockIdx.y * n + e) * 5;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] = -2.0 * a * acc[d];
        if (AMP) o[4] = 2.0 * acc[4];
    }
}

AdjointSepLayout adjoint_sep_layout(const Geom& g, int T, int64_t n, int num_cus, int blocks_per_cu)
{
    AdjointSepLayout L;
    L.T = T;
    L.sq_x = (g.n0 + T - 1) / T;
    L.sq_y = (g.n1 + T - 1) / T;
    L.wt_y = (L.sq_y + 1) / 2;
    L.nwt = ((L.sq_x + 1) / 2) * L.wt_y;
    L.ntiles = ((g.n0 + 15) / 16) * ((g.n1 + 15) / 16);
    L.egroups = (n + kBlock - 1) / kBlock;
    // workgroup tiles per workgroup: the fewest rounds of resident workgroups (as adjoint_layout)
    const int64_t slots = (int64_t)num_cus * (blocks_per_cu > 0 ? blocks_per_cu : 1);
    int64_t best = INT64_MAX;
    L.per = L.nwt;
    for (int per = 1; per <= L.nwt; ++per) {
        const int64_t splits = (L.nwt + per - 1) / per;
        if (splits > 65535 || (per > 1 && splits == (L.nwt + per - 2) / (per - 1))) continue;
        const int64_t span = (L.egroups * splits + slots - 1) / slots * per;
        if (span <= best) {
            best = span;
            L.per = per;
        }
    }
    L.splits = (L.nwt + L.per - 1) / L.per;
    const size_t sq = (size_t)L.sq_x * L.sq_y;
    L.tab_bytes = sq * (T == 16 ? sizeof(SqTab<16>) : sizeof(SqTab<32>));
    L.part_bytes = (size_t)L.splits * (size_t)n * 5 * sizeof(double);
    L.bytes = L.tab_bytes + L.part_bytes + (size_t)L.ntiles * sizeof(double);
    return L;
}

int adjoint_sep_occupancy(int T, bool amp)
{
    int nb = 0;
    const hipError_t e =
        T == 16 ? (amp ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_adjoint_sep<16, true>, kBlock, 0)
                       : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_adjoint_sep<16, false>, kBlock, 0))
                : (amp ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_adjoint_sep<32, true>, kBlock, 0)
                       : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_adjoint_sep<32, false>, kBlock, 0));
    return e == hipSuccess && nb > 0 ? nb : 1;
}

template <int T>
static hipError_t launch_adjoint_sep_t(const Geom& g, const AdjointSepLayout& L, const double* emit, const double* amp,
                                       int64_t n, const float2* field, const float* dLdI, const float* target,
                                       double* loss, void* scratch, float* grad_pos, float* grad_phase,
                                       float* grad_amp, hipStream_t st, const float4* fwd_partial, int fwd_splits,
                                       float2* field_out)
{
    SqTab<T>* tab = static_cast<SqTab<T>*>(scratch);
    double* partial = reinterpret_cast<double*>(static_cast<char*>(scratch) + L.tab_bytes);
    double* loss_tile = reinterpret_cast<double*>(static_cast<char*>(scratch) + L.tab_bytes + L.part_bytes);
    const dim3 sq((unsigned)(L.sq_x * L.sq_y));
    if (fwd_partial != nullptr)
        hipLaunchKernelGGL((k_adj_sep_pixels<T, true>), sq, dim3(kAdjTile), 0, st, g, fwd_partial, fwd_splits, nullptr,
                           field_out, nullptr, target, L.sq_y, tab, loss_tile);
    else
        hipLaunchKernelGGL((k_adj_sep_pixels<T, false>), sq, dim3(kAdjTile), 0, st, g, nullptr, 0, field, nullptr, dLdI,
                           target, L.sq_y, tab, loss_tile);
    const dim3 grid((unsigned)L.egroups, (unsigned)L.splits);
    if (grad_amp != nullptr)
        hipLaunchKernelGGL((k_adjoint_sep<T, true>), grid, dim3(kBlock), 0, st, g, emit, amp, n, tab, L.sq_x, L.sq_y,
                           L.wt_y, L.nwt, L.per, partial);
    else
        hipLaunchKernelGGL((k_adjoint_sep<T, false>), grid, dim3(kBlock), 0, st, g, emit, amp, n, tab, L.sq_x, L.sq_y,
                           L.wt_y, L.nwt, L.per, partial);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_adjoint_finalize(partial, L.splits, n, grad_pos, grad_phase, grad_amp, loss_tile, L.ntiles,
                                   target != nullptr ? loss : nullptr, st);
}

hipError_t launch_adjoint_sep(const Geom& g, const AdjointSepLayout& L, const double* emit, const double* amp,
                              int64_t n, const float2* field, const float* dLdI, const float* target, double* loss,
                              void* scratch, float* grad_pos, float* grad_phase, float* grad_amp, hipStream_t st,
                              const float4* fwd_partial, int fwd_splits, float2* field_out)
{
    if (fwd_partial != nullptr && target == nullptr) return hipErrorInvalidValue;
    if (g.foldw == 0 && (g.nf || g.secondorder)) return hipErrorInvalidValue;  // needs W folded into A
    return L.T == 16 ? launch_adjoint_sep_t<16>(g, L, emit, amp, n, field, dLdI, target, loss, scratch, grad_pos,
                                                grad_phase, grad_amp, st, fwd_partial, fwd_splits, field_out)
                     : launch_adjoint_sep_t<32>(g, L, emit, amp, n, field, dLdI, target, loss, scratch, grad_pos,
                                                grad_phase, grad_amp, st, fwd_partial, fwd_splits, field_out);
}

}  // namespace idisim
