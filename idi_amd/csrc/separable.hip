// Forward sums as matrix products over the emitters (tile variants 17..22; no reference counterpart).
//
// Over a small rectangle of pixels the phase of a pair is, but for a small mixed remainder, a row part
// plus a column part (geometry.hpp, sep_mixed):
//   tau = [A + dq(x, cy) . r'] + [dq(cx, y) - dq(c)] . r' + m(x, y) . r'
// so with X = a e^{2 pi i [A + ...]} per (row, emitter), Y per (column, emitter) and
// M = 2 pi m . r' (a few 1e-3 rad; the planner bounds it),
//   E(x, y) = sum_j X Y e^{i M} = sum_j X Y  +  2 pi i m(x, y) . sum_j r'_j X Y
//                                 - 1/2 (2 pi |mu| dx dy)^2 sum_j (mu' . r'_j)^2 X Y   (variant 22)
// to first order in M, or with the second order along the leading direction mu of m (m = dx dy mu +
// higher orders, mu' = mu / |mu|).  m lies nearly in two directions (sep_basis_of), and variants 17,
// 19 and 21 keep those alone.  Each sum is a complex matrix product over the emitters, which the
// matrix cores form; a rectangle of a x b pixels takes a + b sincos per emitter instead of the
// a b / 2 of the mirror-pair tiles.
//
// The sums without a remainder keep FP32's precision: X and Y are formed in FP32 and split into two
// FP16 parts each (22 bits; X_hi Y_hi + X_hi Y_lo + X_lo Y_hi, the products exact, the sums in FP32).
// The split by itself costs 7e-8 relative L2, whatever the amplitudes (kHalfTop).  The remainder's sums are
// weighted by M and need 1e-3 of that: the high parts alone (variant 22, whose M is ten times as large,
// splits the one along mu).
// Relative L2 of the field against 64 bits, with the mirror-pair tiles in brackets: 100000 emitters on 512 x 512
// pixels 3.8e-7 to 4.0e-7 (6.1e-7 to 7.5e-7), 12345 on 333 x 211 in the far field 3.6e-7 (6.3e-7), 64 shots of
// 1000 to 50000 on 256 x 256 at 0.1 m (variant 22, intensity) 5.9e-7 (1.6e-6), 1e6 with amplitudes on
// 1024 x 1024 4.3e-7 (3.8e-7).
//
// A wave owns one rectangle.  v_mfma_f32_32x32x16_f16 (16x16x32 for T = 16) takes 8 (16) emitters per
// instruction as K = (re, im) pairs; lane l holds row l % T of X and column l % T of Y for 4 of them,
// so every phasor is formed in the lane and register that the instruction reads it from, and only the
// emitter records (FP64, about the workgroup's centre, once per workgroup of 2 x 2 rectangles) go
// through LDS.
//
// What bounds it: per step of 8 emitters a wave of 32 x 32 pixels issues 77 vector, 12 transcendental
// and 10 matrix instructions.  Counters of variant 20 (100000 emitters, 512 x 512): the matrix cores are busy
// for 0.60 of the cycles and the vector instructions take 0.36 at least; with one wave per SIMD the two
// hardly overlap, and the clock falls to 1.65 GHz under the counters (2.12 with the mirror-pair kernel).  That image takes
// 1.05 ms against 3.33 ms with variant 13.  Sharing X between two blocks of columns (variants 19, 20:
// one wave per SIMD, 512 registers) saves a quarter of the vector instructions and 10% of the time.
#include "mfma_util.hpp"

namespace idisim {

namespace {
// Emitters between two merges of the FP32 sums into the long ones, as in the other tiles.  A step of 8 or 16
// emitters rounds into its sum six times: with 512 emitters an image of random phases is 4.0e-7 off 64 bits,
// with 256 3.1e-7 (the mirror-pair tiles 3.2e-7), with 128 2.5e-7 in 3% more time.
constexpr int kSepMerge = kChunk;
static_assert(kSepMerge % kBlock == 0, "a lane's staged emitters share the sign of their merge interval");

// Shape of a kernel.  T: rows of a wave's rectangle and columns of its NB blocks (T x NB T pixels);
// NE: directions along which the mixed remainder is kept (3: all; 2: sep_basis_of); Q2: for larger
// remainders (M of 1e-2), the second-order term along mu, and the first-order sum along mu with both
// parts of the split, as FP16's rounding of M would come near the tolerance.
template <int T_, int NB_, int NE_, bool Q2_>
struct SepShape {
    static constexpr int T = T_, NB = NB_, NE = NE_;
    static constexpr bool Q2 = Q2_;
    static constexpr int R = SepTraits<T>::kRegs, kStep = SepTraits<T>::kStep;
    static constexpr int kRows = 2 * T, kCols = 2 * T * NB;  // workgroup tile: 2 x 2 waves
    static constexpr bool kBasis = NE == 2 || Q2;  // the remainder along the wave's own directions
    static constexpr bool kLdsSums = T == 32;  // long sums in LDS (registers hold only T = 16's)
    static constexpr int kStoreUnroll = kLdsSums ? 1 : NB * R;  // the FP64 store is long
    // emitters staged at a time: two per lane where one workgroup fills a CU, so that the FP64 chains of
    // two records overlap
    static constexpr int kStage = NB == 2 ? 2 * kChunk : kChunk;
    static constexpr int kSlots = kStage + 2 * kStep;  // the pipelined loop reads one step past the end
    static constexpr int kWaves = NB == 2 ? 1 : (T == 32 ? 2 : (NE == 2 ? 4 : 3));  // waves per SIMD
};

template <class S>
struct SepAcc {
    typename SepTraits<S::T>::acc_t e0[S::NB][2];         // sum X Y (re, im)
    typename SepTraits<S::T>::acc_t e1[S::NB][S::NE][2];  // sum (b_k . r') X Y
    typename SepTraits<S::T>::acc_t e2[S::NB][2];         // sum (mu' . r')^2 X Y (Q2)
};

// LDS of a workgroup: the staged emitters and, for T = 32, the long sums in FP64 (32 or 64 per lane).
template <class S>
struct SepLds {
    float4 r[S::kSlots];  // r' (scaled), A
    // the weights of the remainder's sums as FP16: r' as (x, y) and (z, z), the same for all waves, or its
    // components along the directions of each wave's rectangle: both (NE = 2), or the two across mu (Q2)
    half2_t h[S::kBasis ? 4 : 2][S::kSlots];
    float amp[S::kSlots];
    float c[S::Q2 ? 4 : 1][S::Q2 ? S::kSlots : 1];     // mu' . r' of each wave
    half2_t c2[S::Q2 ? 4 : 1][S::Q2 ? S::kSlots : 1];  // its square, twice
    double k[S::kLdsSums ? 4 : 1][S::kLdsSums ? 2 * S::NB * S::R : 1][64];
    float amax[4];
    float b[4][3][3];  // orthonormal directions of each wave's rectangle, mu / |mu| first
};

// The operands of one step of kStep emitters: X (high and low parts), its products with the
// remainder's weights, Y as (cos, -sin), which against (re, im) of X gives the real part, and Y turned
// by 90 degrees, (sin, cos), which gives the imaginary part.
template <class S>
struct SepFrags {
    Frag xh, xl, x1[S::NE], x2;
    Frag ch, cl;  // Q2: X mu' . r'
    Frag yh[S::NB], yl[S::NB], zh[S::NB], zl[S::NB];
};

// The staged words of a lane's four emitters of a step.
template <class S>
struct SepRecs {
    float4 r[4];
    half2_t h[4], z[4], c2[4];
    float a[4], c[4];
};

// e: the lane's first of four emitters.  AMP: the phasors carry the amplitudes.
template <class S, bool AMP>
__device__ __forceinline__ void sep_load(const SepLds<S>& s, int e, int w, SepRecs<S>& q)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        q.r[i] = s.r[e + i];
        q.h[i] = s.h[S::kBasis ? w : 0][e + i];
        if constexpr (!S::kBasis) q.z[i] = s.h[1][e + i];
        if constexpr (S::Q2) {
            q.c[i] = s.c[w][e + i];
            q.c2[i] = s.c2[w][e + i];
        }
        if (AMP) q.a[i] = s.amp[e + i];
    }
}

template <class S, bool AMP>
__device__ __forceinline__ void sep_gen(const SepRecs<S>& q, const float (&gx)[3], const float (&gy)[S::NB][3],
                                        SepFrags<S>& f)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 r = q.r[i];
        const half2_t h0 = q.h[i];
        float t = fmaf(gx[0], r.x, r.w);
        t = fmaf(gx[1], r.y, t);
        t = fmaf(gx[2], r.z, t);
        float c = __builtin_amdgcn_cosf(t), sn = __builtin_amdgcn_sinf(t);
        if (AMP) {
            c *= q.a[i];
            sn *= q.a[i];
        }
        split_half<AMP>(c, sn, f.xh.p[i], f.xl.p[i]);
        constexpr int k0 = S::Q2 ? 1 : 0;
        f.x1[k0].p[i] = f.xh.p[i] * half2_t{h0.x, h0.x};
        f.x1[k0 + 1].p[i] = f.xh.p[i] * half2_t{h0.y, h0.y};
        if constexpr (!S::kBasis) f.x1[2].p[i] = f.xh.p[i] * q.z[i];
        if constexpr (S::Q2) {
            f.x2.p[i] = f.xh.p[i] * q.c2[i];
            split_half(c * q.c[i], sn * q.c[i], f.ch.p[i], f.cl.p[i]);
        }
#pragma unroll
        for (int b = 0; b < S::NB; ++b) {
            float u = gy[b][0] * r.x;
            u = fmaf(gy[b][1], r.y, u);
            u = fmaf(gy[b][2], r.z, u);
            split_half<AMP>(__builtin_amdgcn_cosf(u), -__builtin_amdgcn_sinf(u), f.yh[b].p[i], f.yl[b].p[i]);
            f.zh[b].p[i] = rot90(f.yh[b].p[i]);
            f.zl[b].p[i] = rot90(f.yl[b].p[i]);
        }
    }
}

template <class S>
__device__ __forceinline__ void sep_mma(const SepFrags<S>& f, SepAcc<S>& acc)
{
    using Tr = SepTraits<S::T>;
#pragma unroll
    for (int b = 0; b < S::NB; ++b) {
        Tr::mma(f.xh, f.yh[b], acc.e0[b][0]);
        Tr::mma(f.xh, f.zh[b], acc.e0[b][1]);
#pragma unroll
        for (int k = 0; k < S::NE; ++k) {
            Tr::mma(S::Q2 && k == 0 ? f.ch : f.x1[k], f.yh[b], acc.e1[b][k][0]);
            Tr::mma(S::Q2 && k == 0 ? f.ch : f.x1[k], f.zh[b], acc.e1[b][k][1]);
            if (k == 0) {
                Tr::mma(f.xh, f.yl[b], acc.e0[b][0]);
                Tr::mma(f.xh, f.zl[b], acc.e0[b][1]);
            }
        }
        if constexpr (S::Q2) {
            Tr::mma(f.x2, f.yh[b], acc.e2[b][0]);
            Tr::mma(f.x2, f.zh[b], acc.e2[b][1]);
            Tr::mma(f.ch, f.yl[b], acc.e1[b][0][0]);
            Tr::mma(f.ch, f.zl[b], acc.e1[b][0][1]);
            Tr::mma(f.cl, f.yh[b], acc.e1[b][0][0]);
            Tr::mma(f.cl, f.zh[b], acc.e1[b][0][1]);
        }
        Tr::mma(f.xl, f.yh[b], acc.e0[b][0]);
        Tr::mma(f.xl, f.zh[b], acc.e0[b][1]);
    }
}

// The matrix instructions of one step spread between the vector instructions of the next, for the shape with the
// most of them in one wave per SIMD (variant 20: 1.138 against 1.158 ms with amplitudes and 1.094 against
// 1.100 without, 100000 emitters on 512 x 512); the compiler's own order is better elsewhere (variant 17 with
// amplitudes 1.140 against 1.164, 18 1.267 against 1.281, 19 1.010 against 1.026).
template <class S>
__device__ __forceinline__ void sep_interleave()
{
    if constexpr (S::NB == 2 && S::NE == 3) {
        constexpr int kMma = S::NB * (6 + 2 * S::NE);
        constexpr int kValu = 4 * (8 + S::NE + 10 * S::NB);
#pragma unroll
        for (int i = 0; i < kMma; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, kValu / kMma, 0);
        }
    }
}

// The long sums of a lane's pixels, word i = b R + register of block b, part p (re, im).  T = 16: FP32 with
// compensations in registers; T = 32: FP64 in LDS, added to without reading them back (ds_add_f64; four
// words read, compensated and written cost 1.151 against 1.053 ms for 100000 emitters on 512 x 512).
template <class S>
struct SepOut {
    static constexpr int N = S::NB * S::R;
    float v[S::kLdsSums ? 1 : 4][N];
    double (*k)[64];
    int l;
    __device__ __forceinline__ void clear(int p, int i)
    {
        if constexpr (S::kLdsSums)
            k[p * N + i][l] = 0.0;
        else
            v[p][i] = v[2 + p][i] = 0.f;
    }
    __device__ __forceinline__ void add(int p, int i, float x)
    {
        if constexpr (S::kLdsSums)
            (void)__hip_atomic_fetch_add(&k[p * N + i][l], (double)x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else
            kahan_add(v[p][i], v[2 + p][i], x);
    }
    __device__ __forceinline__ void scale(int p, int i, float f)  // by a power of two
    {
        if constexpr (S::kLdsSums) {
            k[p * N + i][l] *= (double)f;
        } else {
            v[p][i] *= f;
            v[2 + p][i] *= f;
        }
    }
    __device__ __forceinline__ double value(int p, int i) const
    {
        if constexpr (S::kLdsSums)
            return k[p * N + i][l];
        else
            return (double)v[p][i] - (double)v[2 + p][i];
    }
    // the sum and its compensation, as the split partials hold them (value = x - y)
    __device__ __forceinline__ float2 parts(int p, int i) const
    {
        if constexpr (S::kLdsSums) {
            const double d = k[p * N + i][l];
            const float sum = (float)d;
            return make_float2(sum, (float)((double)sum - d));
        } else {
            return make_float2(v[p][i], v[2 + p][i]);
        }
    }
};

// Pixel of word index i (b R + register) of lane l in wave w of a workgroup tile.
template <class S>
__device__ __forceinline__ void sep_pixel(int tx0, int ty0, int w, int l, int i, int& x, int& y)
{
    x = tx0 + S::T * (w >> 1) + SepTraits<S::T>::row(i % S::R, l / S::T);
    y = ty0 + S::T * S::NB * (w & 1) + S::T * (i / S::R) + l % S::T;
}

// The sums of the workgroup's 2 x 2 rectangles over emitters [e0, e1), into o (sep_pixel's order).
//
// The instruction truncates its sums of eight products downwards: 7e-10 per emitter in both parts of the
// field, which grows with the number of emitters (1.1e-6 of the field of 1e6, where the mirror-pair
// tiles have 3.8e-7).  So the sign of X changes from one merge interval to the next (and from one split to
// the next: `split`), and with it that of what is merged; X's weights for the remainder's sums change too.
template <class S, bool HAS_AMP>
__device__ __forceinline__ void sep_tile(const Geom& g, const double* __restrict__ emit,
                                         const double* __restrict__ amp, int64_t e0, int64_t e1, int split, int tx0,
                                         int ty0, SepLds<S>& s, SepOut<S>& o)
{
    constexpr int T = S::T, NB = S::NB, R = S::R, NE = S::NE;
    constexpr bool Q2 = S::Q2;
    constexpr float hx = 0.5f * (T - 1), hy = 0.5f * (NB * T - 1);
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, grp = l / T;
    const int sx = tx0 + T * (w >> 1), sy = ty0 + T * NB * (w & 1);  // the wave's rectangle
    const bool active = sx < g.n0 && sy < g.n1;
    const float inv = 1.f / g.sepscale;

    // the records' centre: of the whole workgroup tile, also where the detector ends inside it
    const Frame c = pixel_frame(g, tx0 + (T - 0.5), ty0 + (T * NB - 0.5));
    float gx[3], gy[NB][3];
    {
        const double cx = sx + (double)hx, cy = sy + (double)hy;
        const Frame fc = pixel_frame(g, cx, cy), fx = pixel_frame(g, (double)(sx + l % T), cy);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            gx[k] = (float)(-g.krev * (fx.u[k] - c.u[k])) * inv;
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const Frame fy = pixel_frame(g, cx, (double)(sy + T * b + l % T));
#pragma unroll
            for (int k = 0; k < 3; ++k) gy[b][k] = (float)(-g.krev * (fy.u[k] - fc.u[k])) * inv;
        }
    }
    if (S::kBasis && l == 0) {
        double r[3];
        pixel_pos(g, sx + (double)hx, sy + (double)hy, r);
        float b[2][3];
        sep_basis_of(make_sep_frame(g, r), b);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            s.b[w][0][k] = b[0][k];
            s.b[w][1][k] = b[1][k];
            s.b[w][2][k] = b[0][(k + 1) % 3] * b[1][(k + 2) % 3] - b[0][(k + 2) % 3] * b[1][(k + 1) % 3];
        }
    }

    // amplitudes: scaled by the power of two that brings the largest of the range to [2^13, 2^14)
    float ascale = 1.f, aback = 1.f;
    if (HAS_AMP && amp != nullptr) {
        float m = 0.f;
        for (int64_t e = e0 + tid; e < e1; e += kBlock) m = fmaxf(m, fabsf((float)amp[e]));
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
        if (l == 0) s.amax[w] = m;
        __syncthreads();
        m = fmaxf(fmaxf(s.amax[0], s.amax[1]), fmaxf(s.amax[2], s.amax[3]));
        if (m > 0.f && m < INFINITY) {
            const int ex = min(max(ilogbf(m) + 1 - kHalfTop, -120), 120);
            ascale = ldexpf(1.f, -ex);
            aback = ldexpf(1.f, ex);
        }
    }
    SepAcc<S> acc;
    o.k = s.k[S::kLdsSums ? w : 0];
    o.l = l;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                acc.e0[b][p][i] = 0.f;
                if (Q2) acc.e2[b][p][i] = 0.f;
#pragma unroll
                for (int k = 0; k < NE; ++k) acc.e1[b][k][p][i] = 0.f;
                o.clear(p, b * R + i);
            }
        }
    }

    // the long sums take what the accumulators hold, without `npad` padding emitters, and these start anew
    auto merge = [&](float sign, float npad) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int i = 0; i < R; ++i) {
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    o.add(p, b * R + i, sign * (p ? acc.e0[b][p][i] : acc.e0[b][p][i] - npad));
                    acc.e0[b][p][i] = 0.f;
                }
            }
        }
    };
    // X's sign of an emitter: that of its merge interval
    auto sign_of = [&](int64_t e) { return (((e - e0) / kSepMerge + split) & 1) ? -1.f : 1.f; };

    for (int64_t base = e0; base < e1; base += S::kStage) {
        const int cnt = (e1 - base) < (int64_t)S::kStage ? (int)(e1 - base) : S::kStage;
        const int pad = (cnt + 2 * S::kStep - 1) / (2 * S::kStep) * (2 * S::kStep);
        __syncthreads();  // the previous emitters have been consumed by every lane
#pragma unroll
        for (int q = 0; q < S::kStage; q += kBlock) {
            const int j = q + tid;
            if (j >= pad) break;
            const float sign = sign_of(base + q);
            SplitRec r = {};
            if (j < cnt) {
                const int64_t e = base + j;
                const double* a4 = emit + 4 * e;
                const double ea = (HAS_AMP && amp != nullptr) ? amp[e] : 1.0;
                r = make_split_rec(g, c, a4[0], a4[1], a4[2], a4[3], ea);
                // half a revolution, within [-1/2, 1/2] as A itself
                if (!HAS_AMP && sign < 0.f) r.A -= copysignf(0.5f, r.A);
            } else if (!HAS_AMP) {
                // the last steps' missing emitters: at the origin, with phases 0 and 1/2 in turn,
                // +1 and -1 in every pixel; an odd one is taken off below
                r.A = ((j - cnt) & 1) ? 0.5f : 0.f;
            }
            const float x = r.x * g.sepscale, y = r.y * g.sepscale, z = r.z * g.sepscale;
            s.r[j] = make_float4(x, y, z, r.A);
            const float sx = sign * x, sy = sign * y, sz = sign * z;
            if constexpr (S::kBasis) {
                constexpr int k0 = Q2 ? 1 : 0;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float(*d)[3] = s.b[v];
                    s.h[v][j] = half2_t{(_Float16)(d[k0][0] * sx + d[k0][1] * sy + d[k0][2] * sz),
                                        (_Float16)(d[k0 + 1][0] * sx + d[k0 + 1][1] * sy + d[k0 + 1][2] * sz)};
                    if constexpr (Q2) {
                        const float q1 = d[0][0] * sx + d[0][1] * sy + d[0][2] * sz;
                        s.c[v][j] = q1;
                        s.c2[v][j] = half2_t{(_Float16)(sign * q1 * q1), (_Float16)(sign * q1 * q1)};
                    }
                }
            } else {
                s.h[0][j] = half2_t{(_Float16)sx, (_Float16)sy};
                s.h[1][j] = half2_t{(_Float16)sz, (_Float16)sz};
            }
            if (HAS_AMP) s.amp[j] = r.amp * (sign * ascale);
        }
        const float npad = HAS_AMP ? 0.f : (float)((pad - cnt) & 1);
        __syncthreads();
        if (!active) continue;
        SepFrags<S> f0, f1;
        SepRecs<S> q0, q1;
        if constexpr (T == 32) {
            // the operands of a step are formed during the matrix instructions of the step before
            // (past the last step: of the words left there, unused)
            sep_load<S, HAS_AMP>(s, 4 * grp, w, q0);
            sep_gen<S, HAS_AMP>(q0, gx, gy, f0);
        }
        for (int q = 0; q < pad; q += kSepMerge) {
            const int end = min(q + kSepMerge, pad);
            if constexpr (T == 16) {  // four waves per SIMD overlap by themselves (1.56 against 1.67 ms)
                for (int e = q; e < end; e += S::kStep) {
                    sep_load<S, HAS_AMP>(s, e + 4 * grp, w, q0);
                    sep_gen<S, HAS_AMP>(q0, gx, gy, f0);
                    sep_mma<S>(f0, acc);
                }
            } else {
                for (int e = q; e < end; e += 2 * S::kStep) {
                    sep_load<S, HAS_AMP>(s, e + S::kStep + 4 * grp, w, q1);
                    sep_gen<S, HAS_AMP>(q1, gx, gy, f1);
                    sep_mma<S>(f0, acc);
                    sep_interleave<S>();
                    sep_load<S, HAS_AMP>(s, e + 2 * S::kStep + 4 * grp, w, q0);
                    sep_gen<S, HAS_AMP>(q0, gx, gy, f0);
                    sep_mma<S>(f1, acc);
                    sep_interleave<S>();
                }
            }
            merge(sign_of(base + q), end == pad ? npad : 0.f);
        }
    }
    if (!active) return;
    // the mixed remainder's terms, then the amplitude scale
    double r[3];
    pixel_pos(g, sx + (double)hx, sy + (double)hy, r);
    const SepFrame f = make_sep_frame(g, r);
    const float kap = (float)kTwoPi * inv;
    const float mun = (f.mu[0] * f.mu[0] + f.mu[1] * f.mu[1] + f.mu[2] * f.mu[2]) * kap * kap;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const float dy = (float)(T * b + l % T) - hy;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const float dx = (float)SepTraits<T>::row(i, grp) - hx;
            float m[3];
            sep_mixed(f, dx, dy, m);
            float ar = 0.f, ai = 0.f;
#pragma unroll
            for (int k = 0; k < NE; ++k) {
                float mk = m[k];
                if constexpr (S::kBasis) mk = m[0] * s.b[w][k][0] + m[1] * s.b[w][k][1] + m[2] * s.b[w][k][2];
                ar = fmaf(mk, acc.e1[b][k][0][i], ar);
                ai = fmaf(mk, acc.e1[b][k][1][i], ai);
            }
            float dr = -kap * ai, di = kap * ar;
            if constexpr (Q2) {
                const float q = -0.5f * (dx * dy) * (dx * dy) * mun;
                dr = fmaf(q, acc.e2[b][0][i], dr);
                di = fmaf(q, acc.e2[b][1][i], di);
            }
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                o.add(p, b * R + i, p ? di : dr);
                if (HAS_AMP) o.scale(p, b * R + i, aback);
            }
        }
    }
}
}  // namespace

// The single-shot forward: blockIdx.x a workgroup tile, blockIdx.y an emitter split.
template <class S, bool HAS_AMP>
__global__ __launch_bounds__(kBlock, S::kWaves) void k_fwd_sep(Geom g, const double* __restrict__ emit,
                                                               const double* __restrict__ amp, int64_t n, int tiles_y,
                                                               int64_t per_split, float4* __restrict__ partial,
                                                               void* out, int kind)
{
    __shared__ SepLds<S> s;
    const int tx0 = (blockIdx.x / tiles_y) * S::kRows, ty0 = (blockIdx.x % tiles_y) * S::kCols;
    const int64_t e0 = (int64_t)blockIdx.y * per_split;
    const int64_t e1 = (e0 + per_split < n) ? e0 + per_split : n;
    SepOut<S> o;
    sep_tile<S, HAS_AMP>(g, emit, amp, e0, e1, blockIdx.y, tx0, ty0, s, o);
    const Geom gs = item_geom();  // store frames formed here (see k_batched_pair)
    const size_t npix = (size_t)gs.n0 * gs.n1;
#pragma unroll S::kStoreUnroll
    for (int i = 0; i < S::NB * S::R; ++i) {
        int x, y;
        sep_pixel<S>(tx0, ty0, threadIdx.x >> 6, threadIdx.x & 63, i, x, y);
        if (x < gs.n0 && y < gs.n1) {
            const size_t idx = (size_t)x * gs.n1 + y;
            if (partial != nullptr) {
                const float2 re = o.parts(0, i), im = o.parts(1, i);
                partial[(size_t)blockIdx.y * npix + idx] = make_float4(re.x, im.x, re.y, im.y);
            } else {
                store_split(gs, x, y, o.value(0, i), o.value(1, i), out, kind, idx);
            }
        }
    }
}

// Persistent batched form (the queue protocol of k_batched_split).
template <class S, bool HAS_AMP>
__global__ __launch_bounds__(kBlock, S::kWaves) void k_batched_sep(Geom g0, const double* __restrict__ emit,
                                                                   const double* __restrict__ amp,
                                                                   const WorkItem* __restrict__ items, int nitems,
                                                                   int* __restrict__ counter, int tiles_y, void* out,
                                                                   int kind)
{
    __shared__ SepLds<S> s;
    __shared__ int s_item;
    const size_t npix = (size_t)g0.n0 * g0.n1;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_item = atomicAdd(counter, 1);
        __syncthreads();
        const int it = s_item;
        if (it >= nitems) break;
        const WorkItem wi = items[it];
        const Geom g = item_geom();
        const int tx0 = (wi.tile / tiles_y) * S::kRows, ty0 = (wi.tile % tiles_y) * S::kCols;
        SepOut<S> o;
        sep_tile<S, HAS_AMP>(g, emit, amp, wi.e0, wi.e1, 0, tx0, ty0, s, o);
        char* outs = static_cast<char*>(out) +
                     (size_t)wi.shot * npix * (kind == OUT_INTENSITY ? sizeof(float) : sizeof(float2));
        const Geom gs = item_geom();  // as in k_batched_pair
#pragma unroll S::kStoreUnroll
        for (int i = 0; i < S::NB * S::R; ++i) {
            int x, y;
            sep_pixel<S>(tx0, ty0, threadIdx.x >> 6, threadIdx.x & 63, i, x, y);
            if (x < gs.n0 && y < gs.n1)
                store_split(gs, x, y, o.value(0, i), o.value(1, i), outs, kind, (size_t)x * gs.n1 + y);
        }
    }
}

__global__ void k_sep_reset(int* counter) { *counter = 0; }

template <class S, bool A>
static hipError_t launch_sep_t(const Geom& g, const double* emit, const double* amp, int64_t n, int splits,
                               float4* partial, void* out, int kind, hipStream_t st)
{
    const int tiles_x = (g.n0 + S::kRows - 1) / S::kRows, tiles_y = (g.n1 + S::kCols - 1) / S::kCols;
    hipLaunchKernelGGL((k_fwd_sep<S, A>), dim3(tiles_x * tiles_y, splits), dim3(kBlock), 0, st, g, emit, amp, n,
                       tiles_y, split_size(n, splits), partial, out, kind);
    return hipGetLastError();
}

template <class S, bool A>
static hipError_t launch_batched_sep_t(const Geom& g, const double* emit, const double* amp, const WorkItem* items,
                                       int nitems, int* counter, int nblocks, void* out, int kind, hipStream_t st)
{
    hipLaunchKernelGGL(k_sep_reset, dim3(1), dim3(1), 0, st, counter);
    hipLaunchKernelGGL((k_batched_sep<S, A>), dim3(nblocks), dim3(kBlock), 0, st, g, emit, amp, items, nitems, counter,
                       (g.n1 + S::kCols - 1) / S::kCols, out, kind);
    return hipGetLastError();
}

template <class S, bool A>
static int occupancy_sep_t()
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_batched_sep<S, A>, kBlock, 0) != hipSuccess) return 1;
    return nb > 0 ? nb : 1;
}

using Sep32 = SepShape<32, 1, 2, false>;
using Sep32V = SepShape<32, 1, 3, false>;
using Sep32W = SepShape<32, 2, 2, false>;
using Sep32WV = SepShape<32, 2, 3, false>;
using Sep16 = SepShape<16, 1, 2, false>;
using Sep16Q = SepShape<16, 1, 3, true>;

#define IDISIM_DISPATCH_SEP(FN, ...)                                              \
    switch (v) {                                                                  \
        case kTileSep32: return a ? FN<Sep32, true>(__VA_ARGS__) : FN<Sep32, false>(__VA_ARGS__);       \
        case kTileSep32V: return a ? FN<Sep32V, true>(__VA_ARGS__) : FN<Sep32V, false>(__VA_ARGS__);    \
        case kTileSep32W: return a ? FN<Sep32W, true>(__VA_ARGS__) : FN<Sep32W, false>(__VA_ARGS__);    \
        case kTileSep32WV: return a ? FN<Sep32WV, true>(__VA_ARGS__) : FN<Sep32WV, false>(__VA_ARGS__); \
        case kTileSep16: return a ? FN<Sep16, true>(__VA_ARGS__) : FN<Sep16, false>(__VA_ARGS__);       \
        case kTileSep16Q: return a ? FN<Sep16Q, true>(__VA_ARGS__) : FN<Sep16Q, false>(__VA_ARGS__);    \
        default: break;                                                           \
    }

hipError_t launch_fwd_sep(int v, bool a, const Geom& g, const double* emit, const double* amp, int64_t n, int splits,
                          float4* partial, void* out, int kind, hipStream_t st)
{
    if (!(g.sepscale > 0.f) || (g.foldw == 0 && (g.nf || g.secondorder))) return hipErrorInvalidValue;
    IDISIM_DISPATCH_SEP(launch_sep_t, g, emit, amp, n, splits, partial, out, kind, st)
    return hipErrorInvalidValue;
}

hipError_t launch_batched_sep(int v, bool a, const Geom& g, const double* emit, const double* amp,
                              const WorkItem* items, int nitems, int* counter, int nblocks, void* out, int kind,
                              hipStream_t st)
{
    if (!(g.sepscale > 0.f) || (g.foldw == 0 && (g.nf || g.secondorder))) return hipErrorInvalidValue;
    IDISIM_DISPATCH_SEP(launch_batched_sep_t, g, emit, amp, items, nitems, counter, nblocks, out, kind, st)
    return hipErrorInvalidValue;
}

int occupancy_batched_sep(int v, bool a)
{
    IDISIM_DISPATCH_SEP(occupancy_sep_t)
    return 1;
}

}  // namespace idisim
