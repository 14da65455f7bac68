// Per-type stroke evaluation: the drop-in replacement for the reference's
// stroke_forward / stroke_backward (source/strokelib/src/strokes_forward.cu,
// strokes_backward.cu; bound in source/strokelib/strokes.py:167,217).
//
// Mapping: one lane per stroke, a wavefront covers 64 consecutive strokes and
// walks a block-private range of points.  The stroke's parameters and its
// rotation are loaded once per lane and kept in registers; the point (x,
// radius, view direction) is wave-uniform and broadcast.  Outputs
// alpha[N,S] / color[N,S,3] are written lane-contiguous.  The adjoint keeps the
// stroke's parameter gradients in registers across the whole point range, adds
// the block's wavefronts together in LDS and issues one atomic per parameter per
// stroke per block (blocks are few and long: about 1024 over all stroke tiles);
// dL/dx is summed across the wavefront before a single atomic per point.
#include "n3ds_capi.h"
#include "n3ds_stroke_common.h"

namespace n3ds {

constexpr int WAVES = 4;
constexpr int BLOCK = 64 * WAVES;

template <int BASE, int CID>
__global__ __launch_bounds__(BLOCK) void stroke_fwd_kernel(
    float* __restrict__ alpha_out, float* __restrict__ color_out, float* __restrict__ sdf_out,
    float* __restrict__ tex_out, const float* __restrict__ x, const float* __restrict__ radius,
    const float* __restrict__ viewdir, const float* __restrict__ sp, const float* __restrict__ cp, int64_t N,
    int64_t S, int64_t spr, int P, int Q, uint32_t flags, float delta, int laplace, int isr, int64_t ppb) {
    constexpr int NB = num_base_params(BASE);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    const int64_t k = (int64_t)blockIdx.y * 64 + lane;
    const bool kv = k < S;
    const int64_t kk = kv ? k : S - 1;
    const float* row = sp + kk * P;
    float prm[NB > 0 ? NB : 1];
#pragma unroll
    for (int i = 0; i < NB; i++) prm[i] = row[i];
    const float* crow = cp + kk * Q;
    float col[num_color_params(CID)];
#pragma unroll
    for (int i = 0; i < num_color_params(CID); i++) col[i] = crow[i];
    const Frame F = load_frame(row, P, flags);
    const int64_t n0 = (int64_t)blockIdx.x * ppb;
    const int64_t n1 = min(N, n0 + ppb);
    const float kscale = laplace ? 2.f : 0.5f;
    for (int64_t n = n0 + wave; n < n1; n += WAVES) {
        V3 xw = ld3(x + 3 * n);
        float r = radius[n];
        V3 dir = (CID >= 2) ? ld3(viewdir + 3 * (n / spr)) : v3s(0.f);
        V3 p = inverse_xform(xw, F, flags);
        float sdf = sdf_eval(BASE, p, prm);
        if (isr) {
            if (flags & F_SS) r = r / F.scale.x;
            else if (flags & F_MS) r = r / radius_factor(ref_dir(BASE, p, prm), F.scale);
        }
        float sc = kscale / (delta * r);
        float a = alpha_from_sdf(sdf, sc, delta, laplace);
        V3 c = color_eval_t<CID>(p, dir, col);
        if (kv) {
            int64_t o = n * S + k;
            alpha_out[o] = a;
            color_out[3 * o + 0] = c.x;
            color_out[3 * o + 1] = c.y;
            color_out[3 * o + 2] = c.z;
            if (sdf_out) sdf_out[o] = sdf;
            if (tex_out) {
                float u, v;
                texcoord_eval(BASE, p, row, (flags & F_MS) != 0, u, v);
                tex_out[2 * o + 0] = u;
                tex_out[2 * o + 1] = v;
            }
        }
    }
}

template <int BASE, int CID>
__global__ __launch_bounds__(BLOCK) void stroke_bwd_kernel(
    float* __restrict__ gshape, float* __restrict__ gcolor, float* __restrict__ gx,
    const float* __restrict__ galpha, const float* __restrict__ gcol_in, const float* __restrict__ gsdf,
    const float* __restrict__ x, const float* __restrict__ radius, const float* __restrict__ viewdir,
    const float* __restrict__ alpha, const float* __restrict__ sp, const float* __restrict__ cp, int64_t N,
    int64_t S, int64_t spr, int P, int Q, uint32_t flags, float delta, int laplace, int isr, int exact,
    int64_t ppb) {
    constexpr int NB = num_base_params(BASE);
    constexpr int NQ = num_color_params(CID);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    const int64_t k = (int64_t)blockIdx.y * 64 + lane;
    const bool kv = k < S;
    const int64_t kk = kv ? k : S - 1;
    const float* row = sp + kk * P;
    float prm[NB > 0 ? NB : 1];
#pragma unroll
    for (int i = 0; i < NB; i++) prm[i] = row[i];
    const float* crow = cp + kk * Q;
    float col[NQ];
#pragma unroll
    for (int i = 0; i < NQ; i++) col[i] = crow[i];
    const Frame F = load_frame(row, P, flags);
    float gb[NB > 0 ? NB : 1];
#pragma unroll
    for (int i = 0; i < (NB > 0 ? NB : 1); i++) gb[i] = 0.f;
    float gc[NQ];
#pragma unroll
    for (int i = 0; i < NQ; i++) gc[i] = 0.f;
    float gs1 = 0.f;
    V3 gs3 = v3s(0.f), gang = v3s(0.f), gtr = v3s(0.f);
    const int64_t n0 = (int64_t)blockIdx.x * ppb;
    const int64_t n1 = min(N, n0 + ppb);
    const float kscale = laplace ? 2.f : 0.5f;
    for (int64_t n = n0 + wave; n < n1; n += WAVES) {
        const int64_t o = n * S + kk;
        V3 xw = ld3(x + 3 * n);
        float r = radius[n];
        V3 dir = (CID >= 2) ? ld3(viewdir + 3 * (n / spr)) : v3s(0.f);
        V3 p = inverse_xform(xw, F, flags);
        float ga = kv ? galpha[o] : 0.f;
        V3 gcv = kv ? ld3(gcol_in + 3 * o) : v3s(0.f);
        float gsd = (kv && gsdf) ? gsdf[o] : 0.f;
        float fac = 1.f;
        if (isr) {
            if (flags & F_SS) r = r / F.scale.x;
            else if (flags & F_MS) { fac = radius_factor(ref_dir(BASE, p, prm), F.scale); r = r / fac; }
        }
        float sc = kscale / (delta * r);
        float sdf = 0.f;
        float a;
        if (exact) {
            sdf = sdf_eval(BASE, p, prm);
            a = alpha_from_sdf(sdf, sc, delta, laplace);
        } else {
            a = kv ? alpha[o] : 0.f;
        }
        float gsdf_tot = ga * dalpha_dsdf(sdf, a, sc, delta, laplace, exact) + gsd;
        V3 gp = color_grad_t<CID>(p, dir, col, gcv, gc, exact != 0);
        V3 dsdp;
        if (exact) dsdp = grad_ex(BASE, p, prm, gsdf_tot, gb);
        else dsdp = grad_ref(BASE, p, prm, gsdf_tot, gb);
        gp = gp + dsdp * gsdf_tot;
        if (exact && isr && (flags & (F_SS | F_MS))) {
            float gsc = ga * dalpha_dscale(sdf, a, sc, delta, laplace);
            if (flags & F_SS) {
                gs1 += gsc * sc / F.scale.x;
            } else {
                radius_factor_adjoint(BASE, p, prm, F.scale, gsc * sc / fac, gp, gs3, gb);
            }
        }
        V3 gxv = xform_adjoint(gp, p, xw, F, flags, gs1, gs3, gang, gtr);
        if (gx) {
            if (!kv) gxv = v3s(0.f);
            float sx = wave_sum(gxv.x), sy = wave_sum(gxv.y), sz = wave_sum(gxv.z);
            if (lane == 0) {
                atomicAdd(gx + 3 * n + 0, sx);
                atomicAdd(gx + 3 * n + 1, sy);
                atomicAdd(gx + 3 * n + 2, sz);
            }
        }
    }
    // the block's wavefronts hold partial sums for the same 64 strokes: add them in LDS,
    // then the first wavefront issues one global atomic per parameter per stroke
    constexpr int NR = (NB > 0 ? NB : 1) + 10 + NQ;
    __shared__ float red[NR * 64];
    for (int i = threadIdx.x; i < NR * 64; i += BLOCK) red[i] = 0.f;
    __syncthreads();
    {
        float v[NR];
#pragma unroll
        for (int i = 0; i < (NB > 0 ? NB : 1); i++) v[i] = NB > 0 ? gb[i] : 0.f;
        constexpr int o = NB > 0 ? NB : 1;
        v[o] = gs1;
        v[o + 1] = gs3.x; v[o + 2] = gs3.y; v[o + 3] = gs3.z;
        v[o + 4] = gang.x; v[o + 5] = gang.y; v[o + 6] = gang.z;
        v[o + 7] = gtr.x; v[o + 8] = gtr.y; v[o + 9] = gtr.z;
#pragma unroll
        for (int i = 0; i < NQ; i++) v[o + 10 + i] = gc[i];
#pragma unroll
        for (int i = 0; i < NR; i++) atomicAdd(&red[i * 64 + lane], v[i]);
    }
    __syncthreads();
    if (wave != 0 || !kv) return;
    const float* r = red + lane;
    constexpr int o = NB > 0 ? NB : 1;
    float* grow = gshape + k * P;
#pragma unroll
    for (int i = 0; i < NB; i++) atomicAdd(grow + i, r[i * 64]);
    if (F.off_scale >= 0) {
        if (flags & F_SS) atomicAdd(grow + F.off_scale, r[o * 64]);
        else for (int i = 0; i < 3; i++) atomicAdd(grow + F.off_scale + i, r[(o + 1 + i) * 64]);
    }
    if (F.off_angle >= 0)
        for (int i = 0; i < 3; i++) atomicAdd(grow + F.off_angle + i, r[(o + 4 + i) * 64]);
    if (F.off_trans >= 0)
        for (int i = 0; i < 3; i++) atomicAdd(grow + F.off_trans + i, r[(o + 7 + i) * 64]);
    float* gcrow = gcolor + k * Q;
#pragma unroll
    for (int i = 0; i < NQ; i++) atomicAdd(gcrow + i, r[(o + 10 + i) * 64]);
}

// ---------------------------------------------------------------------------
// Linear transfer: an SDF only matters where alpha lies strictly inside its range
// ---------------------------------------------------------------------------

// LDS ordering between the lanes of one wavefront
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// appends the lanes with `on` to a wavefront's queue of qn entries; returns the new length
template <typename T>
__device__ __forceinline__ int queue_push(T* q, int qn, bool on, T e) {
    const unsigned long long m = __ballot(on);
    if (on)
        q[qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0))] = e;
    return qn + __popcll(m);
}

// Forward of curves.  A curve lies in the box of its Bezier control points, so a point
// further from the box than the largest radius plus delta * radius has alpha = 0 exactly:
// one box test per pair (about 13 operations against some 300 of the closest-point search)
// leaves a tenth of the pairs, which are queued and searched in full wavefronts.  The
// lane-per-stroke kernel above searches all 64 strokes as soon as one of them is near:
// 224 us at 65536 points x 500 cubic curves, bound by its arithmetic; this one is bound by
// the 16 bytes written per pair.
constexpr int CURVE_PTS = 16;  // points a wavefront holds at a time

template <int BASE, int CID>
__global__ __launch_bounds__(BLOCK) void stroke_fwd_curve_kernel(
    float* __restrict__ alpha_out, float* __restrict__ color_out, float* __restrict__ tex_out,
    const float* __restrict__ x, const float* __restrict__ radius, const float* __restrict__ viewdir,
    const float* __restrict__ sp, const float* __restrict__ cp, int64_t N, int64_t S, int64_t spr, float delta,
    int64_t ppb) {
    constexpr int NB = num_base_params(BASE), NC = BASE == QUAD_BEZIER ? 3 : 4;
    __shared__ float sprm[64][NB + 1 - NB % 2];
    __shared__ float sal[WAVES][CURVE_PTS][64];
    __shared__ uint32_t sq[WAVES][128];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    const int64_t k0 = (int64_t)blockIdx.y * 64, k = k0 + lane;
    const bool kv = k < S;
    for (int i = threadIdx.x; i < 64 * NB; i += BLOCK) {
        const int l = i / NB, c = i - l * NB;
        sprm[l][c] = sp[min(k0 + l, S - 1) * NB + c];
    }
    __syncthreads();
    const float* prm = sprm[lane];
    float col[num_color_params(CID)];
#pragma unroll
    for (int i = 0; i < num_color_params(CID); i++) col[i] = cp[min(k, S - 1) * num_color_params(CID) + i];
    // box of the control points (a Catmull-Rom segment's Bezier points from its coefficients)
    V3 K[4];
    if (BASE == CATMULL_ROM) {
        const CatmullCoef cc = catmull_coef(prm);
        K[0] = cc.K[3];
        K[1] = cc.K[3] + cc.K[2] * (1.f / 3.f);
        K[2] = cc.K[3] + cc.K[2] * (2.f / 3.f) + cc.K[1] * (1.f / 3.f);
        K[3] = cc.K[0] + cc.K[1] + cc.K[2] + cc.K[3];
    } else {
#pragma unroll
        for (int i = 0; i < NC; i++) K[i] = ld3(prm + 3 * i);
        if (NC == 3) K[3] = K[2];
    }
    V3 lo = K[0], hi = K[0];
#pragma unroll
    for (int i = 1; i < 4; i++) {
        lo = v3(fminf(lo.x, K[i].x), fminf(lo.y, K[i].y), fminf(lo.z, K[i].z));
        hi = v3(fmaxf(hi.x, K[i].x), fmaxf(hi.y, K[i].y), fmaxf(hi.z, K[i].z));
    }
    const V3 c = (lo + hi) * 0.5f;
    // half extents and reach, padded far beyond the rounding of the test
    const float pad = 1e-5f * (1.f + fmaxf(fabsf(c.x), fmaxf(fabsf(c.y), fabsf(c.z))));
    const V3 h = (hi - lo) * 0.50001f + v3s(pad);
    const float reach = fmaxf(prm[NB - 2], prm[NB - 1]);
    float zero = 0.f * (c.x + c.y + c.z + h.x + h.y + h.z);  // (min and max pass NaN over)
#pragma unroll
    for (int i = 0; i < NB; i++) zero += 0.f * prm[i];
    const bool odd = !(zero == 0.f);  // an infinite or NaN parameter: every pair is searched
    const int64_t n0 = (int64_t)blockIdx.x * ppb, n1 = min(N, n0 + ppb);
    uint32_t* q = sq[wave];
    for (int64_t nb = n0 + wave * CURVE_PTS; nb < n1; nb += WAVES * CURVE_PTS) {
        const int np = (int)min((int64_t)CURVE_PTS, n1 - nb);
        int qn = 0;
        auto search = [&](int i) {  // queue entry i of this lane
            const uint32_t e = q[i];
            const int s = e & 63, p = e >> 6;
            const float r = radius[nb + p];
            const float sdf = sdf_eval(BASE, ld3(x + 3 * (nb + p)), sprm[s]);
            sal[wave][p][s] = alpha_from_sdf(sdf, 0.5f / (delta * r), delta, false);
        };
        for (int p = 0; p < np; p++) {
            const V3 xp = ld3(x + 3 * (nb + p));
            const V3 d = vmax0(vabs(xp - c) - h);
            const float r = radius[nb + p];
            const float m = (reach + delta * r) * 1.0001f + pad;
            // (a finite point; with a radius that is not positive, alpha may be one far away)
            const bool far = dot(d, d) > m * m && 0.f * (xp.x + xp.y + xp.z) == 0.f && r > 0.f;
            const bool near = odd || !far;
            sal[wave][p][lane] = 0.f;
            qn = queue_push(q, qn, near && kv, (uint32_t)(p << 6 | lane));
            if (qn >= 64) {
                wave_fence();
                qn -= 64;
                search(qn + lane);
                wave_fence();
            }
        }
        wave_fence();
        if (lane < qn) search(lane);
        wave_fence();
        for (int p = 0; p < np; p++) {
            const int64_t n = nb + p, o = n * S + k;
            const V3 dir = (CID >= 2) ? ld3(viewdir + 3 * (n / spr)) : v3s(0.f);
            const V3 cv = color_eval_t<CID>(CID == 1 ? ld3(x + 3 * n) : v3s(0.f), dir, col);
            if (kv) {
                alpha_out[o] = sal[wave][p][lane];
                color_out[3 * o + 0] = cv.x;
                color_out[3 * o + 1] = cv.y;
                color_out[3 * o + 2] = cv.z;
                if (tex_out) {  // curves have no texture coordinates
                    tex_out[2 * o + 0] = 0.f;
                    tex_out[2 * o + 1] = 0.f;
                }
            }
        }
        wave_fence();
    }
}

// Adjoint by live pairs.  Without a gradient of the SDF itself and with a colour that does
// not depend on the position, only pairs with 0 < alpha < 0.9999 (the saved alpha) reach
// the SDF: a hundredth of them.  Every pair's upstream is read once, lane per stroke, for
// the colour sums; the live ones are queued and differentiated in full wavefronts, their
// strokes' frames read from LDS, and summed per stroke in LDS as doubles (64-bit LDS float
// atomics run 6 times as fast as 32-bit ones on this card).  What is not finite in a
// stroke, a point or an upstream gradient reaches the gradients through any pair, as a
// product with zero is then NaN: such a stroke's or point's pairs are all differentiated.
// Looking for them once per block costs 1 us.  The lane-per-stroke kernel above runs the
// SDF's adjoint for 64 strokes as soon as one is live: 791 us at 65536 points x 500 cubic
// curves and 547 us at 262144 x 200 boxes; this one is bound by the 20 bytes read per pair.
constexpr int LWAVES = 8;
constexpr int LUNROLL = 4;  // points in flight per wavefront

template <int BASE, int CID>
__global__ __launch_bounds__(64 * LWAVES) __attribute__((amdgpu_waves_per_eu(4, 8))) void stroke_bwd_live_kernel(
    float* __restrict__ gshape, float* __restrict__ gcolor, float* __restrict__ gx, const float* __restrict__ galpha,
    const float* __restrict__ gcol_in, const float* __restrict__ x, const float* __restrict__ radius,
    const float* __restrict__ viewdir, const float* __restrict__ alpha, const float* __restrict__ sp,
    const float* __restrict__ cp, int64_t N, int64_t S, int64_t spr, int P, int Q, uint32_t flags, float delta, int isr,
    int exact, int64_t ppb) {
    constexpr int NB = num_base_params(BASE), NQ = num_color_params(CID);
    constexpr int NF = (is_curve(BASE) ? 0 : 17) + NB;  // rotation, translation, scale, sz, cz; base parameters
    constexpr int NR = (is_curve(BASE) ? 0 : 10) + NB;  // scale, scales, angles, translation; base parameters
    constexpr int FO = is_curve(BASE) ? 0 : 17, RO = is_curve(BASE) ? 0 : 10;
    __shared__ float frame[64][NF + 1 - NF % 2];
    __shared__ double acc[NR][64];
    __shared__ double csum[NQ][64];
    __shared__ int odd_stroke[64];
    __shared__ uint2 sq[LWAVES][128];  // point of the block << 6 | lane, dL/dalpha
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    const int64_t k = (int64_t)blockIdx.y * 64 + lane;
    const bool kv = k < S;
    const int64_t kk = kv ? k : S - 1;
    const int64_t n0 = (int64_t)blockIdx.x * ppb, n1 = min(N, n0 + ppb);
    bool bad = false;
    if (wave == 0) {
        const float* row = sp + kk * P;
        float zero = 0.f;  // NaN with a parameter that is not finite
        if (!is_curve(BASE)) {
            const Frame F = load_frame(row, P, flags);
#pragma unroll
            for (int i = 0; i < 9; i++) frame[lane][i] = (flags & F_R) ? F.R.r[i / 3][i % 3] : 0.f;
            frame[lane][9] = F.trans.x; frame[lane][10] = F.trans.y; frame[lane][11] = F.trans.z;
            frame[lane][12] = F.scale.x; frame[lane][13] = F.scale.y; frame[lane][14] = F.scale.z;
            frame[lane][15] = F.sz; frame[lane][16] = F.cz;
            // (a point is divided by the scale)
            zero = 0.f * (F.trans.x + F.trans.y + F.trans.z + F.scale.x + F.scale.y + F.scale.z) +
                   0.f * (F.angle.x + F.angle.y + F.angle.z) + (0.f / F.scale.x + 0.f / F.scale.y + 0.f / F.scale.z);
        }
#pragma unroll
        for (int i = 0; i < NB; i++) {
            frame[lane][FO + i] = row[i];
            zero += 0.f * row[i];
        }
        odd_stroke[lane] = !(zero == 0.f);
    } else {
        // (a radius of 0: the adjoint of the radius scale is infinite)
        float zero = 0.f, least = INFINITY;
        for (int64_t n = n0 + threadIdx.x - 64; n < n1; n += 64 * (LWAVES - 1)) {
            const V3 xp = ld3(x + 3 * n);
            const float r = radius[n];
            zero += 0.f * (xp.x + xp.y + xp.z + r);
            least = fminf(least, fabsf(r));
        }
        bad = !(zero == 0.f && least > 0.f);
    }
    for (int i = threadIdx.x; i < NR * 64; i += 64 * LWAVES) (&acc[0][0])[i] = 0.0;
    for (int i = threadIdx.x; i < NQ * 64; i += 64 * LWAVES) (&csum[0][0])[i] = 0.0;
    float col[NQ], gc[NQ];
#pragma unroll
    for (int i = 0; i < NQ; i++) {
        col[i] = cp[kk * Q + i];
        gc[i] = 0.f;
    }
    const bool odd_points = __syncthreads_or(bad) != 0;  // some of the block's
    const bool odd = odd_stroke[lane] != 0;
    uint2* q = sq[wave];
    int qn = 0;
    auto adjoint = [&](int i) {  // queue entry i of this lane
        const uint2 e = q[i];
        const int s = e.x & 63;
        const int64_t n = n0 + (e.x >> 6);
        const float ga = __uint_as_float(e.y);
        const V3 xw = ld3(x + 3 * n);
        float r = radius[n];
        const float* fr = frame[s];
        Frame F;
        if (!is_curve(BASE)) {
#pragma unroll
            for (int j = 0; j < 9; j++) F.R.r[j / 3][j % 3] = fr[j];
            F.trans = ld3(fr + 9);
            F.scale = ld3(fr + 12);
            F.sz = fr[15];
            F.cz = fr[16];
        }
        float prm[NB > 0 ? NB : 1], gb[NB > 0 ? NB : 1];
#pragma unroll
        for (int j = 0; j < NB; j++) {
            prm[j] = fr[FO + j];
            gb[j] = 0.f;
        }
        const V3 p = is_curve(BASE) ? xw : inverse_xform(xw, F, flags);
        float fac = 1.f;
        if (!is_curve(BASE) && isr) {
            if (flags & F_SS) r = r / F.scale.x;
            else if (flags & F_MS) { fac = radius_factor(ref_dir(BASE, p, prm), F.scale); r = r / fac; }
        }
        const float sc = 0.5f / (delta * r);
        float sdf = 0.f, a;
        if (exact) {
            sdf = sdf_eval(BASE, p, prm);
            a = alpha_from_sdf(sdf, sc, delta, false);
        } else {
            a = alpha[n * S + (int64_t)blockIdx.y * 64 + s];
        }
        const float gsdf = ga * dalpha_dsdf(sdf, a, sc, delta, false, exact);
        const V3 dsdp = exact ? grad_ex(BASE, p, prm, gsdf, gb) : grad_ref(BASE, p, prm, gsdf, gb);
        V3 gp = dsdp * gsdf;
        float gs1 = 0.f;
        V3 gs3 = v3s(0.f), gang = v3s(0.f), gtr = v3s(0.f), gxv = gp;
        if (!is_curve(BASE)) {
            if (exact && isr && (flags & (F_SS | F_MS))) {
                const float gsc = ga * dalpha_dscale(sdf, a, sc, delta, false);
                if (flags & F_SS) gs1 += gsc * sc / F.scale.x;
                else radius_factor_adjoint(BASE, p, prm, F.scale, gsc * sc / fac, gp, gs3, gb);
            }
            gxv = xform_adjoint(gp, p, xw, F, flags, gs1, gs3, gang, gtr);
            const float v[10] = {gs1, gs3.x, gs3.y, gs3.z, gang.x, gang.y, gang.z, gtr.x, gtr.y, gtr.z};
#pragma unroll
            for (int j = 0; j < 10; j++)
                if (v[j] != 0.f) atomicAdd(&acc[j][s], (double)v[j]);
        }
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (gb[j] != 0.f) atomicAdd(&acc[RO + j][s], (double)gb[j]);
        if (gx) {
            // a point's entries lie side by side: summed by their first lane, one atomic a run
            // (one a pair took 3360 us at 65536 points x 200 curves with every pair live)
            const int np = __popcll(__ballot(true));  // lanes 0..np - 1 are here
            const uint32_t pt = e.x >> 6, before = __shfl_up(pt, 1, 64);
            const bool head = lane == 0 || before != pt;
            const unsigned long long after = __ballot(head) & ~((2ull << lane) - 1ull);
            const int end = after ? __builtin_ctzll(after) : np;
            for (int off = 1; off < 64; off <<= 1) {
                const bool in = lane + off < end;
                if (__ballot(in) == 0ull) break;
                const float ux = __shfl_down(gxv.x, off, 64), uy = __shfl_down(gxv.y, off, 64),
                            uz = __shfl_down(gxv.z, off, 64);
                if (in) gxv = gxv + v3(ux, uy, uz);
            }
            if (head) {
                atomicAdd(gx + 3 * n + 0, gxv.x);
                atomicAdd(gx + 3 * n + 1, gxv.y);
                atomicAdd(gx + 3 * n + 2, gxv.z);
            }
        }
    };
    for (int64_t nb = n0 + wave * LUNROLL; nb < n1; nb += LWAVES * LUNROLL) {
        float ga[LUNROLL], al[LUNROLL];
        V3 gcv[LUNROLL];
#pragma unroll
        for (int u = 0; u < LUNROLL; u++) {
            const int64_t o = (nb + u) * S + kk;
            const bool on = kv && nb + u < n1;
            ga[u] = on ? galpha[o] : 0.f;
            al[u] = on ? alpha[o] : 0.f;
            gcv[u] = on ? ld3(gcol_in + 3 * o) : v3s(0.f);
        }
#pragma unroll
        for (int u = 0; u < LUNROLL; u++) {
            if (nb + u >= n1) break;
            const V3 dir = (CID >= 2) ? ld3(viewdir + 3 * ((nb + u) / spr)) : v3s(0.f);
            color_grad_t<CID>(v3s(0.f), dir, col, gcv[u], gc, exact != 0);
            bool live = (0.f < al[u] && al[u] < 0.9999f) || !isfinite(ga[u]) || odd;
            if (odd_points) {
                const V3 xp = ld3(x + 3 * (nb + u));
                const float r = radius[nb + u];
                live = live || !(0.f * (xp.x + xp.y + xp.z + r) == 0.f) || r == 0.f;
            }
            live = live && kv;
            if (__ballot(live) == 0ull) continue;
            qn = queue_push(q, qn, live, make_uint2((uint32_t)((nb + u - n0) << 6 | lane), __float_as_uint(ga[u])));
            if (qn >= 64) {
                wave_fence();
                qn -= 64;
                adjoint(qn + lane);
                wave_fence();
            }
        }
    }
    wave_fence();
    if (lane < qn) adjoint(lane);
#pragma unroll
    for (int i = 0; i < NQ; i++) atomicAdd(&csum[i][lane], (double)gc[i]);
    __syncthreads();
    if (wave != 0 || !kv) return;
    float* grow = gshape + k * P;
    auto add = [&](float* to, double v) {
        if (v != 0.0) atomicAdd(to, (float)v);
    };
#pragma unroll
    for (int i = 0; i < NB; i++) add(grow + i, acc[RO + i][lane]);
    if (!is_curve(BASE)) {
        int end = P;
        if (flags & F_T) {
            end -= 3;
            for (int i = 0; i < 3; i++) add(grow + end + i, acc[7 + i][lane]);
        }
        if (flags & F_R) {
            end -= 3;
            for (int i = 0; i < 3; i++) add(grow + end + i, acc[4 + i][lane]);
        }
        if (flags & F_SS) add(grow + end - 1, acc[0][lane]);
        else if (flags & F_MS)
            for (int i = 0; i < 3; i++) add(grow + end - 3 + i, acc[1 + i][lane]);
    }
    float* gcrow = gcolor + k * Q;
#pragma unroll
    for (int i = 0; i < NQ; i++) atomicAdd(gcrow + i, (float)csum[i][lane]);
}

typedef void (*CurveFn)(float*, float*, float*, const float*, const float*, const float*, const float*, const float*,
                        int64_t, int64_t, int64_t, float, int64_t);
typedef void (*LiveFn)(float*, float*, float*, const float*, const float*, const float*, const float*, const float*,
                       const float*, const float*, const float*, int64_t, int64_t, int64_t, int, int, uint32_t, float,
                       int, int, int64_t);
#define N3DS_CURVE(B) \
    {stroke_fwd_curve_kernel<B, 0>, stroke_fwd_curve_kernel<B, 1>, stroke_fwd_curve_kernel<B, 2>, \
     stroke_fwd_curve_kernel<B, 3>}
static const CurveFn kCurve[3][4] = {N3DS_CURVE(9), N3DS_CURVE(10), N3DS_CURVE(11)};
#define N3DS_LIVE(B) \
    {stroke_bwd_live_kernel<B, 0>, nullptr, stroke_bwd_live_kernel<B, 2>, stroke_bwd_live_kernel<B, 3>}
static const LiveFn kLive[NUM_BASE][4] = {N3DS_LIVE(0), N3DS_LIVE(1), N3DS_LIVE(2), N3DS_LIVE(3), N3DS_LIVE(4), N3DS_LIVE(5),
                                          N3DS_LIVE(6), N3DS_LIVE(7), N3DS_LIVE(8), N3DS_LIVE(9), N3DS_LIVE(10), N3DS_LIVE(11)};

typedef void (*FwdFn)(float*, float*, float*, float*, const float*, const float*, const float*, const float*,
                      const float*, int64_t, int64_t, int64_t, int, int, uint32_t, float, int, int, int64_t);
typedef void (*BwdFn)(float*, float*, float*, const float*, const float*, const float*, const float*,
                      const float*, const float*, const float*, const float*, const float*, int64_t, int64_t,
                      int64_t, int, int, uint32_t, float, int, int, int, int64_t);

template <int B, int C>
struct Tab {
    static constexpr FwdFn f = &stroke_fwd_kernel<B, C>;
    static constexpr BwdFn b = &stroke_bwd_kernel<B, C>;
};

#define N3DS_ROW(B) {Tab<B, 0>::f, Tab<B, 1>::f, Tab<B, 2>::f, Tab<B, 3>::f}
#define N3DS_ROWB(B) {Tab<B, 0>::b, Tab<B, 1>::b, Tab<B, 2>::b, Tab<B, 3>::b}
static const FwdFn kFwd[NUM_BASE][4] = {N3DS_ROW(0), N3DS_ROW(1), N3DS_ROW(2), N3DS_ROW(3), N3DS_ROW(4), N3DS_ROW(5),
                                        N3DS_ROW(6), N3DS_ROW(7), N3DS_ROW(8), N3DS_ROW(9), N3DS_ROW(10), N3DS_ROW(11)};
static const BwdFn kBwd[NUM_BASE][4] = {N3DS_ROWB(0), N3DS_ROWB(1), N3DS_ROWB(2), N3DS_ROWB(3), N3DS_ROWB(4), N3DS_ROWB(5),
                                        N3DS_ROWB(6), N3DS_ROWB(7), N3DS_ROWB(8), N3DS_ROWB(9), N3DS_ROWB(10), N3DS_ROWB(11)};

// points per block for about target_blocks blocks over the stroke tiles (the adjoint
// uses fewer, longer blocks: each block ends with an atomic per stroke parameter)
static int64_t points_per_block(int64_t N, int64_t S, int64_t target_blocks = 4096) {
    int64_t tiles = (S + 63) / 64;
    int64_t ppb = (N * tiles + target_blocks - 1) / target_blocks;
    ppb = ppb < 64 ? 64 : (ppb > 16384 ? 16384 : ppb);
    return ((ppb + WAVES - 1) / WAVES) * WAVES;
}

static int check_common(int64_t N, int64_t R, int64_t S, int64_t P, int64_t Q, uint32_t sdf_id, uint32_t color_id) {
    N3DS_REQUIRE(N >= 0 && S >= 0 && R >= 0, "negative size");
    N3DS_REQUIRE((sdf_id >> 4) < (uint32_t)NUM_BASE, "sdf_id %u out of range", sdf_id);
    N3DS_REQUIRE(color_id < 4u, "color_id %u out of range", color_id);
    N3DS_REQUIRE(P == num_shape_params(sdf_id), "shape_params has %lld columns, sdf_id %u needs %d", (long long)P,
                 sdf_id, num_shape_params(sdf_id));
    N3DS_REQUIRE(Q == num_color_params((int)color_id), "color_params has %lld columns, color_id %u needs %d",
                 (long long)Q, color_id, num_color_params((int)color_id));
    N3DS_REQUIRE(N == 0 || (R > 0 && N % R == 0), "n_points (%lld) must be a multiple of n_viewdirs (%lld)",
                 (long long)N, (long long)R);
    N3DS_REQUIRE((uint32_t)((sdf_id & F_SS) != 0) + (uint32_t)((sdf_id & F_MS) != 0) <= 1u,
                 "sdf_id %u sets both single and multi scale", sdf_id);
    return N3DS_OK;
}

}  // namespace n3ds

using namespace n3ds;

N3DS_EXPORT int n3ds_stroke_forward(float* alpha_out, float* color_out, float* sdf_out, float* texcoord_out,
                                    const float* x, const float* radius, const float* viewdir,
                                    const float* shape_params, const float* color_params, int64_t n_points,
                                    int64_t n_viewdirs, int64_t n_strokes, int64_t n_shape_params,
                                    int64_t n_color_params, uint32_t sdf_id, uint32_t color_id, float sdf_delta,
                                    int use_laplace_transform, int inv_scale_radius, void* stream) {
    int st = check_common(n_points, n_viewdirs, n_strokes, n_shape_params, n_color_params, sdf_id, color_id);
    if (st) return st;
    if (n_points == 0 || n_strokes == 0) return N3DS_OK;
    int64_t ppb = points_per_block(n_points, n_strokes);
    dim3 grid((unsigned)((n_points + ppb - 1) / ppb), (unsigned)((n_strokes + 63) / 64));
    // curves with the linear transfer, when only alpha is asked for: pairs out of reach skip
    // the closest-point search (the Laplace tail and the SDF itself reach everywhere)
    if (is_curve((int)(sdf_id >> 4)) && !use_laplace_transform && sdf_delta > 0.f && !sdf_out && (sdf_id & 15u) == 0) {
        hipLaunchKernelGGL(kCurve[(sdf_id >> 4) - QUAD_BEZIER][color_id], grid, dim3(BLOCK), 0, (hipStream_t)stream,
                           alpha_out, color_out, texcoord_out, x, radius, viewdir, shape_params, color_params,
                           n_points, n_strokes, n_points / n_viewdirs, sdf_delta, ppb);
        N3DS_LAUNCH_CHECK();
        return N3DS_OK;
    }
    hipLaunchKernelGGL(kFwd[sdf_id >> 4][color_id], grid, dim3(BLOCK), 0, (hipStream_t)stream, alpha_out, color_out,
                       sdf_out, texcoord_out, x, radius, viewdir, shape_params, color_params, n_points, n_strokes,
                       n_points / n_viewdirs, (int)n_shape_params, (int)n_color_params, sdf_id & 15u, sdf_delta,
                       use_laplace_transform, inv_scale_radius, ppb);
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}

N3DS_EXPORT int n3ds_stroke_backward(float* grad_shape_params, float* grad_color_params, float* grad_x,
                                     const float* grad_alpha, const float* grad_color, const float* grad_sdf,
                                     const float* x, const float* radius, const float* viewdir, const float* alpha,
                                     const float* shape_params, const float* color_params, int64_t n_points,
                                     int64_t n_viewdirs, int64_t n_strokes, int64_t n_shape_params,
                                     int64_t n_color_params, uint32_t sdf_id, uint32_t color_id, float sdf_delta,
                                     int use_laplace_transform, int inv_scale_radius, int adjoint_exact,
                                     void* stream) {
    int st = check_common(n_points, n_viewdirs, n_strokes, n_shape_params, n_color_params, sdf_id, color_id);
    if (st) return st;
    if (n_points == 0 || n_strokes == 0) return N3DS_OK;
    // the linear transfer by live pairs, unless the SDF has a gradient of its own or the
    // colour depends on the position (gradient_rgb): then every pair has an SDF adjoint.  The
    // reference's quadratic adjoint stays on the general path: near a double root its terms
    // grow to 1e6 and amplify the rounding of whichever kernel forms them to a per cent.
    if (!use_laplace_transform && sdf_delta > 0.f && !grad_sdf && alpha && color_id != 1 &&
        !(is_curve((int)(sdf_id >> 4)) && (sdf_id & 15u)) && (adjoint_exact || (sdf_id >> 4) != QUAD_BEZIER)) {
        const int64_t tiles = (n_strokes + 63) / 64;
        int64_t per = (n_points * tiles + 1023) / 1024;  // 4 blocks per CU, two at a time
        per = per < 64 ? 64 : (per > 32768 ? 32768 : per);
        per = (per + LWAVES * LUNROLL - 1) / (LWAVES * LUNROLL) * (LWAVES * LUNROLL);
        hipLaunchKernelGGL(kLive[sdf_id >> 4][color_id], dim3((unsigned)((n_points + per - 1) / per), (unsigned)tiles),
                           dim3(64 * LWAVES), 0, (hipStream_t)stream, grad_shape_params, grad_color_params, grad_x,
                           grad_alpha, grad_color, x, radius, viewdir, alpha, shape_params, color_params, n_points,
                           n_strokes, n_points / n_viewdirs, (int)n_shape_params, (int)n_color_params, sdf_id & 15u,
                           sdf_delta, inv_scale_radius, adjoint_exact, per);
        N3DS_LAUNCH_CHECK();
        return N3DS_OK;
    }
    int64_t ppb = points_per_block(n_points, n_strokes, 1024);
    dim3 grid((unsigned)((n_points + ppb - 1) / ppb), (unsigned)((n_strokes + 63) / 64));
    hipLaunchKernelGGL(kBwd[sdf_id >> 4][color_id], grid, dim3(BLOCK), 0, (hipStream_t)stream, grad_shape_params,
                       grad_color_params, grad_x, grad_alpha, grad_color, grad_sdf, x, radius, viewdir, alpha,
                       shape_params, color_params, n_points, n_strokes, n_points / n_viewdirs, (int)n_shape_params,
                       (int)n_color_params, sdf_id & 15u, sdf_delta, use_laplace_transform, inv_scale_radius,
                       adjoint_exact, ppb);
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}
