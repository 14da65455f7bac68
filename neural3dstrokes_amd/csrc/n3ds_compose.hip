// Ordered "over" compositing of strokes: drop-in replacement for the reference's
// compose_forward / compose_backward (source/strokelib/src/compositing.cu:9-157,
// bound in source/strokelib/strokes.py:339,368).
//
// Mapping: one wavefront per point, lanes over strokes in compositing order
// (stroke S-1 first).  "Over" is associative, so transmittance is an
// exclusive product scan across the wavefront and the adjoint's "composite of
// everything behind stroke k" is an affine suffix scan
//     U_k = d_k a_k + (1 - a_k) U_{k+1}
// evaluated with 64-lane shuffles.  The exact adjoint therefore needs neither
// the reference's suffix-by-subtraction nor its division by (1 - a_k):
//     dD/da_k = T_k (d_k - U_{k+1}),
//     dO/da_k = T_k R_{k+1}   with R_{k+1} = prod_{j behind k} (1 - a_j).
// The reference adjoint (compositing.cu:143-155) is kept as a mode.
//
// Nearly every (point, stroke) pair has alpha = 0 (99.9 % of the pairs of a 500-stroke
// scene), so a chunk of 64 strokes is first looked at through its alphas alone: without
// a nonzero one it leaves the transmittance and the sums as they are, the forward reads
// none of its colours and the adjoint needs no scan for it.  Both are then bound by
// memory: the forward reads 4 bytes per pair instead of 16, the adjoint moves its 36.
#include "n3ds_capi.h"
#include "n3ds_math.h"

namespace n3ds {

constexpr int CWAVES = 4;
constexpr int MAXCH = 128;          // transmittance checkpoints kept per point in the adjoint
constexpr int LDS_GDP_MAX = 8192;   // strokes whose density gradients a block sums in LDS

// LDS ordering between the lanes of one wavefront
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float scan_prod_excl(float f, int lane) {
    float v = f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        float o = __shfl_up(v, off, 64);
        if (lane >= off) v *= o;
    }
    float e = __shfl_up(v, 1, 64);
    return lane == 0 ? 1.f : e;
}

// Front to back over one point's strokes: returns the final transmittance, sums the colours
// into out[0..D) and the density into out[D]; t_in (or nullptr) receives the transmittance
// entering every G-th chunk of 64 strokes.
template <int D>
__device__ __forceinline__ float compose_front(const float* __restrict__ arow, const float* __restrict__ crow,
                                               const float* __restrict__ dp, int64_t S, int lane, float* t_in, int G,
                                               float* out) {
    constexpr int U = 4;  // chunks whose alphas are in flight together
    float T = 1.f, sum[D + 1];
#pragma unroll
    for (int c = 0; c <= D; c++) sum[c] = 0.f;
    for (int64_t base = 0; base < S; base += 64 * U) {
        float av[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t k = S - 1 - (base + 64 * u + lane);
            av[u] = k >= 0 ? arow[k] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t k = S - 1 - (base + 64 * u + lane);
            const int64_t ch = base / 64 + u;
            if (ch * 64 >= S) break;
            if (t_in && lane == 0 && ch % G == 0) t_in[ch / G] = T;
            const float a = av[u];
            if (__ballot(a != 0.f) == 0ull) continue;
            const float f = 1.f - a;
            const float Tk = T * scan_prod_excl(f, lane);
            if (a != 0.f) {
                const float w = a * Tk;
                sum[D] += dp[k] * w;
#pragma unroll
                for (int c = 0; c < D; c++) sum[c] += crow[k * D + c] * w;
            }
            T = __shfl(Tk * f, 63, 64);
        }
    }
#pragma unroll
    for (int c = 0; c <= D; c++) out[c] = wave_sum_halves(sum[c]);  // (wave_sum: adjoint 2 % slower)
    return T;
}

template <int D>
__global__ __launch_bounds__(64 * CWAVES) void compose_fwd_kernel(float* __restrict__ dens_out,
                                                               float* __restrict__ color_out,
                                                               const float* __restrict__ alphas,
                                                               const float* __restrict__ colors,
                                                               const float* __restrict__ dp, int64_t N, int64_t S,
                                                               int64_t ppb) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    const int64_t n0 = (int64_t)blockIdx.x * ppb, n1 = min(N, n0 + ppb);
    for (int64_t n = n0 + wave; n < n1; n += CWAVES) {
        const float* arow = alphas + n * S;
        const float* crow = colors + n * S * D;
        float C[D + 1];  // colour sums, then the density
        const float T = compose_front<D>(arow, crow, dp, S, lane, nullptr, 1, C);
        const float Dn = C[D];
        if (lane == 0) {
            float sc = 1.f / (1.f + 1e-6f - T);
            dens_out[n] = Dn;
#pragma unroll
            for (int c = 0; c < D; c++) color_out[n * D + c] = clampf(C[c] * sc, 0.f, 1.f);
        }
    }
}

template <int D>
__global__ __launch_bounds__(64 * CWAVES) void compose_bwd_kernel(
    float* __restrict__ g_alpha, float* __restrict__ g_colors, float* __restrict__ g_dp,
    const float* __restrict__ g_dens, const float* __restrict__ g_color, const float* __restrict__ alphas,
    const float* __restrict__ colors, const float* __restrict__ dp, int64_t N, int64_t S, int64_t ppb, int exact) {
    extern __shared__ float lds_gdp[];  // [S] if S <= LDS_GDP_MAX, else unused (global atomics)
    // transmittance entering chunk g * G (pass 1) and entering each chunk of the group being
    // walked back to front (pass 2); G = 1 up to MAXCH chunks, so pass 2 recomputes nothing
    __shared__ float t_in[CWAVES][MAXCH];
    __shared__ float t_grp[CWAVES][MAXCH];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    const bool lds = S <= LDS_GDP_MAX;
    if (lds)
        for (int64_t i = threadIdx.x; i < S; i += 64 * CWAVES) lds_gdp[i] = 0.f;
    __syncthreads();
    const int64_t n0 = (int64_t)blockIdx.x * ppb, n1 = min(N, n0 + ppb);
    const int nch = (int)((S + 63) / 64);
    const int G = (nch + MAXCH - 1) / MAXCH;
    for (int64_t n = n0 + wave; n < n1; n += CWAVES) {
        const float* arow = alphas + n * S;
        const float* crow = colors + n * S * D;
        // pass 1, front to back: totals and per-chunk incoming transmittance
        float C[D + 1];
        const float Tn = compose_front<D>(arow, crow, dp, S, lane, t_in[wave], G, C);
        wave_fence();  // t_in is read by every lane
        const float O = 1.f + 1e-6f - Tn;
        const float sc = 1.f / O;
        const float gD = g_dens ? g_dens[n] : 0.f;
        float gC[D];
#pragma unroll
        for (int c = 0; c < D; c++) {
            float s = C[c] * sc;
            gC[c] = (g_color && 0.f <= s && s <= 1.f) ? g_color[n * D + c] : 0.f;
        }
        // pass 2, back to front: affine suffix scan for the composite behind each stroke
        float Ud = 0.f, Uc[D], Rb = 1.f;
#pragma unroll
        for (int c = 0; c < D; c++) Uc[c] = 0.f;
        for (int ch = nch - 1; ch >= 0; ch--) {
            if (G > 1 && (ch % G == G - 1 || ch == nch - 1)) {
                // entering a group from behind: its chunks' incoming transmittance, recomputed
                // front to back from its checkpoint exactly as pass 1 formed it
                const int g0 = (ch / G) * G;
                float Tg = t_in[wave][ch / G];
                for (int c2 = g0; c2 <= ch; c2++) {
                    const int64_t k2 = S - 1 - ((int64_t)c2 * 64 + lane);
                    const float f2 = 1.f - (k2 >= 0 ? arow[k2] : 0.f);
                    if (lane == 0) t_grp[wave][c2 - g0] = Tg;
                    Tg = __shfl(Tg * scan_prod_excl(f2, lane) * f2, 63, 64);
                }
                wave_fence();  // t_grp is read by every lane
            }
            int64_t k = S - 1 - ((int64_t)ch * 64 + lane);
            bool v = k >= 0;
            float a = v ? arow[k] : 0.f;
            float f = 1.f - a;
            float dk = v ? dp[k] : 0.f;
            float ck[D];
#pragma unroll
            for (int c = 0; c < D; c++) ck[c] = v ? crow[k * D + c] : 0.f;
            const float Tin = G == 1 ? t_in[wave][ch] : t_grp[wave][ch % G];
            // without a nonzero alpha the chunk is transparent: everything behind a stroke is
            // what lies behind the chunk, and the carry stays as it is (an infinite or NaN
            // colour or density, whose product with an alpha of zero is NaN, goes the long way)
            float zero = 0.f * dk;
#pragma unroll
            for (int c = 0; c < D; c++) zero += 0.f * ck[c];
            const bool clear = __ballot(a != 0.f || !(zero == 0.f)) == 0ull;
            float Tk = Tin, Ubd = Ud, Rbk = Rb, Ubc[D];
#pragma unroll
            for (int c = 0; c < D; c++) Ubc[c] = Uc[c];
            if (!clear) {
                Tk = Tin * scan_prod_excl(f, lane);
                // inclusive suffix composition (m, bd, bc) of lanes lane..63
                float m = f, bd = dk * a, bc[D];
#pragma unroll
                for (int c = 0; c < D; c++) bc[c] = ck[c] * a;
#pragma unroll
                for (int off = 1; off < 64; off <<= 1) {
                    float m2 = __shfl_down(m, off, 64);
                    float bd2 = __shfl_down(bd, off, 64);
                    float bc2[D];
#pragma unroll
                    for (int c = 0; c < D; c++) bc2[c] = __shfl_down(bc[c], off, 64);
                    if (lane + off < 64) {
                        bd = bd + m * bd2;
#pragma unroll
                        for (int c = 0; c < D; c++) bc[c] = bc[c] + m * bc2[c];
                        m = m * m2;
                    }
                }
                // exclusive (strokes strictly behind this lane) composed with the carry
                float me = __shfl_down(m, 1, 64), bde = __shfl_down(bd, 1, 64), bce[D];
#pragma unroll
                for (int c = 0; c < D; c++) bce[c] = __shfl_down(bc[c], 1, 64);
                if (lane == 63) {
                    me = 1.f;
                    bde = 0.f;
#pragma unroll
                    for (int c = 0; c < D; c++) bce[c] = 0.f;
                }
                Ubd = bde + me * Ud;       // U_{k+1} (density)
                Rbk = me * Rb;             // R_{k+1}
#pragma unroll
                for (int c = 0; c < D; c++) Ubc[c] = bce[c] + me * Uc[c];
                // carry: compose this whole chunk in front of the stroke composite behind it
                const float m0 = __shfl(m, 0, 64), bd0 = __shfl(bd, 0, 64);
                Ud = bd0 + m0 * Ud;
#pragma unroll
                for (int c = 0; c < D; c++) Uc[c] = __shfl(bc[c], 0, 64) + m0 * Uc[c];
                Rb = m0 * Rb;
            }
            float w = a * Tk;
            float ga;
            if (exact) {
                ga = gD * Tk * (dk - Ubd);
#pragma unroll
                for (int c = 0; c < D; c++) ga += gC[c] * (Tk * (ck[c] - Ubc[c]) * O - C[c] * Tk * Rbk) * (sc * sc);
            } else {
                // compositing.cu:143-154 with T = T_{k+1} and suffix = T_{k+1} U_{k+1}
                float Ta = Tk * f;
                float s1 = 1.f / fmaxf(1.f - a, 1e-6f);
                ga = gD * (Ta * dk - Ta * Ubd) * s1;
                float s2 = s1 * sc * sc;
#pragma unroll
                for (int c = 0; c < D; c++) ga += gC[c] * (Ta * ck[c] * (O - a) - Ta * Ubc[c]) * s2;
            }
            if (v) {
                g_alpha[n * S + k] = ga;
#pragma unroll
                for (int c = 0; c < D; c++) g_colors[(n * S + k) * D + c] = a > 0.f ? gC[c] * sc * w : 0.f;
                if (a > 0.f) {
                    if (lds) atomicAdd(&lds_gdp[k], gD * w);
                    else atomicAdd(&g_dp[k], gD * w);
                }
            }
        }
    }
    if (!lds) return;
    __syncthreads();
    for (int64_t i = threadIdx.x; i < S; i += 64 * CWAVES) {
        float v = lds_gdp[i];
        if (v != 0.f) atomicAdd(&g_dp[i], v);
    }
}

static int64_t compose_ppb(int64_t N) {
    int64_t ppb = (N + 4095) / 4096;
    ppb = ppb < CWAVES ? CWAVES : ppb;
    return ((ppb + CWAVES - 1) / CWAVES) * CWAVES;
}

}  // namespace n3ds

using namespace n3ds;

N3DS_EXPORT int n3ds_compose_forward(float* density_out, float* color_out, const float* alphas, const float* colors,
                                     const float* density_params, int64_t n_points, int64_t n_strokes,
                                     int64_t color_dim, void* stream) {
    N3DS_REQUIRE(color_dim == 1 || color_dim == 3, "color_dim must be 1 or 3 (got %lld)", (long long)color_dim);
    N3DS_REQUIRE(n_points >= 0 && n_strokes >= 0, "negative size");
    if (n_points == 0) return N3DS_OK;
    int64_t ppb = compose_ppb(n_points);
    dim3 grid((unsigned)((n_points + ppb - 1) / ppb));
    if (color_dim == 3)
        hipLaunchKernelGGL(compose_fwd_kernel<3>, grid, dim3(64 * CWAVES), 0, (hipStream_t)stream, density_out,
                           color_out, alphas, colors, density_params, n_points, n_strokes, ppb);
    else
        hipLaunchKernelGGL(compose_fwd_kernel<1>, grid, dim3(64 * CWAVES), 0, (hipStream_t)stream, density_out,
                           color_out, alphas, colors, density_params, n_points, n_strokes, ppb);
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}

N3DS_EXPORT int n3ds_compose_backward(float* grad_alphas, float* grad_colors, float* grad_density_params,
                                      const float* grad_density_out, const float* grad_color_out,
                                      const float* alphas, const float* colors, const float* density_params,
                                      int64_t n_points, int64_t n_strokes, int64_t color_dim, int adjoint_exact,
                                      void* stream) {
    N3DS_REQUIRE(color_dim == 1 || color_dim == 3, "color_dim must be 1 or 3 (got %lld)", (long long)color_dim);
    N3DS_REQUIRE(n_points >= 0 && n_strokes >= 0, "negative size");
    N3DS_REQUIRE(n_strokes <= (int64_t)64 * MAXCH * MAXCH, "n_strokes (%lld) exceeds %d", (long long)n_strokes,
                 64 * MAXCH * MAXCH);
    if (n_points == 0 || n_strokes == 0) return N3DS_OK;
    int64_t ppb = compose_ppb(n_points);
    dim3 grid((unsigned)((n_points + ppb - 1) / ppb));
    size_t shm = n_strokes <= LDS_GDP_MAX ? (size_t)n_strokes * sizeof(float) : 0;
    if (color_dim == 3)
        hipLaunchKernelGGL(compose_bwd_kernel<3>, grid, dim3(64 * CWAVES), shm, (hipStream_t)stream, grad_alphas,
                           grad_colors, grad_density_params, grad_density_out, grad_color_out, alphas, colors,
                           density_params, n_points, n_strokes, ppb, adjoint_exact);
    else
        hipLaunchKernelGGL(compose_bwd_kernel<1>, grid, dim3(64 * CWAVES), shm, (hipStream_t)stream, grad_alphas,
                           grad_colors, grad_density_params, grad_density_out, grad_color_out, alphas, colors,
                           density_params, n_points, n_strokes, ppb, adjoint_exact);
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}
