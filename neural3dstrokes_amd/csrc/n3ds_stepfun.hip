// Interval resampling from a step function: the proposal levels' sampler,
// drop-in for source/utils/stepfun.py:sample_intervals (:280-317) with
// sample (:216-254), invert_cdf (:195-202), integrate_weights (:149-170) and
// sorted_interp (:5-24), as called at models.py:168-181.
//
// Mapping: one wavefront per ray.  The ray's bin edges t [m+1], CDF
// cw0 [m+1] and centres [n] are staged in the wave's LDS slice: softmax of the logits by two
// wave reductions (max, sum of exp), the CDF by a 64-lane inclusive scan with
// a running carry, clamped to 1 and closed with exact 0 and 1.  Each lane then
// evaluates centres: the inverse CDF at a sample u is an upper-bound binary
// search in cw0 (cw0 is non-decreasing, so "last entry <= u" is what
// sorted_interp's masked max / min select for sorted t) and one linear
// interpolation; fencepost o takes the midpoint of centres o-1 and o, and the
// first / last the reflection of the end midpoint clamped to the domain.
// Per ray the work is O(m + n log m) and the bytes are the inputs and outputs
// once (HBM / latency bound).
#include <algorithm>

#include "n3ds_capi.h"
#include "n3ds_math.h"

namespace n3ds {

constexpr int SF_MAX_FLOATS = 16384;  // LDS floats per ray slice: 2 (m + 1) + n (<= 64 KB per block)

// LDS ordering between the lanes of one wavefront (no block barrier)
__device__ __forceinline__ void sf_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the inverse CDF at u (sorted_interp(u, cw0, t) for non-decreasing cw0, sorted t)
// first: the first index with cw[idx] > u, in [1, m] after the clamp
__device__ __forceinline__ float sf_center(const float* cw, const float* te, int m, float u, int first) {
    const int k = min(max(first, 1), m);
    const float x0 = cw[k - 1], x1 = cw[k], f0 = te[k - 1], f1 = te[k];
    float off = (u - x0) / (x1 - x0);
    if (off != off) off = 0.f;  // nan_to_num(., 0)
    off = fminf(fmaxf(off, 0.f), 1.f);
    return __fadd_rn(f0, __fmul_rn(off, __fsub_rn(f1, f0)));
}

// 64 entries of cw0 = [0, min(cumsum(w[:-1]), 1), 1]: lane's weight v of bin j after the
// running sum carry; returns the sum so far
__device__ __forceinline__ float sf_cdf(float* cw, int j, int m, float v, float carry, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const float o = __shfl_up(v, off, 64);
        if (lane >= off) v += o;
    }
    v += carry;
    if (j < m - 1) cw[j + 1] = fminf(v, 1.f);
    return __shfl(v, 63, 64);
}

// NB > 0: at most 64 NB bins, their logits and exponentials in registers (0: any number, read
// and exponentiated again for each use): 67 instead of 75 us at 65536 rays, 192 bins and 128
// samples, with the two searches of a lane side by side.  (A second search that no sample of the
// last 64 needs cost 73 instead of 63 us at 65 bins and 64 samples, and side by side past 256
// bins 130 instead of 120 at 300 bins and 128 samples.)
template <int NB>
__global__ __launch_bounds__(256) void sample_intervals_kernel(float* __restrict__ t_out,
                                                               const float* __restrict__ t,
                                                               const float* __restrict__ logits,
                                                               const float* __restrict__ u_base,
                                                               const float* __restrict__ jitter, int jitter_width,
                                                               float max_jitter, int64_t n_rays, int m, int n,
                                                               float minval, float maxval, int waves) {
    extern __shared__ float sf_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    float* cw = sf_lds + (int64_t)wave * (2 * (m + 1) + n);
    float* te = cw + (m + 1);
    float* cs = te + (m + 1);
    for (int64_t r = (int64_t)blockIdx.x * waves + wave; r < n_rays; r += (int64_t)gridDim.x * waves) {
        const float* tr = t + r * (m + 1);
        const float* lr = logits + r * m;
        // softmax over the m bins
        float carry = 0.f;
        if constexpr (NB > 0) {
            float v[NB], mx = -INFINITY, se = 0.f;
#pragma unroll
            for (int s = 0; s < NB; s++) {
                v[s] = lane + 64 * s < m ? lr[lane + 64 * s] : -INFINITY;
                mx = fmaxf(mx, v[s]);
            }
            mx = wave_max(mx);
#pragma unroll
            for (int s = 0; s < NB; s++)
                if (lane + 64 * s < m) {
                    v[s] = expf(v[s] - mx);
                    se += v[s];
                }
            se = wave_sum_halves(se);  // (a sample's bin may turn on its last bit)
#pragma unroll
            for (int s = 0; s < NB; s++) {
                const int j = lane + 64 * s;
                carry = sf_cdf(cw, j, m, j < m - 1 ? v[s] / se : 0.f, carry, lane);
            }
        } else {
            float mx = -INFINITY;
            for (int j = lane; j < m; j += 64) mx = fmaxf(mx, lr[j]);
            mx = wave_max(mx);
            float se = 0.f;
            for (int j = lane; j < m; j += 64) se += expf(lr[j] - mx);
            se = wave_sum_halves(se);
            for (int j0 = 0; j0 < m - 1; j0 += 64) {
                const int j = j0 + lane;
                carry = sf_cdf(cw, j, m, j < m - 1 ? expf(lr[j] - mx) / se : 0.f, carry, lane);
            }
        }
        if (lane == 0) {
            cw[0] = 0.f;
            cw[m] = 1.f;
        }
        for (int j = lane; j <= m; j += 64) te[j] = tr[j];
        sf_wave_sync();
        float* outr = t_out + r * (n + 1);
        const float* jr = jitter ? jitter + r * jitter_width : nullptr;
        auto position = [&](int i) {
            const float u = u_base[i];
            return jr ? __fadd_rn(u, __fmul_rn(jr[jitter_width == 1 ? 0 : i], max_jitter)) : u;
        };
        int i0 = 0;
        for (; NB > 0 && i0 + 64 < n; i0 += 128) {  // two searches side by side
            const int i = i0 + lane, i1 = min(i + 64, n - 1);
            const float u0 = position(i), u1 = position(i1);
            int lo0 = 0, hi0 = m + 1, lo1 = 0, hi1 = m + 1;  // first index with cw[idx] > u
            for (int left = m + 1; left > 0; left >>= 1) {
                const int mid0 = (lo0 + hi0) >> 1, mid1 = (lo1 + hi1) >> 1;
                const bool le0 = cw[min(mid0, m)] <= u0, le1 = cw[min(mid1, m)] <= u1;
                const bool go0 = lo0 < hi0, go1 = lo1 < hi1;
                if (go0 && le0) lo0 = mid0 + 1;
                if (go0 && !le0) hi0 = mid0;
                if (go1 && le1) lo1 = mid1 + 1;
                if (go1 && !le1) hi1 = mid1;
            }
            cs[i] = sf_center(cw, te, m, u0, lo0);
            if (i + 64 < n) cs[i1] = sf_center(cw, te, m, u1, lo1);
        }
        for (int i = i0 + lane; i < n; i += 64) {  // at most 64 are left
            const float u = position(i);
            int lo = 0, hi = m + 1;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (cw[mid] <= u) lo = mid + 1;
                else hi = mid;
            }
            cs[i] = sf_center(cw, te, m, u, lo);
        }
        sf_wave_sync();
        for (int o = lane; o <= n; o += 64) {
            float val;
            if (o == 0 || o == n) {
                const int e = o == 0 ? 0 : n - 1, nb = o == 0 ? 1 : n - 2;  // end centre and its neighbour
                const float ce = cs[e], cn = cs[nb];
                const float midv = (o == 0 ? __fadd_rn(cn, ce) : __fadd_rn(ce, cn)) / 2.f;
                const float refl = __fsub_rn(2.f * ce, midv);
                // clamp_min / clamp_max keep NaN
                val = o == 0 ? (refl < minval ? minval : refl) : (refl > maxval ? maxval : refl);
            } else {
                val = __fadd_rn(cs[o], cs[o - 1]) / 2.f;
            }
            outr[o] = val;
        }
        sf_wave_sync();  // the next ray overwrites the slice
    }
}

// number of entries of the sorted a[0..n) below x (strictly, or at most x when le)
__device__ __forceinline__ int sf_rank(const float* a, int n, float x, bool le) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (le ? a[mid] <= x : a[mid] < x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// max_dilate_weights (stepfun.py:136-146 over max_dilate :120-133, weight_to_pdf :109-112,
// pdf_to_weight :115-117): per ray, the edges t, t[:-1] - d and t[1:] + d merged in
// sorted order (three sorted runs: each element's place is its index plus its rank in
// the other two runs, ties broken run by run), clipped to the domain; the PDF at edge i
// is the max of p_j over the bins with t_j - d <= e_i < t_{j+1} + d (a contiguous range
// of j for sorted t, 0 when some bin does not cover it); back to weights, renormalised.
// LDS per wave: t [m+1], p [m], merged edges [3m+1].
__device__ __forceinline__ void dilate_ray(float* __restrict__ t_out, float* __restrict__ w_out,
                                           const float* __restrict__ t, const float* __restrict__ w, int64_t r, int m,
                                           float dilation, float minval, float maxval, int renormalize, float* ts,
                                           float* ps, float* es) {
    const int lane = threadIdx.x & 63, ne = 3 * m + 1;
    const float eps = 1.1920928955078125e-7f;  // float32 machine epsilon
    const float* tr = t + r * (m + 1);
    const float* wr = w + r * m;
    for (int j = lane; j <= m; j += 64) ts[j] = tr[j];
    sf_wave_sync();
    for (int j = lane; j < m; j += 64) ps[j] = wr[j] / fmaxf(__fsub_rn(ts[j + 1], ts[j]), eps);
    // merged edge positions: run A = t [m+1], B = t[:-1] - d [m], C = t[1:] + d [m]
    for (int k = lane; k < ne; k += 64) {
        float v;
        int pos;
        if (k <= m) {  // A: after B / C entries strictly below
            v = ts[k];
            int lo = 0, hi = m;  // B below v: t_j - d < v
            while (lo < hi) { const int mid = (lo + hi) >> 1; if (__fsub_rn(ts[mid], dilation) < v) lo = mid + 1; else hi = mid; }
            int cb = lo;
            lo = 0; hi = m;      // C below v: t_{j+1} + d < v
            while (lo < hi) { const int mid = (lo + hi) >> 1; if (__fadd_rn(ts[mid + 1], dilation) < v) lo = mid + 1; else hi = mid; }
            pos = k + cb + lo;
        } else if (k <= 2 * m) {  // B: after A entries <= v and C entries < v
            const int j = k - (m + 1);
            v = __fsub_rn(ts[j], dilation);
            const int ca = sf_rank(ts, m + 1, v, true);
            int lo = 0, hi = m;
            while (lo < hi) { const int mid = (lo + hi) >> 1; if (__fadd_rn(ts[mid + 1], dilation) < v) lo = mid + 1; else hi = mid; }
            pos = j + ca + lo;
        } else {  // C: after A and B entries <= v
            const int j = k - (2 * m + 1);
            v = __fadd_rn(ts[j + 1], dilation);
            const int ca = sf_rank(ts, m + 1, v, true);
            int lo = 0, hi = m;
            while (lo < hi) { const int mid = (lo + hi) >> 1; if (__fsub_rn(ts[mid], dilation) <= v) lo = mid + 1; else hi = mid; }
            pos = j + ca + lo;
        }
        es[pos] = fminf(fmaxf(v, minval), maxval);  // torch.clip(min, max)
    }
    sf_wave_sync();
    float* tout = t_out + r * ne;
    float* wout = w_out + r * (ne - 1);
    float wsum = 0.f;
    for (int i = lane; i < ne; i += 64) {
        const float e = es[i];
        tout[i] = e;
        if (i == ne - 1) continue;
        // bins covering e: t_j - d <= e (a prefix j < a) and t_{j+1} + d > e (a suffix j >= b)
        int lo = 0, hi = m;
        while (lo < hi) { const int mid = (lo + hi) >> 1; if (__fsub_rn(ts[mid], dilation) <= e) lo = mid + 1; else hi = mid; }
        const int a = lo;
        lo = 0; hi = m;
        while (lo < hi) { const int mid = (lo + hi) >> 1; if (__fadd_rn(ts[mid + 1], dilation) <= e) lo = mid + 1; else hi = mid; }
        const int b = lo;
        float pd = (b == 0 && a == m) ? -INFINITY : 0.f;
        for (int j = b; j < a; j++) pd = fmaxf(pd, ps[j]);
        const float wd = __fmul_rn(pd, __fsub_rn(es[i + 1], e));
        wout[i] = wd;
        wsum += wd;
    }
    if (renormalize) {
        wsum = fmaxf(wave_sum_halves(wsum), eps);
        for (int i = lane; i < ne - 1; i += 64) wout[i] = wout[i] / wsum;
    }
}

__global__ __launch_bounds__(256) void max_dilate_kernel(float* __restrict__ t_out, float* __restrict__ w_out,
                                                         const float* __restrict__ t, const float* __restrict__ w,
                                                         int64_t n_rays, int m, float dilation, float minval,
                                                         float maxval, int renormalize, int waves) {
    extern __shared__ float sf_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    float* ts = sf_lds + (int64_t)wave * (5 * m + 2);
    for (int64_t r = (int64_t)blockIdx.x * waves + wave; r < n_rays; r += (int64_t)gridDim.x * waves) {
        dilate_ray(t_out, w_out, t, w, r, m, dilation, minval, maxval, renormalize, ts, ts + (m + 1), ts + (2 * m + 1));
        sf_wave_sync();  // the next ray overwrites the slice
    }
}

// At most 64 bins, one per lane.  A lane places its three edges with six binary searches side
// by side (one after the other, run by run, they were 84 dependent LDS reads and two thirds of
// the instructions this is bound by), and the bins covering an edge follow from the merged
// order: the runs' elements are marked at their places, and as many t_j - d (or t_{j+1} + d)
// are at most e_i as there are marks up to the last edge that equals e_i.  Marks leave out
// what lies above the domain, which the clip moved to maxval.  A ray whose edges are not
// sorted goes through dilate_ray.  89 instead of 138 us at 65536 rays x 64 bins (the bytes
// alone are 33 us of a copy's time).
// LDS per wave: t [m+1], p [m], merged edges [3m+1], marks [3m+1].
//
// Up to 21 bins the 3 m + 1 edges are one round of dilate_ray's lanes, whose shorter chain is then
// the faster: 65536 rays x 8 bins 52 against 65 us, x 20 61 against 71, x 24 80 against 75.
constexpr int DILATE_SMALL = 64, DILATE_LEAST = 22;
constexpr int dilate_small_floats(int m) { return 8 * m + 3; }

// entries of a[0, n), n <= 64 + 1, that come before x: below it, or equal too (LE)
template <bool LE>
__device__ __forceinline__ int sf_before(const float* a, int n, float shift, float x) {
    int pos = 0;
#pragma unroll
    for (int step = 64; step > 0; step >>= 1) {
        const float v = a[min(pos + step, n) - 1] + shift;
        if (pos + step <= n && (LE ? v <= x : v < x)) pos += step;
    }
    return pos;
}

__global__ __launch_bounds__(256) void max_dilate_small_kernel(float* __restrict__ t_out, float* __restrict__ w_out,
                                                               const float* __restrict__ t, const float* __restrict__ w,
                                                               int64_t n_rays, int m, float dilation, float minval,
                                                               float maxval, int renormalize) {
    extern __shared__ float sf_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform per wavefront
    const int ne = 3 * m + 1;
    float* ts = sf_lds + wave * dilate_small_floats(m);
    float* ps = ts + (m + 1);
    float* es = ps + m;
    int* mark = (int*)(es + ne);
    const float eps = 1.1920928955078125e-7f;  // float32 machine epsilon
    const bool on = lane < m;
    for (int64_t r = (int64_t)blockIdx.x * 4 + wave; r < n_rays; r += (int64_t)gridDim.x * 4) {
        const float* tr = t + r * (m + 1);
        const float t0 = tr[min(lane, m)], t1 = tr[min(lane + 1, m)], wj = w[r * m + min(lane, m - 1)];
        if (__ballot(on && !(t0 <= t1)) != 0ull) {
            dilate_ray(t_out, w_out, t, w, r, m, dilation, minval, maxval, renormalize, ts, ps, es);
            sf_wave_sync();
            continue;
        }
        if (on) {
            ts[lane] = t0;
            ps[lane] = wj / fmaxf(__fsub_rn(t1, t0), eps);
            if (lane == m - 1) ts[m] = t1;
        }
        sf_wave_sync();
        const float vb = __fsub_rn(t0, dilation), vc = __fadd_rn(t1, dilation);
        // places as in dilate_ray: equal edges in the order t, t - d, t + d
        const int pa = lane + sf_before<false>(ts, m, -dilation, t0) + sf_before<false>(ts + 1, m, dilation, t0);
        const int pb = lane + sf_before<true>(ts, m + 1, 0.f, vb) + sf_before<false>(ts + 1, m, dilation, vb);
        const int pc = lane + sf_before<true>(ts, m + 1, 0.f, vc) + sf_before<true>(ts, m, -dilation, vc);
        const float tm = ts[m];
        const int pm = m + __popcll(__ballot(on && vb < tm)) + __popcll(__ballot(on && vc < tm));
        if (on) {
            es[pa] = fminf(fmaxf(t0, minval), maxval);  // torch.clip(min, max)
            es[pb] = fminf(fmaxf(vb, minval), maxval);
            es[pc] = fminf(fmaxf(vc, minval), maxval);
            mark[pa] = 0;
            mark[pb] = vb <= maxval ? 1 : 0;
            mark[pc] = vc <= maxval ? 2 : 0;
        }
        if (lane == 0) {
            es[pm] = fminf(fmaxf(tm, minval), maxval);
            mark[pm] = 0;
        }
        sf_wave_sync();
        // per word of 64 edges: the marks, and which edges differ from the next one
        float e[3], en[3];
        unsigned long long mb[4], mc[4], last[4];
#pragma unroll
        for (int s = 0; s < 3; s++) {
            const int i = lane + 64 * s;
            e[s] = es[min(i, ne - 1)];
            en[s] = es[min(i + 1, ne - 1)];
            const int k = i < ne ? mark[min(i, ne - 1)] : 0;
            mb[s] = __ballot(k == 1);
            mc[s] = __ballot(k == 2);
            last[s] = __ballot(i < ne && (i == ne - 1 || e[s] != en[s]));
        }
        const int k3 = ne > 192 ? mark[ne - 1] : 0;  // 64 bins: the last edge by itself
        mb[3] = k3 == 1 ? 1ull : 0ull;
        mc[3] = k3 == 2 ? 1ull : 0ull;
        last[3] = ne > 192 ? 1ull : 0ull;
        // marks up to the first such edge at or after word s
        int beforeb[5] = {0}, beforec[5] = {0}, nextb[5] = {0}, nextc[5] = {0};
#pragma unroll
        for (int s = 0; s < 4; s++) {
            beforeb[s + 1] = beforeb[s] + __popcll(mb[s]);
            beforec[s + 1] = beforec[s] + __popcll(mc[s]);
        }
#pragma unroll
        for (int s = 3; s >= 0; s--) {
            const unsigned long long upto = last[s] ^ (last[s] - 1ull);  // up to the lowest bit
            nextb[s] = last[s] ? beforeb[s] + __popcll(mb[s] & upto) : nextb[s + 1];
            nextc[s] = last[s] ? beforec[s] + __popcll(mc[s] & upto) : nextc[s + 1];
        }
        float* tout = t_out + r * ne;
        float* wout = w_out + r * (ne - 1);
        float wd[3], wsum = 0.f;
#pragma unroll
        for (int s = 0; s < 3; s++) {
            const int i = lane + 64 * s;
            const unsigned long long rest = (last[s] >> lane) << lane;
            const unsigned long long upto = rest ^ (rest - 1ull);
            const int a = rest ? beforeb[s] + __popcll(mb[s] & upto) : nextb[s + 1];
            const int b = rest ? beforec[s] + __popcll(mc[s] & upto) : nextc[s + 1];
            wd[s] = 0.f;
            if (i < ne) tout[i] = e[s];
            if (i < ne - 1) {
                float pd = (b == 0 && a == m) ? -INFINITY : 0.f;
                for (int j = b; j < a; j++) pd = fmaxf(pd, ps[j]);
                wd[s] = __fmul_rn(pd, __fsub_rn(en[s], e[s]));
                wsum += wd[s];
            }
        }
        if (ne > 192 && lane == 0) tout[ne - 1] = es[ne - 1];
        if (renormalize) wsum = fmaxf(wave_sum_halves(wsum), eps);
#pragma unroll
        for (int s = 0; s < 3; s++) {
            const int i = lane + 64 * s;
            if (i < ne - 1) wout[i] = renormalize ? wd[s] / wsum : wd[s];
        }
        sf_wave_sync();  // the next ray overwrites the slice
    }
}

}  // namespace n3ds

using namespace n3ds;

N3DS_EXPORT int n3ds_sample_intervals(float* t_out, const float* t, const float* w_logits, const float* u_base,
                                      const float* jitter, int jitter_width, float max_jitter, int64_t n_rays,
                                      int n_bins, int n_samples, float minval, float maxval, void* stream) {
    N3DS_REQUIRE(n_samples > 1, "num_samples must be > 1, is %d.", n_samples);
    N3DS_REQUIRE(n_bins >= 1 && 2 * ((int64_t)n_bins + 1) + n_samples <= SF_MAX_FLOATS,
                 "2 (n_bins + 1) + n_samples = %lld exceeds %d", 2 * ((long long)n_bins + 1) + n_samples, SF_MAX_FLOATS);
    N3DS_REQUIRE(n_rays >= 0, "negative size");
    N3DS_REQUIRE(!jitter || jitter_width == 1 || jitter_width == n_samples,
                 "jitter width must be 1 or n_samples (got %d)", jitter_width);
    if (n_rays == 0) return N3DS_OK;
    N3DS_REQUIRE(t_out && t && w_logits && u_base, "null argument");
    const int per_wave = 2 * (n_bins + 1) + n_samples;
    const int waves = per_wave <= SF_MAX_FLOATS / 4 ? 4 : 1;
    const size_t lds = (size_t)waves * per_wave * sizeof(float);
    const int64_t blocks = std::min<int64_t>((n_rays + waves - 1) / waves, 256 * 32);
    typedef void (*Kernel)(float*, const float*, const float*, const float*, const float*, int, float, int64_t, int,
                           int, float, float, int);
    static const Kernel kernels[5] = {sample_intervals_kernel<0>, sample_intervals_kernel<1>,
                                      sample_intervals_kernel<2>, sample_intervals_kernel<3>,
                                      sample_intervals_kernel<4>};
    hipLaunchKernelGGL(kernels[n_bins <= 256 ? (n_bins + 63) / 64 : 0], dim3((unsigned)blocks), dim3(64 * waves), lds,
                       (hipStream_t)stream, t_out, t, w_logits, u_base, jitter, jitter_width, max_jitter, n_rays,
                       n_bins, n_samples, minval, maxval, waves);
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}

N3DS_EXPORT int n3ds_max_dilate_weights(float* t_out, float* w_out, const float* t, const float* w, int64_t n_rays,
                                        int n_bins, float dilation, float minval, float maxval, int renormalize,
                                        void* stream) {
    N3DS_REQUIRE(n_bins >= 1 && 5 * (int64_t)n_bins + 2 <= 16384, "n_bins %d outside [1, 3276]", n_bins);
    N3DS_REQUIRE(n_rays >= 0, "negative size");
    if (n_rays == 0) return N3DS_OK;
    N3DS_REQUIRE(t_out && w_out && t && w, "null argument");
    if (n_bins >= DILATE_LEAST && n_bins <= DILATE_SMALL) {
        const size_t lds = (size_t)4 * dilate_small_floats(n_bins) * sizeof(float);
        const int64_t blocks = std::min<int64_t>((n_rays + 3) / 4, 256 * 32);
        hipLaunchKernelGGL(max_dilate_small_kernel, dim3((unsigned)blocks), dim3(256), lds, (hipStream_t)stream, t_out,
                           w_out, t, w, n_rays, n_bins, dilation, minval, maxval, renormalize);
        N3DS_LAUNCH_CHECK();
        return N3DS_OK;
    }
    const int per_wave = 5 * n_bins + 2;
    const int waves = per_wave <= 4096 ? 4 : 1;
    const size_t lds = (size_t)waves * per_wave * sizeof(float);
    const int64_t blocks = std::min<int64_t>((n_rays + waves - 1) / waves, 256 * 32);
    hipLaunchKernelGGL(max_dilate_kernel, dim3((unsigned)blocks), dim3(64 * waves), lds, (hipStream_t)stream, t_out,
                       w_out, t, w, n_rays, n_bins, dilation, minval, maxval, renormalize, waves);
    N3DS_LAUNCH_CHECK();
    return N3DS_OK;
}
