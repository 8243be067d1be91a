// qmag_mmf.hip -- the fp32 dequantise-then-dot matmul (src/quants.c:80-133, the
// QMA_NOQ8K path) for several tokens on the fp32 matrix cores.
//
// A workgroup takes 16 rows x up to 32 tokens, its waves the rows' super-blocks
// in turn.  A wave holds a super-block of the 16 rows in its LDS image
// (qmag_mfma.h), dequantises 16 weights per lane and step (each once for all
// the tokens; the one-token kernel does it again for every token) and feeds
// them to v_mfma_f32_16x16x4f32 with the matching 16 values of x: any
// assignment of k to lanes serves as long as both operands use it.  The sums are
// kept as accurate as the one-token kernel's lane tree: chains of 8 products
// (two MFMAs), added pairwise within a super-block and over the waves (one
// chain per step of 64 products gave 1.57e-7 of the result against 9.7e-8),
// and over a long row in chains of super-blocks (mmf_chain).
// What bounds it at 24 tokens x 2048 x 2048 (8.6 us with Q4_K rows, 9.6 with
// Q6_K; the one-token kernel 13.4 and 20.8) is the round trips of a wave's super-block; requesting
// x a step ahead cost more in registers (two waves per SIMD) than it hid: 10.1.
#include "qmag_mfma.h"

namespace qmag {

// the lane's 16 weights of step s
__device__ __forceinline__ float byte_f(uint32_t w, int b) { return (float)((w >> (8 * b)) & 255u); }

template <int WT>
struct Deq16 {
    using Row = WRow<WT, 4>;
    __device__ static __forceinline__ void weights(const Row &w, const typename Row::Raw &r, int s, float (&o)[16])
    {
        const int up = s & 1;
        if constexpr (WT == QMAG_TYPE_Q4_K) {
            const uint32_t byte = 8 * (2u * (uint32_t)(lane_id() >> 5) + (uint32_t)up);
            const uint32_t sc = ((w.S.sl[s >> 1] >> byte) & 7) | (((w.S.sh[s >> 1] >> byte) & 7) << 3);
            const float d1 = w.d() * (float)sc, m1 = w.dmin() * (float)((w.S.m[s >> 1] >> byte) & 63);
            const uint32_t v[4] = {r.v.x, r.v.y, r.v.z, r.v.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t n = (up ? v[k] >> 4 : v[k]) & 0x0F0F0F0Fu;
#pragma unroll
                for (int b = 0; b < 4; b++) o[4 * k + b] = fmaf(d1, byte_f(n, b), -m1);
            }
        } else {
            const uint32_t scw[4] = {w.sc.x, w.sc.y, w.sc.z, w.sc.w};
            const float ds = w.d() * (float)(int)(int8_t)(scw[s] >> (8 * (lane_id() >> 4)));
            const uint32_t l[4] = {r.l[0].x, r.l[0].y, r.l[0].z, r.l[0].w}, h[4] = {r.h.x, r.h.y, r.h.z, r.h.w};
            const uint32_t sh = 2u * (uint32_t)((lane_id() >> 5) + 2 * up);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t q = ((up ? l[k] >> 4 : l[k]) & 0x0F0F0F0Fu) | (((h[k] >> sh) & 0x03030303u) << 4);
#pragma unroll
                for (int b = 0; b < 4; b++) o[4 * k + b] = ds * (byte_f(q, b) - 32.0f);
            }
        }
    }
};

// Super-blocks of a wave per running sum: four, and eight once a wave has more
// than 32 (Q4_K, against 64 bits, in one sum / in chains / the one-token
// kernel: n_in 16,384 1.10e-7 / 1.07e-7 / 1.07e-7, 65,536 1.43e-7 / 1.17e-7 /
// 1.17e-7, 262,144 2.28e-7 / 1.35e-7 / 1.51e-7; chains of eight at 16,384 1.10e-7).
__host__ __device__ __forceinline__ int mmf_chain(int nb, int nw) { return nb > 32 * nw ? 8 : 4; }

template <int WT, int MT, bool LNG>            // LNG: long rows (put_partials)
__global__ __launch_bounds__(512) void mmf_kernel(const uint8_t *__restrict__ W, const float *__restrict__ x,
                                                  float *__restrict__ out, int nb, int n_out, int T)
{
    using Row = WRow<WT, 4>;
    extern __shared__ __align__(16) uint8_t s_dyn[];
    const int lane = lane_id(), lr = lane & 15;
    const int wv = (int)(threadIdx.x >> 6), nw = (int)(blockDim.x >> 6);
    const int row0 = (int)blockIdx.x * 16, t0 = (int)blockIdx.y * 16 * MT;
    WImage<WT, 16> img;
    img.init(s_dyn + wv * img.BYTES, W, row0, n_out, nb);
    const float *xp[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) xp[m] = x + (size_t)min(t0 + 16 * m + lr, T - 1) * nb * QK_K;
    float r[MT][4] = {};
    float *s_part = (float *)(s_dyn + (LNG ? nw * img.BYTES : 0));
    const int chain = mmf_chain(nb, nw);
    int done = 0;
    if (wv < nb) img.request_all(wv);          // wave-uniform
    for (int ib = wv; ib < nb; ib += nw) {
        img.store();
        const Row w(img.block(), img.shift(ib));
        typename Row::Raw raw[2];
        w.read(0, raw[0]);
        w.read(2, raw[1]);
        if (ib + nw < nb) img.request_all(ib + nw);
        v4f acc[MT][4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            float4 a[MT][4];
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int k = 0; k < 4; k++) a[m][k] = ldg4(xp[m] + ib * QK_K + Row::koff(s) + 4 * k);
            float b[16];
            Deq16<WT>::weights(w, raw[s >> 1], s, b);
#pragma unroll
            for (int m = 0; m < MT; m++) {
                v4f c[8];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const v4f z = {0.f, 0.f, 0.f, 0.f};
                    c[2 * k] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][k].x, b[4 * k], z, 0, 0, 0);
                    c[2 * k + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][k].y, b[4 * k + 1], z, 0, 0, 0);
                    c[2 * k] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][k].z, b[4 * k + 2], c[2 * k], 0, 0, 0);
                    c[2 * k + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][k].w, b[4 * k + 3], c[2 * k + 1], 0, 0, 0);
                }
                acc[m][s] = ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
            }
        }
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int i = 0; i < 4; i++) r[m][i] += (acc[m][0][i] + acc[m][1][i]) + (acc[m][2][i] + acc[m][3][i]);
        if constexpr (LNG)
            if (++done % chain == 0) put_partials<MT>(s_part, wv, r, done > chain);
    }
    __syncthreads();                           // every wave is done with its image
    put_partials<MT>(s_part, wv, r, LNG);   // of long rows every wave has a whole chain there
    __syncthreads();
    for (int k = (int)threadIdx.x; k < MT * 256; k += (int)blockDim.x) {
        float p[8];
#pragma unroll
        for (int u = 0; u < 8; u++) p[u] = u < nw ? s_part[u * MT * 256 + k] : 0.0f;
        const float v = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        const int l = k & 63, i = (k >> 6) & 3, m = k >> 8;
        const int t = t0 + 16 * m + 4 * (l >> 4) + i, rw = row0 + (l & 15);
        if (t < T && rw < n_out) out[(size_t)t * n_out + rw] = v;
    }
}

template <int WT>
static int launch_mmf_t(const float *x, const uint8_t *W, int nb, int n_out, int T, float *out, hipStream_t s)
{
    const int mt = T > 16 ? 2 : 1;
    int nw = 1;
    while (nw < 8 && nw < nb) nw *= 2;
    const int chain = mmf_chain(nb, nw);
    const bool lng = long_row(nb, nw, chain);
    const size_t lds = split_lds(nb, nw, chain, mt, WImage<WT, 16>::BYTES);
    const dim3 grid((n_out + 15) / 16, (T + 16 * mt - 1) / (16 * mt)), wg(64 * nw);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, wg, lds, s, W, x, out, nb, n_out, T); };
    if (mt == 1) launch(lng ? mmf_kernel<WT, 1, true> : mmf_kernel<WT, 1, false>);
    else launch(lng ? mmf_kernel<WT, 2, true> : mmf_kernel<WT, 2, false>);
    QMAG_HIP(hipGetLastError());
    return QMAG_OK;
}

// The one-token kernel spreads over the tokens and takes few rows and tokens
// faster; its time grows with rows x tokens x super-blocks, this one's with a
// wave's super-blocks and tiles, of 32 tokens from 17 on, and fewer than five
// super-blocks leave waves without work.  The line was fitted to 210 points a
// type (1 to 16 super-blocks, 2 to 48 tokens, 250 to 8000 rows; at most 9%
// (Q4_K) and 15% off the faster form, 0.2% on average).  That kernel / this
// one, us: Q4_K n_in 256, 1000 rows x 48 3.5 / 6.5, 8000 x 16 5.4 / 4.7; 512,
// 1000 x 32 3.6 / 6.1, 2000 x 48 7.3 / 6.1; 2048, 8000 x 2 5.7 / 8.3, 4000 x 3
// 4.8 / 5.4, 8000 x 3 9.3 / 8.4, 16,000 x 3 15.0 / 15.2, 4000 x 4 5.7 / 5.5,
// 2048 x 24 13.4 / 8.6; 4096, 100 x 48 5.0 / 16.9; Q6_K 512, 8000 x
// 2 4.2 / 6.0, 2048, 4000 x 3 6.9 / 6.5, x 4 8.4 / 6.3, 16,000 x 2 15.2 / 18.8.
bool mmf_supported(int nb, int n_out, int T, int wtype)
{
    const bool q4 = wtype == QMAG_TYPE_Q4_K;
    // 32-bit offsets within 16 rows; 512 threads per 16 rows in one grid
    if (T < (q4 ? 4 : 3) || nb > (1 << 18) || n_out >= (1 << 27)) return false;
    const double least = (q4 ? 14000 : 13000) * (T > 16 ? (q4 ? 2.0 : 1.6) : 1.0) * (nb < 5 ? 5.0 / nb : 1.0);
    return (double)n_out * T >= least;
}

int launch_mmf(const float *x, const void *W, int nb, int n_out, int T, int wtype, float *out, hipStream_t s)
{
    const uint8_t *w = (const uint8_t *)W;
    return wtype == QMAG_TYPE_Q4_K ? launch_mmf_t<QMAG_TYPE_Q4_K>(x, w, nb, n_out, T, out, s)
                                   : launch_mmf_t<QMAG_TYPE_Q6_K>(x, w, nb, n_out, T, out, s);
}

}  // namespace qmag
