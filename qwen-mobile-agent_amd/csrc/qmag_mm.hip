// qmag_mm.hip -- the matmul seam (src/nn.c:307-345) for several tokens: Q4_K /
// Q6_K rows against Q8_K activations on the int8 matrix cores.
//
//   mm_split_kernel  16 rows x up to 64 tokens per workgroup, its waves
//                    splitting the row's super-blocks (few tokens or few rows:
//                    the work is spread over K to fill the chip)
//   mm_tile_kernel   128 rows x 64 tokens per workgroup, the activations of a
//                    super-block staged in LDS for its four waves
//
// The operands, their exactness and the tile loop: qmag_mfma.h.
#include "qmag_mfma.h"

namespace qmag {

// ------------------------------------------------------------ split over K --
// grid: rows / 16 x tokens / (16 MT); wave w of the workgroup's W takes
// super-blocks w, w + W, ... of the 16 rows against all its tokens, reading
// the activations straight from memory (the workgroup's waves share none),
// and the W partial results are added through LDS.
//
// Chains of eight super-blocks per wave and sum (n_in 32,768 over 8 waves and
// 262,144 over 8, against 64 bits: Q4_K 1.06e-7 and 2.22e-7 in one sum, 9.7e-8
// and 1.18e-7 in chains, the matvec's lane tree 1.39e-7 and 1.91e-7; Q6_K
// 9.5e-8 and 2.05e-7, 8.3e-8 and 1.06e-7, tree 8.9e-8 and 1.51e-7).
constexpr int SPLIT_CHAIN = 8;
template <int WT, int MT, bool LNG>            // LNG: long rows (put_partials)
__global__ __launch_bounds__(512) void mm_split_kernel(const uint8_t *__restrict__ W, const int8_t *__restrict__ xq,
                                                       const float *__restrict__ xd,
                                                       const int16_t *__restrict__ xsum, float *__restrict__ out,
                                                       int nb, int n_out, int T)
{
    using Row = WRow<WT, 4>;
    // an image per wave, and the partials (split_lds)
    extern __shared__ __align__(16) uint8_t s_dyn[];
    const int lane = lane_id(), lr = lane & 15, q = lane >> 4;
    const int wv = (int)(threadIdx.x >> 6), nw = (int)(blockDim.x >> 6);
    const int row0 = (int)blockIdx.x * 16, t0 = (int)blockIdx.y * 16 * MT;
    WImage<WT, 16> img;
    img.init(s_dyn + wv * img.BYTES, W, row0, n_out, nb);
    size_t tok[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) tok[m] = (size_t)min(t0 + 16 * m + lr, T - 1) * nb;
    float r[MT][4] = {};
    float *s_part = (float *)(s_dyn + (LNG ? nw * img.BYTES : 0));
    int done = 0;
    if (wv < nb) img.request_all(wv);          // wave-uniform
    for (int ib = wv; ib < nb; ib += nw) {
        v4i a[MT][4];
        float xdl[MT];
        uint2 xs[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) {
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const uint4 v = ld16((const uint8_t *)xq + (tok[m] + ib) * QK_K + Row::koff(s));
                a[m][s] = v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
            }
            xdl[m] = ldg(xd + tok[m] + ib);
            if constexpr (Row::MIN) xs[m] = ld8((const uint8_t *)xsum + (tok[m] + ib) * 32 + 8 * q);
        }
        img.store();
        const Row w(img.block(), img.shift(ib));
        typename Row::Raw raw[4];
#pragma unroll
        for (int s = 0; s < 4; s++) w.read(s, raw[s & ~1]);
        if (ib + nw < nb) img.request_all(ib + nw);
        v4i lo[MT], hi[MT];
        v4f mn[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) {
            lo[m] = hi[m] = v4i{0, 0, 0, 0};
            if constexpr (Row::MIN)
                mn[m] = __builtin_amdgcn_mfma_f32_16x16x16f16(sums_f16(xs[m]), w.mins4(), v4f{0.f, 0.f, 0.f, 0.f}, 0,
                                                              0, 0);
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
            v4i bl, bh;
            w.operands(raw[s & ~1], s, bl, bh);
#pragma unroll
            for (int m = 0; m < MT; m++) {
                lo[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[m][s], bl, lo[m], 0, 0, 0);
                hi[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[m][s], bh, hi[m], 0, 0, 0);
            }
        }
        // result i of a lane: token 4 q + i of the tile, row lr; the token's
        // scale sits in lane 4 q + i
        const float d = w.d();
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float xdi = __shfl(xdl[m], 4 * q + i);
                float v = d * (float)(lo[m][i] + (hi[m][i] << Row::SHIFT));
                if constexpr (Row::MIN) v = fmaf(-w.dmin(), mn[m][i], v);
                r[m][i] = fmaf(xdi, v, r[m][i]);
            }
        if constexpr (LNG)
            if (++done % SPLIT_CHAIN == 0) put_partials<MT>(s_part, wv, r, done > SPLIT_CHAIN);
    }
    __syncthreads();                           // every wave is done with its image
    put_partials<MT>(s_part, wv, r, LNG);   // of long rows every wave has a whole chain there
    __syncthreads();
    for (int k = (int)threadIdx.x; k < MT * 256; k += (int)blockDim.x) {
        // the waves' partials pairwise (as accurate as the matvec's lane tree)
        float p[8];
#pragma unroll
        for (int u = 0; u < 8; u++) p[u] = u < nw ? s_part[u * MT * 256 + k] : 0.0f;
        const float v = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        const int l = k & 63, i = (k >> 6) & 3, m = k >> 8;
        const int t = t0 + 16 * m + 4 * (l >> 4) + i, rw = row0 + (l & 15);
        if (t < T && rw < n_out) out[(size_t)t * n_out + rw] = v;
    }
}

// ------------------------------------------------------------------- tiles --
// grid: rows / 128 x tokens / 64, rows fastest: workgroup i runs on XCD i % 8,
// so each XCD's L2 holds an eighth of the weight rows and every token block
// finds them there.  What bounds it is instruction issue: per 32 rows x 64
// tokens x super-block 34 MFMAs (1,100 cycles) and 390 (Q4_K) or 600 (Q6_K)
// VALU instructions, a third of them the operands, most of the rest the fp32
// part; two waves per SIMD overlap these only in part (2048 -> 8192 x 512
// tokens: 28.4 us, MFMA busy 39% and VALU 60% of the waves' time; the token
// loop before took 280).
//
// One launch takes up to MM_CHAIN super-blocks of the rows and adds to out
// behind the first: sums of eight super-blocks, added up over any longer row,
// would round more than the matvec's lane tree again (n_in 32,768 against 64
// bits: Q6_K 9.8e-8, the tree 8.8e-8, in launches of 32 super-blocks 8.4e-8;
// Q4_K, in one sum 2.13e-7, the tree 1.39e-7, in launches of 64 1.04e-7).
constexpr int MMT = 64, MMR = 128;
template <int WT>
constexpr int MM_CHAIN = WT == QMAG_TYPE_Q4_K ? 64 : 32;

template <int WT>
__global__ __launch_bounds__(256, 2) void mm_tile_kernel(const uint8_t *__restrict__ W,
                                                         const int8_t *__restrict__ xq,
                                                         const float *__restrict__ xd,
                                                         const int16_t *__restrict__ xsum, float *__restrict__ out,
                                                         int nb, int n_out, int T, int ib0)
{
    using Img = WImage<WT, 32>;
    __shared__ __align__(16) TileLds s_t;
    __shared__ __align__(16) uint8_t s_w[4 * Img::BYTES];
    const int lane = lane_id(), lr = lane & 31, h = lane >> 5;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));        // uniform, and known to be
    const int row0 = (int)blockIdx.x * MMR + 32 * wv, t0 = (int)blockIdx.y * MMT;
    Img img;
    img.init(s_w + wv * Img::BYTES, W, row0, n_out, nb);
    img.request_all(ib0);
    TileSrc src;
    const size_t b0 = (size_t)t0 * nb;
    src.init(xq + b0 * QK_K, xd + b0, xsum + b0 * 16, nb, T - 1 - t0);
    v16f r[NT];
    tile_products<WT>(img, ib0, min(ib0 + MM_CHAIN<WT>, nb), src, s_t, r);
    // result i of group m: token t0 + at(m, i), weight row row0 + lr
    auto at = [&](int m, int i) { return 32 * m + 8 * (i >> 2) + 4 * h + (i & 3); };
    float *o = out + (size_t)t0 * n_out + row0 + lr;
    const int tn = row0 + lr < n_out ? T - t0 : 0;         // tokens to write
    if (ib0)
#pragma unroll
        for (int m = 0; m < NT; m++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (at(m, i) < tn) r[m][i] += o[(size_t)at(m, i) * n_out];
#pragma unroll
    for (int m = 0; m < NT; m++)
#pragma unroll
        for (int i = 0; i < 16; i++)
            if (at(m, i) < tn) o[(size_t)at(m, i) * n_out] = r[m][i];
}

// ------------------------------------------------------------------- host --
// The split kernel's time grows with rows x tokens (in steps of 16 tokens); the
// tile kernel builds each weight operand once for 64 tokens, however many there
// are.  So it takes over from MM_TILES tiles on, counted by their tokens where
// there is one row of tiles, and never at 16 tokens or fewer.  Split / tile, us with the quantisation: Q4_K
// 2048 -> 8192 x 64 tokens 17.5 / 17.3 (the line), 16,384 x 32 17.7 / 17.6, x
// 9 9.2 / 17.3, 151,936 x 4 44 / 64, x 16 67 / 65, x 24 96 / 67; 4096 -> 16,384
// x 32 28.6 / 29.4, x 48 39.8 / 29.7; Q6_K 2048 -> 16,384 x 48 22.5 / 22.9, x
// 64 28.0 / 23.2, 49,152 x 16 25.7 / 33.3, x 24 36.5 / 33.5; 8192 -> 16,384 x 48
// 72.3 / 72.4; more than 64 tokens: Q4_K 2048 -> 6000 x 70 18.5 / 17.1, 4096 x 100
// 15.6 / 17.0, 1000 x 460 20.4 / 18.3.
constexpr long MM_TILES_Q4 = 64, MM_TILES_Q6 = 112;
// Waves a row's super-blocks are split over: 8, and 4 once 512 workgroups
// queue (151,936 rows x 4 tokens 44.5 against 49.9 us; 128 workgroups of 8,192
// values 13.1 against 8.4).
constexpr long MM_SPLIT8_WGS = 512;

template <int WT>
static int launch_mm_t(const int8_t *xq, const float *xd, const int16_t *xsum, const void *W, int nb, int n_out,
                       int T, float *out, hipStream_t s)
{
    const uint8_t *w = (const uint8_t *)W;
    const int rt = (n_out + MMR - 1) / MMR, tt = (T + MMT - 1) / MMT;
    const long tiles = WT == QMAG_TYPE_Q4_K ? MM_TILES_Q4 : MM_TILES_Q6;
    const bool fill = tt > 1 ? (long)rt * tt >= tiles : T > 16 && (long)n_out * T >= tiles * MMR * MMT;
    if (fill || n_out >= (1 << 27)) {          // a grid of the split kernel holds fewer rows
        for (int ib0 = 0; ib0 < nb; ib0 += MM_CHAIN<WT>)
            hipLaunchKernelGGL(mm_tile_kernel<WT>, dim3(rt, tt), dim3(256), 0, s, w, xq, xd, xsum, out, nb, n_out, T,
                               ib0);
    } else {
        const int mt = T > 48 ? 4 : (T + 15) / 16;
        const dim3 grid((n_out + 15) / 16, (T + 16 * mt - 1) / (16 * mt));
        const int most = (long)grid.x * grid.y >= MM_SPLIT8_WGS ? 4 : 8;
        int nw = 1;
        while (nw < most && nw < nb) nw *= 2;
        const size_t lds = split_lds(nb, nw, SPLIT_CHAIN, mt, WImage<WT, 16>::BYTES);
        const dim3 wg(64 * nw);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, wg, lds, s, w, xq, xd, xsum, out, nb, n_out, T);
        };
        const bool lng = long_row(nb, nw, SPLIT_CHAIN);
        switch (mt) {
        case 1: launch(lng ? mm_split_kernel<WT, 1, true> : mm_split_kernel<WT, 1, false>); break;
        case 2: launch(lng ? mm_split_kernel<WT, 2, true> : mm_split_kernel<WT, 2, false>); break;
        case 3: launch(lng ? mm_split_kernel<WT, 3, true> : mm_split_kernel<WT, 3, false>); break;
        default: launch(lng ? mm_split_kernel<WT, 4, true> : mm_split_kernel<WT, 4, false>); break;
        }
    }
    QMAG_HIP(hipGetLastError());
    return QMAG_OK;
}

// The matvec kernels take a few tokens faster (they read the rows once and
// loop over the tokens): Q4_K at 3 tokens 9.6 against 9.3 us (16,384 rows) and
// 8.2 against 8.4 (n_in 8192), at 4 59.9 against 44.5 (151,936 rows); Q6_K at
// 3 10.5 against 11.4, at 6 13.5 against 11.4, and rows beyond 4096 values at
// 5 9.4 against 11.8, at 12 14.1 against 11.9.  One row is no different (2048
// values: 4 tokens level, 64 35.3 against 10.2).  They also take what this path
// does not: rows beyond 2^26 values (32-bit offsets within 32 rows) and more
// tokens than a grid holds.
bool mm_supported(int nb, int T, int wtype)
{
    if (nb > (1 << 18) || T > 16 * 65535) return false;
    if (wtype == QMAG_TYPE_Q4_K) return T >= 4;
    return T >= (nb > 16 ? 9 : 6);
}

int launch_mm(const int8_t *xq, const float *xd, const int16_t *xsum, const void *W, int nb, int n_out, int T,
              int wtype, float *out, hipStream_t s)
{
    prof_begin(PROF_MATVEC, s);
    int st;
    if (wtype == QMAG_TYPE_Q4_K) st = launch_mm_t<QMAG_TYPE_Q4_K>(xq, xd, xsum, W, nb, n_out, T, out, s);
    else if (wtype == QMAG_TYPE_Q6_K) st = launch_mm_t<QMAG_TYPE_Q6_K>(xq, xd, xsum, W, nb, n_out, T, out, s);
    else st = launch_mm_t<QMAG_TYPE_Q6_K_R>(xq, xd, xsum, W, nb, n_out, T, out, s);
    prof_end(PROF_MATVEC, s);
    return st;
}

}  // namespace qmag
