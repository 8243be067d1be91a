// qmag_mm.hip -- the matmul seam (src/nn.c:307-345) for several tokens: Q4_K /
// Q6_K rows against Q8_K activations on the int8 matrix cores.
//
//   mm_split_kernel  16 rows x up to 64 tokens per workgroup, its waves
//                    splitting the row's super-blocks (few tokens or few rows:
//                    the work is spread over K to fill the chip)
//   mm_tile_kernel   128 rows x 64 tokens per workgroup, the activations of a
//                    super-block staged in LDS for its four waves
//
// Both fold the sub-block scale into the weight operand, as two int8 digits
// of the product q * scale, so that one MFMA chain per digit runs over a
// whole super-block and no scale is applied to partial results:
//   Q4_K  sc = 8 sh + sl (sl, sh in 0..7): q sl and q sh are at most 105
//   Q6_K  p = (q - 32) sc lies in +-4096: p = 256 hi + lo, both int8
// The two int32 chains, recombined, are the exact integer sum of the
// super-block (src/q8k.c): |sum| <= 256 * 4096 * 127 < 2^31.  Q4_K's min term
// sum_j m_j bsum_j is one f16 MFMA over the 16 sums of 16 values of Q8_K
// (xsum): |xsum| <= 2032 and m <= 63 are exact in f16, and every partial sum
// is an integer below 2^24, so its fp32 accumulator is exact as well.  The
// fp32 part per super-block and result is then xd * (d * S - dmin * M).
#include "qmag_internal.h"

namespace qmag {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// ------------------------------------------------------- weight operands --
// two 16-bit products per instruction; the operands' bytes are values of the
// low byte of each half (Q4_K: no product reaches 256, so four bytes at once)
__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b));
}
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) +
                                            __builtin_bit_cast(u16x2, c));
}

// the two digit operands of 16 Q4_K nibbles (already masked) of one sub-block
// of scale sc
__device__ __forceinline__ void q4_digits(const uint32_t (&n)[4], uint32_t sc, v4i &lo, v4i &hi)
{
    const uint32_t ml = (sc & 7) * 0x00010001u, mh = (sc >> 3) * 0x00010001u;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        lo[k] = (int)pk_mul(n[k], ml);
        hi[k] = (int)pk_mul(n[k], mh);
    }
}

// the two digit operands of 16 Q6_K values q in 0..63 of one group of scale
// sc: p + 128 = q sc + (128 - 32 sc) in 16 bits, hi its upper byte, lo its
// lower byte less 128
__device__ __forceinline__ void q6_digits(const uint32_t (&q)[4], int sc, v4i &lo, v4i &hi)
{
    const uint32_t m = ((uint32_t)sc & 0xffffu) * 0x00010001u;
    const uint32_t c = ((uint32_t)(128 - 32 * sc) & 0xffffu) * 0x00010001u;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t e = pk_mad(q[k] & 0x00ff00ffu, m, c), o = pk_mad((q[k] >> 8) & 0x00ff00ffu, m, c);
        lo[k] = (int)(__builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u);
        hi[k] = (int)__builtin_amdgcn_perm(o, e, 0x07030501u);
    }
}

// the 8 six-bit scales / mins of a Q4_K header, one per byte (src/q8k.c:22-30)
struct Q4Scales {
    uint32_t sc[2], m[2];
    __device__ __forceinline__ explicit Q4Scales(const uint4 &h)
    {
        sc[0] = h.y & 0x3F3F3F3Fu;
        m[0] = h.z & 0x3F3F3F3Fu;
        sc[1] = (h.w & 0x0F0F0F0Fu) | (((h.y >> 6) & 0x03030303u) << 4);
        m[1] = ((h.w >> 4) & 0x0F0F0F0Fu) | (((h.z >> 6) & 0x03030303u) << 4);
    }
};

// A wave's LDS image of one super-block of ROWS weight rows, row-major.  The
// bytes are requested in 16-byte pieces, neighbouring lanes taking a block's
// pieces in order, so that a request touches each cache line once: 16 or 32
// rows with one piece each re-fetch every line several times (a CU's L1 does
// not hold them), and a Q6_K block's pieces at 2-byte alignment cost about
// three times the issue time of dword-aligned ones (measured: 200 cycles a
// request against 64).  A Q6_K block is therefore read from the dword it
// starts in, 0 or 2 bytes ahead of it; its image starts as far in, and the
// reader shifts (misaligned 16-byte LDS reads instead cost 8-10% of the tile
// kernel).

// orders a wave's LDS accesses across its lanes (they execute in order; this
// holds the compiler to it)
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int WT, int ROWS>
struct WImage {
    static constexpr bool Q4 = WT == QMAG_TYPE_Q4_K, REP = WT == QMAG_TYPE_Q6_K_R;
    static constexpr int BLOCK = Q4 ? Q4K_BYTES : Q6K_BYTES, PIECES = Q4 ? 9 : 13;
    static constexpr int STRIDE = Q4 ? 144 : 240;      // 36 or 60 words: 16 rows' reads on distinct banks
    static constexpr int BYTES = ROWS * STRIDE, NP = ROWS * PIECES, WP = (NP + 63) / 64;
    const uint8_t *base, *row;      // the wave's first row (uniform), the lane's row lane % ROWS
    int nb, src[WP], dst[WP];
    uint4 v[WP];
    uint32_t tail;
    uint8_t *img;

    __device__ __forceinline__ void init(uint8_t *lds, const uint8_t *W, int row0, int n_out, int nb_)
    {
        img = lds;
        nb = nb_;
        const int first = min(row0, n_out - 1), rb = nb * BLOCK;
        base = W + (size_t)first * rb;
        row = base + (min(row0 + lane_id() % ROWS, n_out - 1) - first) * rb;
#pragma unroll
        for (int k = 0; k < WP; k++) {
            const int p = min(lane_id() + 64 * k, NP - 1), r = p / PIECES, j = p % PIECES;
            const int rel = (min(row0 + r, n_out - 1) - first) * rb;
            dst[k] = r * STRIDE + 16 * j;
            if constexpr (!REP) src[k] = rel + 16 * j;
            else if (j < 8) src[k] = rel + 64 * nb * ((j >> 1) & 1) + 16 * (2 * (j >> 2) + (j & 1));
            else src[k] = rel + (j < 12 ? 128 * nb + 16 * (j - 8) : 192 * nb);
        }
    }
    // bytes between the dword a block starts in and the block
    __device__ static __forceinline__ int lead(const uint8_t *blk)
    {
        return WT == QMAG_TYPE_Q6_K ? (int)((uintptr_t)blk & 2) : 0;
    }
    __device__ __forceinline__ void request(int k, int ib)
    {
        const uint32_t step = REP ? ((lane_id() + 64 * k) % PIECES < 12 ? 64u : 16u) : (uint32_t)BLOCK;
        const uint8_t *p = base + ((uint32_t)src[k] + (uint32_t)ib * step);
        v[k] = ld16(p - lead(p));
    }
    __device__ __forceinline__ void request_tail(int ib)
    {
        if constexpr (REP) {
            tail = ld2(row + 208 * nb + 2 * ib);
        } else if constexpr (!Q4) {
            const uint8_t *blk = row + ib * BLOCK;
            tail = ld2(blk + 208 - lead(blk)) | (ld2(blk + 208) << 16);
        }
    }
    __device__ __forceinline__ void request_all(int ib)
    {
#pragma unroll
        for (int k = 0; k < WP; k++) request(k, ib);
        request_tail(ib);
    }
    __device__ __forceinline__ void store()
    {
        wave_lds_order();                          // the reads of the block before
#pragma unroll
        for (int k = 0; k < WP; k++)
            if (64 * (k + 1) <= NP || lane_id() < NP - 64 * k) *(uint4 *)(img + dst[k]) = v[k];
        if constexpr (!Q4)
            if (lane_id() < ROWS) *(uint32_t *)(img + lane_id() * STRIDE + 208) = tail;
        wave_lds_order();
    }
    // the lane's row of the image, and the bits its block starts in
    __device__ __forceinline__ const uint8_t *block() const { return img + (lane_id() % ROWS) * STRIDE; }
    __device__ __forceinline__ uint32_t shift(int ib) const { return 8 * (uint32_t)lead(row + ib * BLOCK); }
};

// A super-block's operands from the lane's row in the image: L lanes share a
// row (4: 16 rows, 16x16x64 MFMAs, q = lane / 16; 2: 32 rows, 32x32x32, h =
// lane / 32), each taking 16 consecutive values of one scale per step; koff(s)
// is its first value of step s.
template <int WT, int L>
struct WRow;

template <int L>
struct WRow<QMAG_TYPE_Q4_K, L> {
    static constexpr int SHIFT = 3, STEPS = 16 / L;
    static constexpr bool MIN = true;
    const uint8_t *b;
    uint32_t dd;
    Q4Scales S;
    struct Raw {
        uint4 v;
    };
    __device__ __forceinline__ WRow(const uint8_t *blk, uint32_t) : b(blk), dd(*(const uint32_t *)blk), S(*(const uint4 *)blk) {}
    // step s = 2 g + up: the low (up = 0) or high nibbles of 16 bytes of the
    // 32-byte group G = g (L = 2) or 2 g + (q >> 1) (L = 4), half c
    __device__ static __forceinline__ int group(int s) { return L == 2 ? s >> 1 : 2 * (s >> 1) + (lane_id() >> 5); }
    __device__ static __forceinline__ int half() { return L == 2 ? lane_id() >> 5 : (lane_id() >> 4) & 1; }
    __device__ static __forceinline__ int koff(int s) { return 64 * group(s) + 32 * (s & 1) + 16 * half(); }
    __device__ __forceinline__ void read(int s, Raw &r) const
    {
        if ((s & 1) == 0) r.v = *(const uint4 *)(b + 16 + 32 * group(s) + 16 * half());
    }
    __device__ __forceinline__ void operands(const Raw &r, int s, v4i &lo, v4i &hi) const
    {
        const int up = s & 1;
        const uint32_t n[4] = {(up ? r.v.x >> 4 : r.v.x) & 0x0F0F0F0Fu, (up ? r.v.y >> 4 : r.v.y) & 0x0F0F0F0Fu,
                               (up ? r.v.z >> 4 : r.v.z) & 0x0F0F0F0Fu, (up ? r.v.w >> 4 : r.v.w) & 0x0F0F0F0Fu};
        // sub-block 2 G + up
        const uint32_t sc = L == 2 ? S.sc[s >> 2] >> (8 * (s & 3)) : S.sc[s >> 1] >> (8 * (2 * (lane_id() >> 5) + up));
        q4_digits(n, sc & 63, lo, hi);
    }
    // mins of the lane's 16-value groups: 4 q .. 4 q + 3, or 8 h .. 8 h + 7
    __device__ __forceinline__ v4h mins4() const
    {
        const int q = lane_id() >> 4;
        const uint32_t w = (q >> 1 ? S.m[1] : S.m[0]) >> (16 * (q & 1));
        const _Float16 a = (_Float16)(uint16_t)(w & 63), c = (_Float16)(uint16_t)((w >> 8) & 63);
        return v4h{a, a, c, c};
    }
    __device__ __forceinline__ v8h mins8() const
    {
        const uint32_t w = lane_id() >> 5 ? S.m[1] : S.m[0];
        v8h o;
#pragma unroll
        for (int j = 0; j < 4; j++) o[2 * j] = o[2 * j + 1] = (_Float16)(uint16_t)((w >> (8 * j)) & 63);
        return o;
    }
    __device__ __forceinline__ float d() const { return h2f(dd & 0xffff); }
    __device__ __forceinline__ float dmin() const { return h2f(dd >> 16); }
};

template <int L, bool SHIFTED>
struct WQ6 {
    static constexpr int SHIFT = 8, STEPS = 16 / L;
    static constexpr bool MIN = false;
    const uint8_t *b;
    uint32_t sh0;                              // the block starts this many bits into the image
    uint4 sc;
    uint32_t db;
    struct Raw {
        uint4 l[2], h;
    };
    __device__ __forceinline__ uint4 lds16(int o) const
    {
        const uint4 v = *(const uint4 *)(b + o);
        if constexpr (!SHIFTED) return v;
        const uint32_t n = *(const uint32_t *)(b + o + 16);
        return make_uint4(__builtin_amdgcn_alignbit(v.y, v.x, sh0), __builtin_amdgcn_alignbit(v.z, v.y, sh0),
                          __builtin_amdgcn_alignbit(v.w, v.z, sh0), __builtin_amdgcn_alignbit(n, v.w, sh0));
    }
    __device__ __forceinline__ WQ6(const uint8_t *blk, uint32_t shift)
        : b(blk), sh0(shift), sc(lds16(192)), db((*(const uint32_t *)(blk + 208) >> shift) & 0xffff)
    {
    }
    // L = 2: step s = 4 n + Q, quarter Q of half n, values 16 h ..; L = 4: step
    // s = 2 n + up, quarter Q = (q >> 1) + 2 up, values 16 (q & 1) ..
    // (src/quants.c:56-69); scale 8 n + 2 Q + half
    __device__ static __forceinline__ int half() { return L == 2 ? lane_id() >> 5 : (lane_id() >> 4) & 1; }
    __device__ static __forceinline__ int koff(int s)
    {
        if constexpr (L == 2) return 32 * s + 16 * half();
        return 128 * (s >> 1) + 32 * ((lane_id() >> 5) + 2 * (s & 1)) + 16 * half();
    }
    __device__ __forceinline__ void read(int s, Raw &r) const
    {
        if constexpr (L == 2) {
            const int n = s >> 2, Q = s & 3;
            if (Q < 2) r.l[Q] = lds16(64 * n + 32 * Q + 16 * half());
            if (Q == 0) r.h = lds16(128 + 32 * n + 16 * half());
        } else if ((s & 1) == 0) {
            r.l[0] = lds16(32 * s + 16 * (lane_id() >> 4));
            r.h = lds16(128 + 16 * s + 16 * half());
        }
    }
    __device__ __forceinline__ void operands(const Raw &r, int s, v4i &lo, v4i &hi) const
    {
        const uint4 l = L == 2 ? r.l[s & 1] : r.l[0];
        const uint32_t lw[4] = {l.x, l.y, l.z, l.w}, hw[4] = {r.h.x, r.h.y, r.h.z, r.h.w};
        const bool up = L == 2 ? (s & 2) != 0 : (s & 1) != 0;
        const uint32_t sh = L == 2 ? 2u * (uint32_t)(s & 3) : 2u * (uint32_t)((lane_id() >> 5) + 2 * (s & 1));
        uint32_t q[4];
#pragma unroll
        for (int k = 0; k < 4; k++)
            q[k] = ((up ? lw[k] >> 4 : lw[k]) & 0x0F0F0F0Fu) | (((hw[k] >> sh) & 0x03030303u) << 4);
        const uint32_t w[4] = {sc.x, sc.y, sc.z, sc.w};
        const int si = L == 2 ? (int)(int8_t)(w[s >> 1] >> (16 * (s & 1) + 8 * half()))
                              : (int)(int8_t)(w[s] >> (8 * (lane_id() >> 4)));
        q6_digits(q, si, lo, hi);
    }
    __device__ __forceinline__ float d() const { return h2f(db); }
};
template <int L>
struct WRow<QMAG_TYPE_Q6_K, L> : WQ6<L, true> {
    using WQ6<L, true>::WQ6;
};
template <int L>
struct WRow<QMAG_TYPE_Q6_K_R, L> : WQ6<L, false> {
    using WQ6<L, false>::WQ6;
};

// four int16 group sums as f16
__device__ __forceinline__ v4h sums_f16(uint2 s)
{
    return v4h{(_Float16)(int16_t)(s.x & 0xffff), (_Float16)(int16_t)(s.x >> 16), (_Float16)(int16_t)(s.y & 0xffff),
               (_Float16)(int16_t)(s.y >> 16)};
}

// ------------------------------------------------------------ split over K --
// grid: rows / 16 x tokens / (16 MT); wave w of the workgroup's W takes
// super-blocks w, w + W, ... of the 16 rows against all its tokens, reading
// the activations straight from memory (the workgroup's waves share none),
// and the W partial results are added through LDS.
template <int WT, int MT>
__global__ __launch_bounds__(512) void mm_split_kernel(const uint8_t *__restrict__ W, const int8_t *__restrict__ xq,
                                                       const float *__restrict__ xd,
                                                       const int16_t *__restrict__ xsum, float *__restrict__ out,
                                                       int nb, int n_out, int T)
{
    using Row = WRow<WT, 4>;
    // [waves]: a weight image each, then (the same bytes) [MT][4][64] partials
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
    }
    __syncthreads();                           // every wave is done with its image
    float *s_part = (float *)s_dyn;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int i = 0; i < 4; i++) s_part[((wv * MT + m) * 4 + i) * 64 + lane] = r[m][i];
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
// finds them there.  Wave w: rows 32 w .. 32 w + 31 against both 32-token
// tiles.  Per super-block the 64 Q8_K rows go through registers into one of
// two LDS buffers while the other is consumed, and the next weight block is
// requested into a second register set: one barrier per super-block.
constexpr int MMT = 64, MMR = 128;
constexpr int MM_ROW = QK_K + 16;          // padded LDS row: 16 rows of a read start 4 banks apart

template <int WT>
__global__ __launch_bounds__(256, 2) void mm_tile_kernel(const uint8_t *__restrict__ W,
                                                         const int8_t *__restrict__ xq,
                                                         const float *__restrict__ xd,
                                                         const int16_t *__restrict__ xsum, float *__restrict__ out,
                                                         int nb, int n_out, int T)
{
    using Row = WRow<WT, 2>;
    using Img = WImage<WT, 32>;
    __shared__ __align__(16) int8_t s_a[2][MMT * MM_ROW];
    __shared__ __align__(16) uint8_t s_w[4 * Img::BYTES];
    __shared__ __align__(16) float s_d[2][MMT];
    __shared__ __align__(16) _Float16 s_s[2][Row::MIN ? MMT * 16 : 8];
    const int tid = (int)threadIdx.x, lane = lane_id(), lr = lane & 31, h = lane >> 5, wv = tid >> 6;
    const int row0 = (int)blockIdx.x * MMR + 32 * wv, t0 = (int)blockIdx.y * MMT;
    Img img;
    img.init(s_w + wv * Img::BYTES, W, row0, n_out, nb);

    // staging: thread -> 16-byte piece tid % 16 of tokens tid / 16 + 16 k; scale of token tid; half
    // of token tid / 2's 16 sums
    const int8_t *xp[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        xp[k] = xq + (size_t)min(t0 + (tid >> 4) + 16 * k, T - 1) * nb * QK_K + 16 * (tid & 15);
    const float *dp = xd + (size_t)min(t0 + (tid & 63), T - 1) * nb;
    const int16_t *sp = xsum + (size_t)min(t0 + ((tid & 127) >> 1), T - 1) * nb * 16 + 8 * (tid & 1);
    uint4 va[4], vs = make_uint4(0, 0, 0, 0);
    float vd = 0.0f;
    auto stage_load = [&](int ib) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 4; k++) va[k] = ld16((const uint8_t *)xp[k] + (size_t)ib * QK_K);
        if (tid < 64) vd = ldg(dp + ib);
        if (Row::MIN && tid < 128) vs = ld16((const uint8_t *)(sp + (size_t)ib * 16));
    };
    auto stage_store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 4; k++)
            *(uint4 *)(s_a[buf] + ((tid >> 4) + 16 * k) * MM_ROW + 16 * (tid & 15)) = va[k];
        if (tid < 64) s_d[buf][tid] = vd;
        if (Row::MIN && tid < 128) {
            const v4h a = sums_f16(make_uint2(vs.x, vs.y)), b = sums_f16(make_uint2(vs.z, vs.w));
            *(v8h *)(s_s[buf] + 8 * tid) = v8h{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        }
    };

    // the eighth part s of block ib's requests
    auto request = [&](int s, int ib) __attribute__((always_inline)) {
        if (s < Img::WP) img.request(s, ib);
        if (s == 7) img.request_tail(ib);
        if (s < 4) va[s] = ld16((const uint8_t *)xp[s] + (size_t)ib * QK_K);
        if (s == 5 && tid < 64) vd = ldg(dp + ib);
        if (Row::MIN && s == 6 && tid < 128) vs = ld16((const uint8_t *)(sp + (size_t)ib * 16));
    };
    v16f r[2], tot[2];
#pragma unroll
    for (int i = 0; i < 16; i++) r[0][i] = r[1][i] = tot[0][i] = tot[1][i] = 0.0f;
    img.request_all(0);
    stage_load(0);
    img.store();
    stage_store(0);
    __syncthreads();
    for (int ib = 0; ib < nb; ib++) {
        const int buf = ib & 1, nx = min(ib + 1, nb - 1);
        const Row w(img.block(), img.shift(ib));
        const int8_t *pa = s_a[buf] + lr * MM_ROW + 16 * h;
        v16i lo[2], hi[2];
        v16f mn[2];
#pragma unroll
        for (int i = 0; i < 16; i++) lo[0][i] = lo[1][i] = hi[0][i] = hi[1][i] = 0;
        const float d = w.d();
        float nm = 0.0f;
        // Step by step: the next step's LDS reads, a share of the next
        // super-block's requests (all at once they hold the wave for the time
        // the address unit takes to accept them), this step's four MFMAs, and
        // the next step's operands while those run.
        auto mma = [&](auto build) __attribute__((always_inline)) {
            typename Row::Raw raw;
            v4i bl[2], bh[2], a[2][2];
            w.read(0, raw);
            a[0][0] = *(const v4i *)pa;
            a[0][1] = *(const v4i *)(pa + 32 * MM_ROW);
            build(raw, 0, bl[0], bh[0]);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const int c = s & 1, n = c ^ 1;
                if (s < 7) {
                    w.read(s + 1, raw);
                    a[n][0] = *(const v4i *)(pa + 32 * (s + 1));
                    a[n][1] = *(const v4i *)(pa + 32 * MM_ROW + 32 * (s + 1));
                }
                request(s, nx);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < 2; m++) {
                    lo[m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[c][m], bl[c], lo[m], 0, 0, 0);
                    hi[m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[c][m], bh[c], hi[m], 0, 0, 0);
                }
                if (s < 7) build(raw, s + 1, bl[n], bh[n]);
                for (int i = 0; i < 4; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, Row::MIN ? 6 : 13, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if constexpr (Row::MIN) {
            nm = -w.dmin();
            const v8h mb = w.mins8();
#pragma unroll
            for (int m = 0; m < 2; m++) {
                v16f z;
#pragma unroll
                for (int i = 0; i < 16; i++) z[i] = 0.0f;
                mn[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const v8h *)(s_s[buf] + (32 * m + lr) * 16 + 8 * h),
                                                               mb, z, 0, 0, 0);
            }
        }
        mma([&](const typename Row::Raw &r, int s, v4i &bl, v4i &bh) __attribute__((always_inline)) { w.operands(r, s, bl, bh); });
        // result i of a lane: token 8 (i / 4) + 4 h + i % 4 of the tile, row lr
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float4 x4 = *(const float4 *)(s_d[buf] + 32 * m + 8 * g + 4 * h);
                const float xv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int i = 4 * g + k;
                    float v = d * (float)(lo[m][i] + (hi[m][i] << Row::SHIFT));
                    if constexpr (Row::MIN) v = fmaf(nm, mn[m][i], v);
                    r[m][i] = fmaf(xv[k], v, r[m][i]);
                }
            }
        if constexpr (!Row::MIN) {
            // sums of eight super-blocks are added up apart: one running sum
            // over a long row would round more than the matvec's lane tree
            // (n_in 8192: 1.07e-7 of the result against 7.4e-8)
            if ((ib & 7) == 7)
#pragma unroll
                for (int m = 0; m < 2; m++) {
                    tot[m] += r[m];
#pragma unroll
                    for (int i = 0; i < 16; i++) r[m][i] = 0.0f;
                }
        }
        img.store();                           // the wave's own image: its reads are done
        stage_store(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = t0 + 32 * m + 8 * (i >> 2) + 4 * h + (i & 3);
            if (t < T && row0 + lr < n_out) out[(size_t)t * n_out + row0 + lr] = Row::MIN ? r[m][i] : tot[m][i] + r[m][i];
        }
}

// ------------------------------------------------------------------- host --
// The split kernel fills the chip with few tiles, the tile kernel shares the
// activations and builds each weight operand for 64 tokens instead of 16 MT
// per wave.  Measured around the lines drawn here (n_in 2048, us per call with
// the quantisation, split / tile): Q4_K 32 tiles 9.2 / 16.4, 64 tiles 18.2 /
// 17.6, 128 tiles 30 / 17.9, 512 tiles 99 / 30.8; Q6_K 64 tiles 17.3 / 23.4,
// 128 tiles 28 / 23.7, 512 tiles 94 / 38.
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
    if ((long)rt * tt >= (WT == QMAG_TYPE_Q4_K ? MM_TILES_Q4 : MM_TILES_Q6) && tt <= 65535) {
        hipLaunchKernelGGL(mm_tile_kernel<WT>, dim3(rt, tt), dim3(256), 0, s, w, xq, xd, xsum, out, nb, n_out, T);
    } else {
        const int mt = T > 48 ? 4 : (T + 15) / 16;
        const dim3 grid((n_out + 15) / 16, (T + 16 * mt - 1) / (16 * mt));
        const int most = (long)grid.x * grid.y >= MM_SPLIT8_WGS ? 4 : 8;
        int nw = 1;
        while (nw < most && nw < nb) nw *= 2;
        const size_t part = sizeof(float) * 256 * (size_t)mt, image = WImage<WT, 16>::BYTES;
        const size_t lds = (size_t)nw * (part > image ? part : image);
        const dim3 wg(64 * nw);
        switch (mt) {
        case 1: hipLaunchKernelGGL((mm_split_kernel<WT, 1>), grid, wg, lds, s, w, xq, xd, xsum, out, nb, n_out, T); break;
        case 2: hipLaunchKernelGGL((mm_split_kernel<WT, 2>), grid, wg, lds, s, w, xq, xd, xsum, out, nb, n_out, T); break;
        case 3: hipLaunchKernelGGL((mm_split_kernel<WT, 3>), grid, wg, lds, s, w, xq, xd, xsum, out, nb, n_out, T); break;
        default: hipLaunchKernelGGL((mm_split_kernel<WT, 4>), grid, wg, lds, s, w, xq, xd, xsum, out, nb, n_out, T); break;
        }
    }
    QMAG_HIP(hipGetLastError());
    return QMAG_OK;
}

// The matvec kernels take a few tokens faster (they read the rows once and
// loop over the tokens): Q4_K at 3 tokens 9.6 against 9.3 us (16,384 rows) and
// 8.2 against 8.4 (n_in 8192), at 4 59.9 against 44.5 (151,936 rows); Q6_K at
// 3 10.5 against 11.4, at 6 13.5 against 11.4, and rows beyond 4096 values at
// 5 9.4 against 11.8, at 12 14.1 against 11.9.  They also take what this path
// does not: Q6_K rows that do not start on 4 bytes, rows beyond 2^26 values
// (32-bit offsets within 32 rows) and more tokens than a grid holds.
bool mm_supported(int nb, int T, int wtype, const void *W)
{
    if (nb > (1 << 18) || T > 16 * 65535) return false;
    if (wtype == QMAG_TYPE_Q4_K) return T >= 4;
    return T >= (nb > 16 ? 9 : 6) && ((uintptr_t)W & 3) == 0;
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
