// qmag_mfma.h -- Q4_K / Q6_K rows x Q8_K activations on the int8 matrix cores:
// the weight operands, the LDS image they are built from, and the 32-row x
// 64-token product loop of the matmul.
//
// The sub-block scale is folded into the weight operand, as two int8 digits
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
#pragma once

#include "qmag_internal.h"
#include "qmag_wimage.h"

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
// the two digit operands of 16 Q4_K nibbles (already masked) of one sub-block,
// its scale's digits sl, sh in both halves of ml, mh
__device__ __forceinline__ void q4_digits(const uint32_t (&n)[4], uint32_t ml, uint32_t mh, v4i &lo, v4i &hi)
{
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
    const unsigned short ms = (unsigned short)sc, cs = (unsigned short)(128 - 32 * sc);
    const u16x2 m = {ms, ms}, c = {cs, cs};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t e = __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, q[k] & 0x00ff00ffu) * m + c);
        const uint32_t o = __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, (q[k] >> 8) & 0x00ff00ffu) * m + c);
        lo[k] = (int)(__builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u);
        hi[k] = (int)__builtin_amdgcn_perm(o, e, 0x07030501u);
    }
}

// the 8 six-bit scales / mins of a Q4_K header, one per byte (src/q8k.c:22-30)
// the scales as their two digits
struct Q4Scales {
    uint32_t sl[2], sh[2], m[2];
    __device__ __forceinline__ explicit Q4Scales(const uint4 &h)
    {
        const uint32_t s0 = h.y & 0x3F3F3F3Fu, s1 = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
        sl[0] = s0 & 0x07070707u;
        sl[1] = s1 & 0x07070707u;
        sh[0] = (s0 >> 3) & 0x07070707u;
        sh[1] = (s1 >> 3) & 0x07070707u;
        m[0] = h.z & 0x3F3F3F3Fu;
        m[1] = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
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
// kernel).  Every address is WImageMap's (qmag_wimage.h).

// orders a wave's LDS accesses across its lanes (they execute in order; this
// holds the compiler to it)
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int WT, int ROWS>
struct WImage : WImageMap<WT, ROWS> {
    using M = WImageMap<WT, ROWS>;
    using M::BLOCK, M::BYTES, M::lead, M::NP, M::PIECES, M::Q4, M::REP, M::STRIDE, M::WP;
    const uint8_t *base;                // the dword that the wave's first row starts in (uniform)
    uint32_t row;                       // from there, the lane's row lane % ROWS
    int nb;
    uint32_t src[WP];
    int dst[WP];
    uint4 v[WP];
    uint32_t tail;
    uint8_t *img;

    __device__ __forceinline__ void init(uint8_t *lds, const uint8_t *W, int row0, int n_out, int nb_)
    {
        img = lds;
        nb = nb_;
        const int first = M::row(0, row0, n_out), rb = nb * BLOCK;
        const uint32_t skew = M::skew(first, rb);
        base = W + (size_t)first * rb - skew;
        row = skew + (uint32_t)M::row_off(lane_id() % ROWS, row0, n_out, rb);
#pragma unroll
        for (int k = 0; k < WP; k++) {
            const int p = M::piece(lane_id(), k), r = p / PIECES, j = p % PIECES;
            const int rel = M::row_off(r, row0, n_out, rb);
            dst[k] = M::dst(r, j);
            src[k] = skew + (uint32_t)(rel + M::src(j, nb));
        }
    }
    __device__ __forceinline__ void request(int k, int ib)
    {
        v[k] = ld16(base + M::from(src[k], ib, M::piece(lane_id(), k) % PIECES));
    }
    __device__ __forceinline__ void request_tail(int ib)
    {
        if constexpr (Q4) return;
        const uint32_t t = row + (uint32_t)(ib * M::tail_step() + M::tail0(nb));
        if constexpr (REP) tail = ld2(base + t);
        else tail = ld2(base + (t - lead(t))) | (ld2(base + t) << 16);
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
    __device__ __forceinline__ uint32_t shift(int ib) const
    {
        if constexpr (WT != QMAG_TYPE_Q6_K) return 0;
        return 8 * lead(row + (uint32_t)ib * BLOCK);
    }
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
        const int word = L == 2 ? s >> 2 : s >> 1;
        const uint32_t byte = L == 2 ? (uint32_t)(s & 3) : 2u * (uint32_t)(lane_id() >> 5) + (uint32_t)up;
        const uint32_t sel = 0x0C000C00u | (byte * 0x00010001u);            // that byte in both halves
        q4_digits(n, __builtin_amdgcn_perm(0u, S.sl[word], sel), __builtin_amdgcn_perm(0u, S.sh[word], sel), lo, hi);
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
// The partial results of a workgroup whose nw waves split the nb super-blocks,
// in LDS as [waves][MT][4][64].  One running sum per wave rounds the more the
// longer the row, so where a wave has more than `chain` super-blocks (a long
// row) it adds its sums there after every chain of them: each kernel's chain is
// as long as leaves the error against 64 bits at or below a lane tree's.
__host__ __device__ __forceinline__ bool long_row(int nb, int nw, int chain) { return nb > chain * nw; }
template <int MT>
__device__ __forceinline__ void put_partials(float *s_part, int wv, float (&r)[MT][4], bool add)
{
    float *p = s_part + wv * MT * 256 + lane_id();
    if (add)
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int i = 0; i < 4; i++) r[m][i] += p[(4 * m + i) * 64];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            p[(4 * m + i) * 64] = r[m][i];
            r[m][i] = 0.0f;
        }
}
// LDS bytes of such a workgroup: an image per wave, then the partials, in the
// images' place unless the rows are long
inline size_t split_lds(int nb, int nw, int chain, int mt, int image)
{
    const size_t part = sizeof(float) * 256 * (size_t)mt;
    return (size_t)nw * (long_row(nb, nw, chain) ? part + image : part > (size_t)image ? part : image);
}

// ------------------------------------------------------------------- tiles --
// A workgroup of four waves: wave w holds 32 weight rows, all four share 64
// activation rows (tokens).  Per super-block those go through registers
// into one of two LDS buffers while the other is consumed, and the wave's next
// 32 weight blocks through registers into its image: one barrier per
// super-block.
constexpr int TILE_ROW = QK_K + 16;        // padded LDS row: 16 rows of a read start 4 banks apart
constexpr int NT = 2;                      // 32-token groups of a tile
struct TileLds {
    int8_t a[2][32 * NT * TILE_ROW];
    float d[2][32 * NT];
    _Float16 s[2][32 * NT * 16];
};

// The Q8_K rows a thread stages: 16-byte piece tid % 16 of tokens tid / 16 +
// 16 k, the scale of token tid, half of the 16 sums of token tid / 2 (tokens past
// the last repeat it), from the uniform bases of the workgroup's first token.
// The offsets are 32-bit (64 rows of at most 2^26 values): as pointers they
// cost registers that the Q6_K loop does not have.
struct TileSrc {
    const int8_t *xq;
    const float *xd;
    const int16_t *xs;
    uint32_t x[2 * NT], d, s;
    __device__ __forceinline__ void init(const int8_t *q, const float *scales, const int16_t *sums, int nb, int last)
    {
        const uint32_t tid = threadIdx.x;
        auto row = [last](uint32_t t) { return (uint32_t)min((int)t, last); };
        xq = q;
        xd = scales;
        xs = sums;
#pragma unroll
        for (int k = 0; k < 2 * NT; k++) x[k] = row((tid >> 4) + 16 * k) * (uint32_t)(nb * QK_K) + 16 * (tid & 15);
        d = row(tid & (32 * NT - 1)) * (uint32_t)nb;
        s = row((tid & (64 * NT - 1)) >> 1) * (uint32_t)(nb * 16) + 8 * (tid & 1);
    }
};

// r[m][i] of a lane: token 32 m + 8 (i / 4) + 4 (lane / 32) + i % 4, weight row
// lane % 32, over the super-blocks ib0 .. nb - 1 (ib0 a multiple of eight).  The
// image's block ib0 has been requested.
template <int WT, class Img>
__device__ __forceinline__ void tile_products(Img &img, int ib0, int nb, const TileSrc &src, TileLds &lds,
                                              v16f (&r)[NT])
{
    using Row = WRow<WT, 2>;
    const int tid = (int)threadIdx.x, lane = lane_id(), lr = lane & 31, h = lane >> 5;
    uint4 va[2 * NT], vs = make_uint4(0, 0, 0, 0);
    float vd = 0.0f;
    // the eighth part s of block ib's requests
    auto request = [&](int s, int ib, bool weights) __attribute__((always_inline)) {
        if (weights && s < Img::WP) img.request(s, ib);
        if (weights && s == 7) img.request_tail(ib);
        if (s < 2 * NT) va[s] = ld16((const uint8_t *)src.xq + (size_t)ib * QK_K + src.x[s]);
        if (s == 5 && tid < 32 * NT) vd = ldg(src.xd + ib + src.d);
        if (Row::MIN && s == 6 && tid < 64 * NT) vs = ld16((const uint8_t *)(src.xs + (size_t)ib * 16 + src.s));
    };
    auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 2 * NT; k++)
            *(uint4 *)(lds.a[buf] + ((tid >> 4) + 16 * k) * TILE_ROW + 16 * (tid & 15)) = va[k];
        if (tid < 32 * NT) lds.d[buf][tid] = vd;
        if (Row::MIN && tid < 64 * NT) {
            const v4h a = sums_f16(make_uint2(vs.x, vs.y)), b = sums_f16(make_uint2(vs.z, vs.w));
            *(v8h *)(lds.s[buf] + 8 * tid) = v8h{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        }
    };
    v16f tot[NT];
#pragma unroll
    for (int m = 0; m < NT; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) r[m][i] = tot[m][i] = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; s++) request(s, ib0, false);
    img.store();
    stage(0);
    __syncthreads();
    for (int ib = ib0; ib < nb; ib++) {
        const int buf = ib & 1, nx = min(ib + 1, nb - 1);
        const Row w(img.block(), img.shift(ib));
        const int8_t *pa = lds.a[buf] + lr * TILE_ROW + 16 * h;
        v16i lo[NT], hi[NT];
#pragma unroll
        for (int m = 0; m < NT; m++)
#pragma unroll
            for (int i = 0; i < 16; i++) lo[m][i] = hi[m][i] = 0;
        // Step by step: the next step's LDS reads, a share of the next
        // super-block's requests (all at once they hold the wave for the time
        // the address unit takes to accept them, 700-2,000 cycles), this
        // step's MFMAs, and the next step's operands while those run.
        typename Row::Raw raw;
        v4i bl[2], bh[2], a[2][NT];
        w.read(0, raw);
#pragma unroll
        for (int m = 0; m < NT; m++) a[0][m] = *(const v4i *)(pa + 32 * m * TILE_ROW);
        w.operands(raw, 0, bl[0], bh[0]);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int c = s & 1, n = c ^ 1;
            if (s < 7) {
                w.read(s + 1, raw);
#pragma unroll
                for (int m = 0; m < NT; m++) a[n][m] = *(const v4i *)(pa + 32 * m * TILE_ROW + 32 * (s + 1));
            }
            request(s, nx, true);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < NT; m++) {
                lo[m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[c][m], bl[c], lo[m], 0, 0, 0);
                hi[m] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[c][m], bh[c], hi[m], 0, 0, 0);
            }
            if (s < 7) w.operands(raw, s + 1, bl[n], bh[n]);
            __builtin_amdgcn_sched_barrier(0);
        }
        // the min term last: its 32 results would be as many registers through
        // the steps
        v16f mn[NT];
        const float d = w.d();
        float nm = 0.0f;
        if constexpr (Row::MIN) {
            nm = -w.dmin();
            const v8h mb = w.mins8();
#pragma unroll
            for (int m = 0; m < NT; m++) {
                v16f z;
#pragma unroll
                for (int i = 0; i < 16; i++) z[i] = 0.0f;
                mn[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const v8h *)(lds.s[buf] + (32 * m + lr) * 16 + 8 * h),
                                                               mb, z, 0, 0, 0);
            }
        }
#pragma unroll
        for (int m = 0; m < NT; m++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float4 x4 = *(const float4 *)(lds.d[buf] + 32 * m + 8 * g + 4 * h);
                const float xv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int i = 4 * g + k;
                    float v = d * (float)(lo[m][i] + (hi[m][i] << Row::SHIFT));
                    if constexpr (Row::MIN) v = fmaf(nm, mn[m][i], v);
                    r[m][i] = fmaf(xv[k], v, r[m][i]);
                }
            }
        // sums of eight super-blocks are added up apart: one running sum
        // over a long row would round more than the matvec's lane tree (n_in
        // 8192: Q6_K 1.07e-7 of the result against 7.4e-8; Q4_K weights of
        // random bytes 1.04e-7 against 8.5e-8, now 7.5e-8).  With its
        // registers Q4_K of 4096 values and more takes 3% longer where a CU
        // has one workgroup (4096 x 4096 x 256 30.2 -> 31.1 us).
        if ((ib & 7) == 7 && ib + 1 < nb)
#pragma unroll
            for (int m = 0; m < NT; m++) {
                tot[m] += r[m];
#pragma unroll
                for (int i = 0; i < 16; i++) r[m][i] = 0.0f;
            }
        img.store();
        stage(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < NT; m++) r[m] += tot[m];
}

}  // namespace qmag
