// qmag_prefill.hip -- the MoE FFN layer for a batch of tokens (prefill,
// src/nn.c:509-649 with T > 1) as a grouped expert GEMM on int8 MFMA.
//
//   router_tile_kernel   per 256-wide k chunk, part[kc][T][E] = x . Wr^T, fp32
//                        MFMA; topk_kernel sums the chunks and adds the bias
//   topk_kernel          (qmag_moe.hip) softmax/top-k, Q8_K(x), shared gate
//   group_kernel         (token, slot) pairs bucketed by expert; the shared
//                        expert is bucket E with one pair per token
//   gateup_tile_kernel   h = silu(x.G) * (x.U) per pair: chunks of up to 64
//                        pairs of one expert x 64 rows of h
//   q8k_quant_kernel     Q8_K(h) per pair
//   down_tile_kernel     y[pair] = Q8_K(h) . D^T per chunk x 128 rows
//                        (both: the tile loop of qmag_mfma.h)
//   combine_kernel       out[t] = sum_k w_k y[t,k] + gs y[t,shared] in the
//                        reference order (nn.c:614-629), plus an optional
//                        residual
//
// Integer parity: the MFMA chains give the exact integer sum of each
// super-block (qmag_mfma.h); only the fp32 epilogue (scale * xd * integer sum)
// is associated differently from the reference's per-sub-block fp32 terms,
// well inside 1e-4 of max|y|.
//
// Every expert's weights are read once per 64-pair chunk (the shared
// expert's by every chunk of 64 tokens); the pair buffers (h: T*S*F fp32,
// y: T*S*N fp32) stay in HBM between kernels.
#include <type_traits>

#include "qmag_mfma.h"

namespace qmag {

// --------------------------------------------------------------- router --
// grid: (T / 64) x (E / 64) x (N / 256), 512 threads; a workgroup = 64 tokens
// x 64 experts x one 256-wide k chunk kc.  The 64 x rows and 64 router rows
// of the chunk are staged in LDS by DMA (one 1 KB row per instruction,
// rows padded by 16 bytes so the 16 rows one read touches start 4 banks
// apart), and wave w computes tokens 16 (w & 3) .. +16 against experts
// 32 (w >> 2) .. +32 as two 16 x 16 tiles.  Each tile's product over the
// chunk is 64 v_mfma_f32_16x16x4f32 into four accumulators (lane quarter q
// takes k = 16 u + 4 q .. +4 of step u, accumulator u % 4), summed as
// (a0 + a1) + (a2 + a3) and stored as the chunk's partial
// part[kc][token][expert]; topk_kernel adds the chunks in order and then
// the bias.  Each x and router row is read by 4 (not 16) workgroups, from
// LDS instead of registers, so one workgroup per CU suffices.  Rows past T or
// E are clamped to the last one: they only reach outputs that are not
// stored.
constexpr int RT_ROWS = 64;                    // tokens (experts) per workgroup
constexpr int RT_STRIDE = 256 + 4;             // padded LDS row, floats
__global__ __launch_bounds__(512) void router_tile_kernel(const float *__restrict__ Wr,
                                                          const float *__restrict__ x, int N, int E, int T,
                                                          float *__restrict__ part)
{
    __shared__ __align__(16) float s_x[RT_ROWS * RT_STRIDE], s_w[RT_ROWS * RT_STRIDE];
    const int tb = (int)blockIdx.x, eb = (int)blockIdx.y, kc = (int)blockIdx.z;
    const int lane = lane_id(), wv = (int)(threadIdx.x >> 6), lr = lane & 15, q = lane >> 4;
#pragma unroll
    for (int i = 0; i < RT_ROWS / 8; i++) {
        const int r = wv + 8 * i;
        const int tok = min(tb * RT_ROWS + r, T - 1), e = min(eb * RT_ROWS + r, E - 1);
        __builtin_amdgcn_global_load_lds((const QMAG_GLOBAL void *)(x + (size_t)tok * N + kc * 256 + lane * 4),
                                         (__attribute__((address_space(3))) void *)(s_x + r * RT_STRIDE), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((const QMAG_GLOBAL void *)(Wr + (size_t)e * N + kc * 256 + lane * 4),
                                         (__attribute__((address_space(3))) void *)(s_w + r * RT_STRIDE), 16, 0, 0);
    }
    __syncthreads();
    const int t0 = 16 * (wv & 3), e0 = 32 * (wv >> 2);
    const float *xa = s_x + (t0 + lr) * RT_STRIDE + 4 * q;
    const float *wa = s_w + (e0 + lr) * RT_STRIDE + 4 * q;
    v4f acc[2][4];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[j][c] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const float4 a = *(const float4 *)(xa + 16 * u);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float4 b = *(const float4 *)(wa + 16 * RT_STRIDE * j + 16 * u);
            v4f &c = acc[j][u & 3];
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
        }
    }
    // lane holds tile rows 4q + i (tokens) x column lr (expert)
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const v4f sum = (acc[j][0] + acc[j][1]) + (acc[j][2] + acc[j][3]);
        const int eo = eb * RT_ROWS + e0 + 16 * j + lr;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int to = tb * RT_ROWS + t0 + 4 * q + i;
            if (to < T && eo < E) part[((size_t)kc * T + to) * E + eo] = sum[i];
        }
    }
}

// ---------------------------------------------------------------- group --
// grp layout: cnt[E+1], off[E+2]; chunk[c] = {bucket
// (-1 past the last chunk), pairs, offset of its first pair in perm, 0}, one
// int4 per MC-pair chunk, so a workgroup learns all it needs from one load;
// perm[T*S] (16 t + slot, bucketed by expert).  Positions
// inside a bucket come from LDS atomics; every pair's result is computed
// independently of its neighbours, so the order does not change any output.
//
// Chunk order (the dispatch order of the chunked GEMMs): every full chunk
// first, then the partial ones by decreasing size, so the longest
// workgroups start first and the grid ends on the shortest ones.
constexpr int MC = 64;            // pairs per chunk of the chunked GEMMs (two 32-row MFMA tiles)
// the tile loop stages at most 64 rows, and the group kernel's chunk scans run
// within one wave
static_assert(MC == 64, "chunk size is tied to the tile loop");

__global__ __launch_bounds__(1024) void group_kernel(const int *__restrict__ sel, int T, int K, int E,
                                                     int *__restrict__ grp,
                                                     int4 *__restrict__ chunk, int max_chunks,
                                                     int *__restrict__ perm)
{
    __shared__ int s_cnt[257], s_off[258], s_fill[257], s_inc[257], s_finc[257];
    __shared__ int s_bin[MC], s_binf[MC];     // partial chunks by MC - size
    __shared__ int s_nch, s_wtot[2][5];
    const int tid = (int)threadIdx.x;
    for (int e = tid; e <= E; e += 1024) {
        s_cnt[e] = 0;
        s_fill[e] = 0;
    }
    if (tid < MC) {
        s_bin[tid] = 0;
        s_binf[tid] = 0;
    }
    __syncthreads();
    // ids come from the top-k (always < E); clamp anyway, this indexes LDS
    auto expert = [&](int p) { return min(max(sel[p], 0), E - 1); };
    for (int p = tid; p < T * K; p += 1024) atomicAdd(&s_cnt[expert(p)], 1);
    if (tid == 0) s_cnt[E] = T;      // shared expert: every token
    __syncthreads();
    // inclusive prefix sums of the pair counts and the full-chunk counts over
    // the E + 1 <= 257 buckets: a scan inside each of waves 0-4, then the
    // totals of the waves before; the partial chunks are counted per size
    {
        const int lane = tid & 63, wv = tid >> 6;
        const int c = tid <= E ? s_cnt[tid] : 0;
        if (c % MC) atomicAdd(&s_bin[MC - c % MC], 1);
        int ci = c, fi = c / MC;
        if (wv < 5) {                          // wave-uniform
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(ci, d), of = __shfl_up(fi, d);
                if (lane >= d) {
                    ci += o;
                    fi += of;
                }
            }
            if (lane == 63) {
                s_wtot[0][wv] = ci;
                s_wtot[1][wv] = fi;
            }
        }
        __syncthreads();
        if (tid <= E) {
            for (int w = 0; w < wv; w++) {
                ci += s_wtot[0][w];
                fi += s_wtot[1][w];
            }
            s_inc[tid] = ci;
            s_finc[tid] = fi;
        }
        __syncthreads();
    }
    // exclusive prefix of the size bins (one wave; bin i holds chunks of
    // MC - i pairs, so increasing i is decreasing size)
    if (tid < MC) {
        const int v = s_bin[tid];
        int incl = v;
#pragma unroll
        for (int d = 1; d < MC; d <<= 1) {
            const int o = __shfl_up(incl, d, MC);
            if (tid >= d) incl += o;
        }
        s_bin[tid] = incl - v;
        if (tid == MC - 1) s_nch = s_finc[E] + incl;
    }
    __syncthreads();
    if (tid <= E) {
        int *cnt = grp, *off = grp + (E + 1);
        const int c = s_cnt[tid];
        s_off[tid] = s_inc[tid] - c;
        cnt[tid] = c;
        off[tid] = s_inc[tid] - c;
        const int nf = c / MC, f0 = s_finc[tid] - nf, o = s_inc[tid] - c;
        for (int i = 0; i < nf; i++) chunk[f0 + i] = make_int4(tid, MC, o + i * MC, 0);
        if (c % MC) {
            const int bin = MC - c % MC;
            chunk[s_finc[E] + s_bin[bin] + atomicAdd(&s_binf[bin], 1)] = make_int4(tid, c % MC, o + nf * MC, 0);
        }
        if (tid == E) off[E + 1] = s_inc[E];
    }
    __syncthreads();
    for (int p = tid; p < T * K; p += 1024) {
        const int e = expert(p);
        perm[s_off[e] + atomicAdd(&s_fill[e], 1)] = 16 * (p / K) + p % K;
    }
    for (int t = tid; t < T; t += 1024) perm[s_off[E] + t] = 16 * t + K;
    for (int i = s_nch + tid; i < max_chunks; i += 1024) chunk[i] = make_int4(-1, 0, 0, 0);
}

// --------------------------------------------------------------- gate / up --
// grid: (max MC-pair chunks) x (F / 64); a workgroup = one chunk of up to 64
// pairs of one bucket x 64 rows of h, wave w 16 of them: the gate rows are
// rows 0-15 of its 32, the same rows of up rows 16-31, so silu(g) * u pairs
// lanes lr and lr + 16 of one result.  The super-blocks of its rows stream
// through the wave's LDS image in line order; chunks of at most 32 pairs run
// one tile.  The pair ids are read while block 0 of the weights is in flight.
// Instruction issue and the rounds of workgroups bound it (two per CU by
// registers).  512 tokens of n_embd 2048, n_ff 512, 256 experts, top 8: the
// layer takes 168 us against 187 with rows held whole in registers (16 rows x
// 64 bytes per request, 16-pair tiles).  One 32-pair tile per chunk at three or
// four workgroups per CU was slower (the registers spill; 285 us).
__device__ __forceinline__ int pair_of(int code, int S) { return (code >> 4) * S + (code & 15); }

__global__ __launch_bounds__(256, 2) void gateup_tile_kernel(
    const uint8_t *__restrict__ gate_exps, const uint8_t *__restrict__ up_exps,
    const uint8_t *__restrict__ gate_sh, const uint8_t *__restrict__ up_sh, int E, int S, int F, int nb,
    const int4 *__restrict__ chunk, const int *__restrict__ perm, const int8_t *__restrict__ xq,
    const float *__restrict__ xd, const int16_t *__restrict__ xs, float *__restrict__ h)
{
    using Img = WImage<QMAG_TYPE_Q4_K, 32, true>;
    __shared__ __align__(16) TileLds<2> s_t;
    __shared__ __align__(16) uint8_t s_w[4 * Img::BYTES];
    __shared__ int s_code[MC];
    const int rchunks = F / 64;
    const int u = (int)blockIdx.x / rchunks, rc = (int)blockIdx.x % rchunks;
    const int4 ck = chunk[u];
    if (ck.x < 0) return;
    const int e = ck.x, npair = ck.y;
    const int tid = (int)threadIdx.x, lane = lane_id(), lr = lane & 31, hf = lane >> 5, wv = tid >> 6;
    const int row0 = rc * 64 + 16 * wv;
    const size_t rowb = (size_t)nb * Q4K_BYTES, off = ((size_t)e * F + row0) * rowb;
    Img img;
    img.init2(s_w + wv * Img::BYTES, e < E ? gate_exps + off : gate_sh + (size_t)row0 * rowb,
              e < E ? up_exps + off : up_sh + (size_t)row0 * rowb, nb);
    img.request_all(0);
    auto code = [&](int t) { return perm[ck.z + min(t, npair - 1)]; };
    if (tid < MC) s_code[tid] = code(tid);
    auto run = [&](auto nt) __attribute__((always_inline)) {
        constexpr int NT = decltype(nt)::value;
        TileSrc<NT> src;
        src.init(xq, xd, xs, nb, [&](int t) { return code(t) >> 4; });
        v16f r[NT];
        tile_products<QMAG_TYPE_Q4_K, NT, false>(img, nb, src, (TileLds<NT> &)s_t, r);
#pragma unroll
        for (int m = 0; m < NT; m++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const float g = r[m][i];
                const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(g), __float_as_uint(g), false, false);
                const float up = __uint_as_float(sw[1]);          // in lanes lr < 16: lane lr + 16's value
                const int t = 32 * m + 8 * (i >> 2) + 4 * hf + (i & 3);
                if (lr < 16 && t < npair)
                    h[(size_t)pair_of(s_code[t], S) * F + row0 + lr] = (g / (1.0f + expf(-g))) * up;
            }
    };
    if (npair > 32) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 1>{});
}

// ----------------------------------------------------------------- down --
// grid: (max MC-pair chunks) x (N / 128); a workgroup = one chunk of up to 64
// pairs of one bucket x 128 rows, 32 per wave.
constexpr int DN_ROWS = 128;

__global__ __launch_bounds__(256, 2) void down_tile_kernel(
    const uint8_t *__restrict__ down_exps, int t_down, const uint8_t *__restrict__ down_sh, int t_down_sh, int E,
    int S, int N, int nb, const int4 *__restrict__ chunk, const int *__restrict__ perm,
    const int8_t *__restrict__ hq, const float *__restrict__ hd, const int16_t *__restrict__ hs,
    float *__restrict__ y)
{
    constexpr int IMG = WImage<QMAG_TYPE_Q6_K, 32>::BYTES;
    static_assert(IMG >= WImage<QMAG_TYPE_Q4_K, 32>::BYTES, "");
    __shared__ __align__(16) TileLds<2> s_t;
    __shared__ __align__(16) uint8_t s_w[4 * IMG];
    __shared__ int s_code[MC];
    const int rblocks = N / DN_ROWS;
    const int u = (int)blockIdx.x / rblocks, rb = (int)blockIdx.x % rblocks;
    const int4 ck = chunk[u];
    if (ck.x < 0) return;
    const int e = ck.x, npair = ck.y;
    const int tid = (int)threadIdx.x, lane = lane_id(), lr = lane & 31, hf = lane >> 5, wv = tid >> 6;
    const int row0 = rb * DN_ROWS + 32 * wv;
    auto code = [&](int t) { return perm[ck.z + min(t, npair - 1)]; };
    auto run = [&](auto type, auto nt) __attribute__((always_inline)) {
        constexpr int WT = decltype(type)::value, NT = decltype(nt)::value;
        WImage<WT, 32> img;
        const size_t slab = (size_t)N * nb * img.BLOCK;
        img.init(s_w + wv * IMG, e < E ? down_exps + (size_t)e * slab : down_sh, row0, N, nb);
        img.request_all(0);
        if (tid < MC) s_code[tid] = code(tid);
        TileSrc<NT> src;
        src.init(hq, hd, hs, nb, [&](int t) { return pair_of(code(t), S); });
        v16f r[NT];
        tile_products<WT, NT, false>(img, nb, src, (TileLds<NT> &)s_t, r);
#pragma unroll
        for (int m = 0; m < NT; m++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int t = 32 * m + 8 * (i >> 2) + 4 * hf + (i & 3);
                if (t < npair) y[(size_t)pair_of(s_code[t], S) * N + row0 + lr] = r[m][i];
            }
    };
    using std::integral_constant;
    const bool q6 = (e < E ? t_down : t_down_sh) == QMAG_TYPE_Q6_K, two = npair > 32;
    if (q6 && two) run(integral_constant<int, QMAG_TYPE_Q6_K>{}, integral_constant<int, 2>{});
    else if (q6) run(integral_constant<int, QMAG_TYPE_Q6_K>{}, integral_constant<int, 1>{});
    else if (two) run(integral_constant<int, QMAG_TYPE_Q4_K>{}, integral_constant<int, 2>{});
    else run(integral_constant<int, QMAG_TYPE_Q4_K>{}, integral_constant<int, 1>{});
}

// -------------------------------------------------------------- combine --
// One thread per 4 consecutive outputs of one token: the 9 slot rows (and the
// residual) are requested as float4 before any is used; each element is
// summed in the reference's order with unfused multiply and add.
__global__ __launch_bounds__(256) void combine_kernel(const float *__restrict__ y, const float *__restrict__ w,
                                                      const float *__restrict__ gs, int T, int K, int N,
                                                      const float *__restrict__ resid, float *__restrict__ out)
{
    const size_t i = 4 * ((size_t)blockIdx.x * 256 + threadIdx.x);   // N % 4 == 0
    if (i >= (size_t)T * N) return;
    const int t = (int)(i / N), r = (int)(i % N), S = K + 1;
    float4 v[9];                                                       // K <= 8
#pragma unroll
    for (int k = 0; k < 9; k++) v[k] = *(const float4 *)(y + ((size_t)t * S + min(k, K)) * N + r);
    const float4 rs = resid ? *(const float4 *)(resid + i) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        if (k < K) {
            const float wk = w[t * K + k];
            acc.x = __fadd_rn(acc.x, __fmul_rn(wk, v[k].x));
            acc.y = __fadd_rn(acc.y, __fmul_rn(wk, v[k].y));
            acc.z = __fadd_rn(acc.z, __fmul_rn(wk, v[k].z));
            acc.w = __fadd_rn(acc.w, __fmul_rn(wk, v[k].w));
        }
    }
    const float g = gs[t];
    const float4 sh = v[8];                    // row min(8, K) = K: the shared slot
    acc.x = __fadd_rn(acc.x, __fmul_rn(g, sh.x));
    acc.y = __fadd_rn(acc.y, __fmul_rn(g, sh.y));
    acc.z = __fadd_rn(acc.z, __fmul_rn(g, sh.z));
    acc.w = __fadd_rn(acc.w, __fmul_rn(g, sh.w));
    if (resid) {
        acc.x = __fadd_rn(acc.x, rs.x);
        acc.y = __fadd_rn(acc.y, rs.y);
        acc.z = __fadd_rn(acc.z, rs.z);
        acc.w = __fadd_rn(acc.w, rs.w);
    }
    *(float4 *)(out + i) = acc;
}

// ------------------------------------------------------------------ host --
int launch_router_mfma(const qmag_moe_layer *L, const float *x, int T, float *part, hipStream_t s)
{
    const int N = L->n_embd, E = L->n_expert;
    if (N % 256) return fail(QMAG_ERR_ARG, "router: n_embd=%d", N);
    hipLaunchKernelGGL(router_tile_kernel, dim3((T + RT_ROWS - 1) / RT_ROWS, (E + RT_ROWS - 1) / RT_ROWS, N / 256),
                       dim3(512), 0, s, L->gate_inp, x, N, E, T, part);
    QMAG_HIP(hipGetLastError());
    return QMAG_OK;
}

int moe_grouped(const qmag_moe_layer *L, int T, const int *sel, const float *w, const float *gs,
                const int8_t *xq, const float *xd, const int16_t *xs, float *h, int8_t *hq, float *hd,
                int16_t *hs, const float *resid, float *out, hipStream_t s)
{
    const int N = L->n_embd, F = L->n_ff, E = L->n_expert, K = L->n_used, S = K + 1;
    int st;
    // upper bound of the MC-pair chunks: sum ceil(n_e / MC) <= T*K/MC + E,
    // plus the shared bucket
    const int max_chunks = (T * K + MC - 1) / MC + E + (T + MC - 1) / MC;
    // int4 chunk descriptors first (16-byte aligned), then the int tables
    int4 *chunk = (int4 *)workspace(WS_GRP, sizeof(int4) * (size_t)max_chunks +
                                                sizeof(int) * ((size_t)2 * (E + 2) + (size_t)T * S),
                                    &st);
    if (st) return st;
    int *grp = (int *)(chunk + max_chunks), *perm = grp + 2 * (E + 2);
    float *y = (float *)workspace(WS_Y, sizeof(float) * (size_t)T * S * N, &st);
    if (st) return st;

    prof_begin(PROF_GROUP, s);
    hipLaunchKernelGGL(group_kernel, dim3(1), dim3(1024), 0, s, sel, T, K, E, grp, chunk, max_chunks, perm);
    prof_end(PROF_GROUP, s);
    prof_begin(PROF_GATEUP, s);
    hipLaunchKernelGGL(gateup_tile_kernel, dim3(max_chunks * (F / 64)), dim3(256), 0, s,
                       (const uint8_t *)L->gate_exps, (const uint8_t *)L->up_exps, (const uint8_t *)L->gate_shexp,
                       (const uint8_t *)L->up_shexp, E, S, F, N / QK_K, chunk, perm, xq, xd, xs, h);
    prof_end(PROF_GATEUP, s);
    prof_begin(PROF_HQUANT, s);
    st = launch_q8k_quant(h, T * S * (F / QK_K), hq, hd, hs, s);
    prof_end(PROF_HQUANT, s);
    if (st) return st;
    prof_begin(PROF_DOWN, s);
    hipLaunchKernelGGL(down_tile_kernel, dim3(max_chunks * (N / DN_ROWS)), dim3(256), 0, s,
                       (const uint8_t *)L->down_exps, L->t_down_exps, (const uint8_t *)L->down_shexp,
                       L->t_down_shexp, E, S, N, F / QK_K, chunk, perm, hq, hd, hs, y);
    prof_end(PROF_DOWN, s);
    prof_begin(PROF_COMBINE, s);
    hipLaunchKernelGGL(combine_kernel, dim3((unsigned)(((size_t)T * N / 4 + 255) / 256)), dim3(256), 0, s, y, w, gs,
                       T, K, N, resid, out);
    prof_end(PROF_COMBINE, s);
    QMAG_HIP(hipGetLastError());
    return QMAG_OK;
}

}  // namespace qmag
