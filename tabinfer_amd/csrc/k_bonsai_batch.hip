// k_bonsai_batch.hip — the Bonsai decoder's kernels for a prompt's tokens together (T >= 2):
// Model::forward per prompt token (native/crates/n2-core/src/model.rs:349-501, ops.rs), with
// every per-token operation on T rows at once and the projections on the matrix cores
// (k_tern_gemm.hip). Token by token a 48-token prompt through two layers took 3610 us (16
// launches a token and every weight read 48 times); as one batch it takes 157 us,
// 26 of them lm_head, the rest 20 launches of 3-10 us and four around them.
//
// Rows are [token][width]. Widths are multiples of 1024; a row belongs to one workgroup of 256
// threads, thread t holding elements 4 (t + 256 k) .. + 3.
#include "ti_internal.h"
#include "ti_bonsai_batch.h"
#include <math.h>

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// totals / maxima of one value per thread of a 256-thread workgroup, in every thread
__device__ __forceinline__ float wg_sum(float v, float* red) {
    v = ti_wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}
__device__ __forceinline__ float wg_max(float v, float* red) {
    v = ti_wave_max(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// n2 quantize_act of a row (tern.rs:196-222): scale = 127 / amax (1 if amax = 0), codes
// clamp(round-half-away(v * scale), -127, 127), sums per 64 (16 threads x 4 elements)
template <int NK>
__device__ __forceinline__ void quant_row(const v4f (&v)[NK], int n, uint32_t* __restrict__ act, int32_t* __restrict__ xsum,
                                          float* __restrict__ scale_out, float* red) {
    const int t = threadIdx.x;
    float mx = 0.0f;
#pragma unroll
    for (int k = 0; k < NK; k++)
#pragma unroll
        for (int i = 0; i < 4; i++) mx = fmaxf(mx, fabsf(v[k][i]));
    const float amax = wg_max(mx, red);
    const float qs = amax > 0.0f ? 127.0f / amax : 1.0f;
    if (t == 0) *scale_out = qs;
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int e4 = t + 256 * k;
        uint32_t w = 0;
        int bs = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float rq = roundf(v[k][i] * qs);
            rq = fminf(fmaxf(rq, -127.0f), 127.0f);
            const int q = (int)rq;
            bs += q;
            w |= (uint32_t)(q & 0xff) << (8 * i);
        }
        bs += ti_xor_i(bs, 8);
        bs += ti_xor_i(bs, 4);
        bs += ti_xor_i(bs, 2);
        bs += ti_xor_i(bs, 1);
        if (4 * e4 < n) {
            act[e4] = w;
            if ((t & 15) == 0) xsum[e4 >> 4] = bs;
        }
    }
}

// x = emb[hist[pos + t]] (first layer) or x + add / add_scale[t]; RMSNorm (ops.rs:14-22); n2 quantizer
template <int NK>
__global__ __launch_bounds__(256) void k_bb_norm(float* __restrict__ x, const float* __restrict__ add,
                                                 const float* __restrict__ add_scale, const float* __restrict__ w, float eps,
                                                 int H, const uint32_t* __restrict__ hist, const uint16_t* __restrict__ emb,
                                                 int vocab, uint32_t* __restrict__ act, int32_t* __restrict__ xsum,
                                                 float* __restrict__ scale) {
    __shared__ float red[2][4];
    const int t = threadIdx.x;
    const size_t tok = blockIdx.x;
    v4f v[NK], a[NK], wv[NK];
    const uint16_t* er = nullptr;
    if (emb) {
        uint32_t id = hist[tok];
        id = id < (uint32_t)vocab ? id : (uint32_t)(vocab - 1);
        er = emb + (size_t)id * H;
    }
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int e = min(4 * (t + 256 * k), H - 4);
        wv[k] = *reinterpret_cast<const v4f*>(w + e);
        if (er) {
            const ushort4 h = *reinterpret_cast<const ushort4*>(er + e);
            v[k] = v4f{ti_h2f(h.x), ti_h2f(h.y), ti_h2f(h.z), ti_h2f(h.w)};
        } else {
            v[k] = *reinterpret_cast<const v4f*>(x + tok * H + e);
            a[k] = *reinterpret_cast<const v4f*>(add + tok * H + e);
        }
    }
    const float inv_add = er ? 0.0f : 1.0f / add_scale[tok];
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int e = 4 * (t + 256 * k);
        const bool in = e < H;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (!er) {
                const float d = a[k][i] * inv_add;
                v[k][i] = v[k][i] + d;
            }
            if (in) ss = ss + v[k][i] * v[k][i];
        }
        if (in) *reinterpret_cast<v4f*>(x + tok * H + e) = v[k];
    }
    const float mean = wg_sum(ss, red[0]) / (float)H;
    const float inv = 1.0f / sqrtf(mean + eps);
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const bool in = 4 * (t + 256 * k) < H;
#pragma unroll
        for (int i = 0; i < 4; i++) v[k][i] = in ? v[k][i] * inv * wv[k][i] : 0.0f;
    }
    quant_row<NK>(v, H, act + tok * (H / 4), xsum + tok * (H / 64), scale + tok, red[1]);
}

// SwiGLU of the scaled gate/up (ops.rs:110-117) + quantizer
template <int NK>
__global__ __launch_bounds__(256) void k_bb_swiglu(const float* __restrict__ g, const float* __restrict__ u,
                                                   const float* __restrict__ gu_scale, int I, uint32_t* __restrict__ act,
                                                   int32_t* __restrict__ xsum, float* __restrict__ scale) {
    __shared__ float red[4];
    const int t = threadIdx.x;
    const size_t tok = blockIdx.x;
    v4f gv[NK], uv[NK];
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int e = min(4 * (t + 256 * k), I - 4);
        gv[k] = *reinterpret_cast<const v4f*>(g + tok * I + e);
        uv[k] = *reinterpret_cast<const v4f*>(u + tok * I + e);
    }
    const float inv = 1.0f / gu_scale[tok];
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const bool in = 4 * (t + 256 * k) < I;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float gg = gv[k][i] * inv;
            const float uu = uv[k][i] * inv;
            gv[k][i] = in ? (gg / (1.0f + expf(-gg))) * uu : 0.0f;
        }
    }
    quant_row<NK>(gv, I, act + tok * (I / 4), xsum + tok * (I / 64), scale + tok, red);
}

// One wave a (token, head of q | k | v), hd 128: lane i holds the rotary pair (i, i + 64). q and k
// are scaled, RMS-normalised and rotated (model.rs:399-418); k and the scaled v go to the cache.
__global__ __launch_bounds__(256) void k_bb_rope(const float* __restrict__ q, const float* __restrict__ k,
                                                 const float* __restrict__ v, const float* __restrict__ act_scale,
                                                 const float* __restrict__ qn, const float* __restrict__ kn,
                                                 const float* __restrict__ rope, float eps, float* __restrict__ qrot,
                                                 float* __restrict__ kc, float* __restrict__ vc, int T, int nHq, int nKv) {
    constexpr int HD = 128;
    const int lane = threadIdx.x & 63, heads = nHq + 2 * nKv;
    const long u = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= (long)T * heads) return;
    const int t = (int)(u / heads), h = (int)(u % heads);
    const float inv = 1.0f / act_scale[t];
    const bool isq = h < nHq, isk = !isq && h < nHq + nKv;
    const int hk = isk ? h - nHq : h - nHq - nKv;
    const float* src = isq ? q + ((size_t)t * nHq + h) * HD : (isk ? k : v) + ((size_t)t * nKv + hk) * HD;
    float a = src[lane] * inv, b = src[lane + 64] * inv;
    float* dst = isq ? qrot + ((size_t)t * nHq + h) * HD : (isk ? kc : vc) + ((size_t)t * nKv + hk) * HD;
    if (isq || isk) {
        const float* nw = isq ? qn : kn;
        const float mean = ti_wave_sum(a * a + b * b) / (float)HD;
        const float rinv = 1.0f / sqrtf(mean + eps);
        a = a * rinv * nw[lane];
        b = b * rinv * nw[lane + 64];
        const float c = rope[(size_t)t * HD + lane], s = rope[(size_t)t * HD + 64 + lane];
        const float y0 = a * c - b * s, y1 = b * c + a * s;
        a = y0;
        b = y1;
    }
    dst[lane] = a;
    dst[lane + 64] = b;
}

// Causal attention over the f32 cache on the f32 matrix cores (v_mfma_f32_16x16x4_f32: f32
// operands, products and sums). Workgroup: KV head x 8 tokens (16 query rows: token r / 2, query
// head r % 2 of the KV head) x one range of keys; its 4 waves take every fourth tile of 16 keys
// with a running maximum and meet at the end. The products are taken transposed, S^T = K Q^T and
// O^T = V^T P^T, so a lane's scores are the P operand of the second one as they stand (key
// 4j + i of query row l%16) and a query's maximum, sum and rescale live in its own lanes.
// K and V tiles go through the wave's own LDS (whole 512-byte rows from memory, 16-byte pieces of
// 16 rows as operands). At 48 tokens over 148 positions: 6.8 us, nearly all latency
// (the token-by-token kernels took 6.3 us a token).
struct AttnBuf {
    v4f k[16][33], v[16][33];
};
__global__ __launch_bounds__(256, 2) void k_bb_attn(const float* __restrict__ qrot, const float* __restrict__ kc,
                                                    const float* __restrict__ vc, int T, int pos, int nHq, int nKv,
                                                    int ntile, int nsplit, float* __restrict__ po, float* __restrict__ pml) {
    constexpr int HD = 128;
    __shared__ AttnBuf s_buf[4];
    __shared__ float s_m[4][16], s_l[4][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, j = lane >> 4;
    const int hk = blockIdx.x % nKv, tt = (blockIdx.x / nKv) % ntile, split = blockIdx.x / (nKv * ntile);
    const int t0 = 8 * tt;
    const int tq = min(t0 + (r >> 1), T - 1), head = 2 * hk + (r & 1);
    const int S = pos + min(t0 + 8, T);                // keys the last of these tokens sees
    const int kt = (S + 15) / 16;
    const int k0 = (int)((long)kt * split / nsplit), k1 = (int)((long)kt * (split + 1) / nsplit);
    const float scale = 1.0f / sqrtf((float)HD);
    AttnBuf& L = s_buf[wave];
    const size_t kvd = (size_t)nKv * HD;

    v4f q[8];                                          // dims 16 p + 4 j .. + 3 of this query row
#pragma unroll
    for (int p = 0; p < 8; p++) q[p] = *reinterpret_cast<const v4f*>(qrot + ((size_t)tq * nHq + head) * HD + 16 * p + 4 * j);
    const int lr = lane >> 5, lp = lane & 31;          // loads: rows 2 i + lr, piece lp
    v4f kr[8], vr[8];
    auto load = [&](int tile) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const size_t row = min(16 * tile + 2 * i + lr, S - 1);
            kr[i] = *reinterpret_cast<const v4f*>(kc + row * kvd + hk * HD + 4 * lp);
            vr[i] = *reinterpret_cast<const v4f*>(vc + row * kvd + hk * HD + 4 * lp);
        }
    };
    float m = -INFINITY, l = 0.0f;
    v4f o[8] = {};                                     // tile (h, e): dims 64 h + 4 c + e, c = 4 j + i in element i
    if (k0 + wave < k1) load(k0 + wave);
    for (int tile = k0 + wave; tile < k1; tile += 4) {
        ti_wave_lds_fence();                           // the last tile is read
#pragma unroll
        for (int i = 0; i < 8; i++) {
            L.k[2 * i + lr][lp] = kr[i];
            L.v[2 * i + lr][lp] = vr[i];
        }
        ti_wave_lds_fence();
        if (tile + 4 < k1) load(tile + 4);
        v4f s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int p = 0; p < 8; p++) {
            const v4f kk = L.k[r][4 * p + j];
#pragma unroll
            for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[e], q[p][e], s, 0, 0, 0);
        }
        float tm = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int key = 16 * tile + 4 * j + i;
            s[i] = key <= pos + tq ? s[i] * scale : -INFINITY;
            tm = fmaxf(tm, s[i]);
        }
        tm = fmaxf(tm, ti_xor(tm, 16));
        tm = fmaxf(tm, ti_xor(tm, 32));
        const float mn = fmaxf(m, tm);
        const float mr = mn == -INFINITY ? 0.0f : mn;  // no key so far: every weight 0
        const float alpha = expf(m - mr);
        m = mn;
        l = l * alpha;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s[i] = expf(s[i] - mr);
            l += s[i];
        }
#pragma unroll
        for (int t = 0; t < 8; t++) o[t] = o[t] * alpha;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const v4f vv = L.v[4 * j + i][16 * h + r];
#pragma unroll
                for (int e = 0; e < 4; e++)
                    o[4 * h + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[e], s[i], o[4 * h + e], 0, 0, 0);
            }
    }
    l += ti_xor(l, 16);
    l += ti_xor(l, 32);
    __syncthreads();                                   // every wave's tiles are read
    v4f* so = reinterpret_cast<v4f*>(s_buf);           // [wave][16 rows][33 pieces]
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            so[(wave * 16 + r) * 33 + 16 * h + 4 * j + i] = v4f{o[4 * h][i], o[4 * h + 1][i], o[4 * h + 2][i], o[4 * h + 3][i]};
    if (j == 0) {
        s_m[wave][r] = m;
        s_l[wave][r] = l;
    }
    __syncthreads();
    for (int e = tid; e < 16 * 32; e += 256) {
        const int row = e >> 5, p = e & 31;
        const int t = t0 + (row >> 1);
        if (t >= T) continue;
        const float M = fmaxf(fmaxf(s_m[0][row], s_m[1][row]), fmaxf(s_m[2][row], s_m[3][row]));
        const float mr = M == -INFINITY ? 0.0f : M;
        float Lt = 0.0f;
        v4f a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float f = expf(s_m[w][row] - mr);
            Lt += s_l[w][row] * f;
            a = a + so[(w * 16 + row) * 33 + p] * f;
        }
        const size_t slot = ((size_t)t * nHq + 2 * hk + (row & 1)) * nsplit + split;
        reinterpret_cast<v4f*>(po)[slot * 32 + p] = a;
        if (p == 0) {
            pml[2 * slot] = M;
            pml[2 * slot + 1] = Lt;
        }
    }
}

// the splits' partials -> attention output of a token, quantized
template <int NK>
__global__ __launch_bounds__(256) void k_bb_merge(const float* __restrict__ po, const float* __restrict__ pml, int nsplit,
                                                  int nq, uint32_t* __restrict__ act, int32_t* __restrict__ xsum,
                                                  float* __restrict__ scale) {
    __shared__ float red[4];
    const int t = threadIdx.x;
    const size_t tok = blockIdx.x;
    v4f v[NK];
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int e = 4 * (t + 256 * k);
        v[k] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        if (e >= nq) continue;
        const size_t slot = (tok * (nq / 128) + e / 128) * nsplit;
        float M = -INFINITY;
        for (int s = 0; s < nsplit; s++) M = fmaxf(M, pml[2 * (slot + s)]);
        float Lt = 0.0f;
        for (int s = 0; s < nsplit; s++) {
            const float f = expf(pml[2 * (slot + s)] - M);
            Lt += pml[2 * (slot + s) + 1] * f;
            v[k] = v[k] + reinterpret_cast<const v4f*>(po)[(slot + s) * 32 + (e & 127) / 4] * f;
        }
        v[k] = v[k] / Lt;
    }
    quant_row<NK>(v, nq, act + tok * (nq / 4), xsum + tok * (nq / 64), scale + tok, red);
}

}  // namespace

#define BY_WIDTH(n, CALL)                                                                      \
    do {                                                                                       \
        if ((n) <= 1024) { CALL(1); } else if ((n) <= 2048) { CALL(2); }                       \
        else if ((n) <= 4096) { CALL(4); } else if ((n) <= 6144) { CALL(6); } else { CALL(8); } \
    } while (0)

int ti_bb_norm(ti_ctx* c, const ti_bb_rows& R, float* x, const float* add, const float* add_scale, const float* w, float eps,
               int H, const uint32_t* hist, const uint16_t* emb, int vocab, float* scale) {
#define C_(K) k_bb_norm<K><<<R.T, 256, 0, c->stream>>>(x, add, add_scale, w, eps, H, hist, emb, vocab, R.act, R.xsum, scale)
    BY_WIDTH(H, C_);
#undef C_
    TI_LAUNCHED("k_bb_norm");
    return TI_OK;
}

int ti_bb_swiglu(ti_ctx* c, const ti_bb_rows& R, const float* g, const float* u, const float* gu_scale, int I, float* scale) {
#define C_(K) k_bb_swiglu<K><<<R.T, 256, 0, c->stream>>>(g, u, gu_scale, I, R.act, R.xsum, scale)
    BY_WIDTH(I, C_);
#undef C_
    TI_LAUNCHED("k_bb_swiglu");
    return TI_OK;
}

int ti_bb_rope(ti_ctx* c, const float* q, const float* k, const float* v, const float* act_scale, const float* qn,
               const float* kn, const float* rope, float eps, float* qrot, float* kc, float* vc, int T, int nHq, int nKv) {
    const long units = (long)T * (nHq + 2 * nKv);
    k_bb_rope<<<(unsigned)((units + 3) / 4), 256, 0, c->stream>>>(q, k, v, act_scale, qn, kn, rope, eps, qrot, kc, vc, T, nHq, nKv);
    TI_LAUNCHED("k_bb_rope");
    return TI_OK;
}

int ti_bb_attn(ti_ctx* c, const ti_bb_rows& R, const float* qrot, const float* kc, const float* vc, int pos, int nHq, int nKv,
               float* po, float* pml, long rowsplits, float* scale) {
    const int ntile = (R.T + 7) / 8, nq = nHq * 128;
    // key ranges: enough workgroups for the CUs twice over, at least a tile a wave, and the
    // partials within their buffer
    const int kt = (pos + R.T + 15) / 16;
    long ns = (2L * c->cus + nKv * ntile - 1) / (nKv * ntile);
    if (ns > (kt + 3) / 4) ns = (kt + 3) / 4;
    if (ns > TI_BB_SPLITS) ns = TI_BB_SPLITS;
    if (ns > rowsplits / ((long)R.T * nHq)) ns = rowsplits / ((long)R.T * nHq);
    TI_REQUIRE(ns >= 1, "bonsai: %d tokens exceed the attention scratch", R.T);
    k_bb_attn<<<(unsigned)(nKv * ntile * ns), 256, 0, c->stream>>>(qrot, kc, vc, R.T, pos, nHq, nKv, ntile, (int)ns, po, pml);
    TI_LAUNCHED("k_bb_attn");
#define C_(K) k_bb_merge<K><<<R.T, 256, 0, c->stream>>>(po, pml, (int)ns, nq, R.act, R.xsum, scale)
    BY_WIDTH(nq, C_);
#undef C_
    TI_LAUNCHED("k_bb_merge");
    return TI_OK;
}
