// k_pattn.hip — causal attention of a prompt's tokens over the int8 KV cache (attnBlock's T > 1 case,
// models/qwen3.js:2534-2577), head_dim 128, both products on the matrix cores at f32 accuracy.
//
// Workgroup (4 waves): one KV head, one range of keys, 64 query rows (row = token x query head of the
// KV head); a wave owns 16 rows and meets the others only over the staged keys. Key blocks of 64 are
// staged in LDS as MFMA operands (K codes f16, V codes bf16, exact), the next block's loads in flight meanwhile.
//   - S^T = K Q^T, one v_mfma_f32_16x16x32_f16 per 32-dim scale group, 16 keys and q half: q = hi + lo in
//     f16 (to 2^-22), each group's sum scaled by its key's scale in f32. Transposed, a lane's scores are
//     those of one query row, keys 4j..4j+3 of each 16: the P operand of the second product as they
//     stand, and the row's running maximum and sum live in its own four lanes.
//   - O^T = V^T P^T with P times the V scale of (key, group) in f32, split into three bf16, exactly: bf16 has
//     f32's exponents, so a weight is as exact as in f32 beside any other, and what one key's scale is does not
//     touch another's. (Two f16 under a common power of two take 5% less time, but lose all of a weight
//     2^-36 of the largest scale of its keys.) The codes are exact in bf16.
// What bounds it is latency first (up to 16384 keys a workgroup has 2 to 4 blocks; its loads of q are issued
// before all else, and three workgroups share a CU), then the VALU work of the weights (scale, mask, exponential,
// four scaled three-fold splits). With 32 rows a wave, whose operands are read from LDS for two products, only two
// fit (with ranges of any length and weights in two halves, 256 tokens at 3840: 47.7 against 46.7 us, at 0: 26
// against 15).
// The ranges' partials (o, m, l; m in log2) are merged by k_pattn_merge, which also quantizes the output
// into the o projection's fragments (k_gemm.hip) when asked.
// 256 tokens x 16 heads over 4096 keys: 51.3 us with the merge, against 353 of k_attn_multi_q8 (P V as f32
// FMAs, a workgroup per 16 rows); error against 64 bits 2.4e-7, against 2.5e-7.
#include "ti_dev.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v4f_u __attribute__((ext_vector_type(4), aligned(4)));   // the caller's q need not be aligned

constexpr int HD = 128, NG = HD / 32, KB = 64;         // KB: keys of a staged block
constexpr int VSTRIDE = 65;                            // 16-byte pieces of a V operand tile (1 of padding: writes of
                                                       // eight tiles would meet in one bank)
constexpr float MLOW = -3.0e38f;

struct PattnArgs {
    const float* qr;
    const uint8_t* kq;
    const float* ks;
    const uint8_t* vq;
    const float* vs;
    float* po;
    float* pml;
    int S0, T, nHq, nKv, G, nsplit, per, nblk;         // S0: keys token 0 sees; per: keys of a range (multiple of KB)
    int kvs;                                           // code slots of a cached position
};

struct PattnLds {
    ti_h8 k[KB / 16][NG][64];                          // [16 keys][group][lane]: key lane % 16, dims 8 (lane / 16)..
    ti_b8 v[KB / 32][8][VSTRIDE];                       // [32 keys][16 dims][lane]: dim lane % 16, keys 4j.., 16 + 4j..
    float ks[NG][KB], vs[NG][KB];
};

// 4 x 4 bytes: in, w[r] = row r's four bytes; out, w[e] = byte e of rows 0..3
__device__ __forceinline__ void tr4_bytes(uint32_t (&w)[4]) {
    const uint32_t a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u);   // r0b0 r1b0 r0b1 r1b1
    const uint32_t b = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);   // r0b2 r1b2 r0b3 r1b3
    const uint32_t c = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
    const uint32_t d = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
    w[0] = __builtin_amdgcn_perm(c, a, 0x05040100u);
    w[1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
    w[2] = __builtin_amdgcn_perm(d, b, 0x05040100u);
    w[3] = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

__global__ __launch_bounds__(256, 3) void k_pattn(PattnArgs a) {
    __shared__ PattnLds L;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, j = lane >> 4;
    // KV head fastest: an XCD (every eighth workgroup) keeps to few heads' keys
    const int hk = blockIdx.x % a.nKv, blk = (blockIdx.x / a.nKv) % a.nblk, split = blockIdx.x / (a.nKv * a.nblk);
    const int nrows = a.G * a.T;
    const int row0 = blk * 64 + wave * 16;
    const int wgtop = min((blk + 1) * 64, nrows) - 1;
    const int c0 = split * a.per;
    const int c1 = min(a.S0 + wgtop / a.G, c0 + a.per);    // keys [c0, c1) that any row of the workgroup sees
    const size_t code_row = (size_t)a.kvs * HD, scale_row = (size_t)a.nKv * NG;
    const uint8_t* kp = a.kq + hk * HD;
    const uint8_t* vp = a.vq + hk * HD;
    const float* ksp = a.ks + hk * NG;
    const float* vsp = a.vs + hk * NG;
    const float sscale = 1.44269504088896341f / (127.0f * sqrtf((float)HD));

    // a block's loads of this thread: K 2 x 16 codes of key 16 wave + m; V 2 blocks of 4 keys x 4 dims; one scale each
    uint4 kr[2];
    uint32_t vr[2][4];
    float ksr, vsr;
    const int vdb = lane & 31, vkb = (lane >> 5) + 2 * wave;
    auto load = [&](int t0) {
#pragma unroll
        for (int u = 0; u < 2; u++)
            kr[u] = *reinterpret_cast<const uint4*>(kp + min(t0 + 16 * wave + m, c1 - 1) * code_row + 16 * (j + 4 * u));
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                vr[u][r] = *reinterpret_cast<const uint32_t*>(vp + min(t0 + 4 * (vkb + 8 * u) + r, c1 - 1) * code_row + 4 * vdb);
        const size_t s = min(t0 + (tid >> 2), c1 - 1) * scale_row + (tid & 3);
        ksr = ksp[s];
        vsr = vsp[s];
    };
    // this lane's query row: m of the wave's 16 (past the last: that one again)
    const int gr = min(row0 + m, nrows - 1), tok = gr / a.G, hq = hk * a.G + gr % a.G;
    v4f_u qv[NG][2];
    {
        const float* q = a.qr + ((size_t)tok * a.nHq + hq) * HD + 8 * j;
#pragma unroll
        for (int g = 0; g < NG; g++) {
            qv[g][0] = *reinterpret_cast<const v4f_u*>(q + 32 * g);
            qv[g][1] = *reinterpret_cast<const v4f_u*>(q + 32 * g + 4);
        }
    }
    if (c0 < c1) load(c0);

    float neg = -1.0f;                                     // opaque: q - hi as one v_fma_mix, not convert and subtract
    asm("" : "+s"(neg));
    // Q operand: dims 32 g + 8 j.., hi and lo; and the keys the row sees
    ti_h8 qh[NG], ql[NG];
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float v = qv[g][e / 4][e % 4];
            const _Float16 hi = (_Float16)v;
            qh[g][e] = hi;
            ql[g][e] = (_Float16)fmaf((float)hi, neg, v);
        }
    const int lim = min(c1, a.S0 + tok);
    // every row of the wave sees the keys below this
    const int all = min(c1, a.S0 + min(row0, nrows - 1) / a.G);

    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    v4f o[8];
    float mx = MLOW, l = 0.0f;
#pragma unroll
    for (int d = 0; d < 8; d++) o[d] = zero;
    for (int t0 = c0; t0 < c1; t0 += KB) {
        __syncthreads();                                   // the last block is read
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int c = j + 4 * u;
            L.k[wave][c >> 1][(c & 1) * 32 + m] = ti_i8x8_h8(kr[u].x, kr[u].y);
            L.k[wave][c >> 1][(c & 1) * 32 + 16 + m] = ti_i8x8_h8(kr[u].z, kr[u].w);
            const int kb = vkb + 8 * u, kk = kb & 7;       // 4-key block of its 32 keys
            tr4_bytes(vr[u]);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                ti_b8* p = &L.v[kb >> 3][vdb >> 2][(kk & 3) * 16 + 4 * (vdb & 3) + e];
                reinterpret_cast<uint2*>(p)[kk >> 2] = ti_i8x4_b4(vr[u][e]);
            }
        }
        L.ks[tid & 3][tid >> 2] = ksr;
        L.vs[tid & 3][tid >> 2] = vsr;
        __syncthreads();
        if (t0 + KB < c1) load(t0 + KB);
        TI_ISSUE_FENCE();
#pragma unroll 1
        for (int h = 0; h < KB / 32; h++) {                // 32 keys
            const int k0 = t0 + 32 * h;
            if (k0 >= c1) break;                           // workgroup-uniform
            v4f s[2];
#pragma unroll
            for (int b = 0; b < 2; b++) {
                s[b] = zero;
#pragma unroll
                for (int g = 0; g < NG; g++) {
                    const ti_h8 kk = L.k[2 * h + b][g][lane];
                    const v4f sc = *reinterpret_cast<const v4f*>(&L.ks[g][32 * h + 16 * b + 4 * j]);
                    v4f d = __builtin_amdgcn_mfma_f32_16x16x32_f16(kk, qh[g], zero, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_f16(kk, ql[g], d, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) s[b][i] = fmaf(d[i], sc[i], s[b][i]);
                }
            }
            const bool masked = k0 + 32 > all;             // wave-uniform
            float tm = MLOW;
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    s[b][i] = s[b][i] * sscale;
                    if (masked) s[b][i] = k0 + 16 * b + 4 * j + i < lim ? s[b][i] : MLOW;
                    tm = fmaxf(tm, s[b][i]);
                }
            tm = fmaxf(tm, ti_xor(tm, 16));
            tm = fmaxf(tm, ti_xor(tm, 32));
            const float mn = fmaxf(mx, tm);
            if (__any(mn > mx)) {                          // rare once the first blocks are in
                const float alpha = __builtin_amdgcn_exp2f(mx - mn);
                l = l * alpha;
#pragma unroll
                for (int d = 0; d < 8; d++) o[d] = o[d] * alpha;
                mx = mn;
            }
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float p = __builtin_amdgcn_exp2f(s[b][i] - mx);
                    if (masked) p = k0 + 16 * b + 4 * j + i < lim ? p : 0.0f;
                    s[b][i] = p;
                }
            l += ((s[0][0] + s[0][1]) + (s[0][2] + s[0][3])) + ((s[1][0] + s[1][1]) + (s[1][2] + s[1][3]));
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const v4f v0 = *reinterpret_cast<const v4f*>(&L.vs[g][32 * h + 4 * j]);
                const v4f v1 = *reinterpret_cast<const v4f*>(&L.vs[g][32 * h + 16 + 4 * j]);
                float w[8];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    w[e] = s[0][e] * v0[e];
                    w[4 + e] = s[1][e] * v1[e];
                }
                ti_b8 p[3];
                ti_bf16x3(w, p);
#pragma unroll
                for (int d = 2 * g; d < 2 * g + 2; d++) {
                    const ti_b8 vv = L.v[h][d][lane];
#pragma unroll
                    for (int i = 2; i >= 0; i--) o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, p[i], o[d], 0, 0, 0);
                }
            }
        }
    }
    l += ti_xor(l, 16);
    l += ti_xor(l, 32);
    if (row0 + m >= nrows) return;
    const size_t slot = ((size_t)tok * a.nHq + hq) * a.nsplit + split;
#pragma unroll
    for (int d = 0; d < 8; d++)
        *reinterpret_cast<v4f*>(a.po + slot * HD + 16 * d + 4 * j) = o[d];
    if (j == 0) {
        a.pml[2 * slot] = mx;
        a.pml[2 * slot + 1] = l;
    }
}

// The projections of T tokens -> what the kernel above reads (attnPrep of each token, models/qwen3.js:2228-2308):
// a wave per (token, head of q | k | v), lane l holding dims l and l + 64. q and k RMS-normalised (rope_norm's
// order) and rotated by the table's rows, k and v quantized into their cache rows (snorm int8). One launch
// of 5.4 us at 256 tokens x 32 heads against 7.9 + 7.9 + 4.7 for the rotations (which formed every angle
// in f64) and the cache write.
__global__ __launch_bounds__(256) void k_pattn_prep(const float* __restrict__ q, const float* __restrict__ k,
                                                    const float* __restrict__ v, const uint16_t* __restrict__ qw,
                                                    const uint16_t* __restrict__ kw, const float* __restrict__ rope, float eps,
                                                    float* __restrict__ qr, uint32_t* __restrict__ kq, float* __restrict__ ks,
                                                    uint32_t* __restrict__ vq, float* __restrict__ vs, int pos, int T, int nHq,
                                                    int nKv, int kvs) {
    const int lane = threadIdx.x & 63, heads = nHq + 2 * nKv;
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= T * heads) return;                            // wave-uniform
    const int t = u / heads, h = u % heads;
    const bool isq = h < nHq, isv = h >= nHq + nKv;
    const int hk = isv ? h - nHq - nKv : h - nHq;
    const float* src = isq ? q + ((size_t)t * nHq + h) * HD : (isv ? v : k) + ((size_t)t * nKv + hk) * HD;
    float a = src[lane], b = src[lane + 64];
    if (!isv) {
        const uint16_t* w = isq ? qw : kw;
        const float w0 = ti_h2f(w[lane]), w1 = ti_h2f(w[lane + 64]);
        const float* cs = rope + (size_t)(pos + t) * HD;
        const float c = cs[lane], sn = cs[lane + 64];
        float ss = a * a + b * b;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss = ss + ti_xor(ss, o);
        float mean = ss / (float)HD;
        mean = mean + eps;
        const float inv = 1.0f / sqrtf(mean);
        a = a * inv;
        a = a * w0;
        b = b * inv;
        b = b * w1;
        const float y0 = a * c + -b * sn, y1 = b * c + a * sn;
        a = y0;
        b = y1;
    }
    if (isq) {
        float* d = qr + ((size_t)t * nHq + h) * HD;
        d[lane] = a;
        d[lane + 64] = b;
        return;
    }
    const float m0 = fmaxf(ti_max32_nonneg(fabsf(a)), 1e-12f), m1 = fmaxf(ti_max32_nonneg(fabsf(b)), 1e-12f);
    const uint32_t d0 = ti_quad_or(snorm_code(a, m0) << (8 * (lane & 3))), d1 = ti_quad_or(snorm_code(b, m1) << (8 * (lane & 3)));
    uint32_t* codes = (isv ? vq : kq) + ((size_t)(pos + t) * kvs + hk) * (HD / 4);
    float* sc = (isv ? vs : ks) + ((size_t)(pos + t) * nKv + hk) * NG;
    if ((lane & 3) == 0) {
        codes[lane >> 2] = d0;
        codes[16 + (lane >> 2)] = d1;
    }
    if ((lane & 31) == 0) {
        sc[lane >> 5] = m0;
        sc[2 + (lane >> 5)] = m1;
    }
}

// The ranges' partials of a (token, head) -> its output row, a wave each. FRAG: quantized into the o
// projection's fragments (tokens past T of the last tile of 16 as zeros); else out [T][nHq][128]. Lane
// l holds dims 8 (l / 4) + l % 4 and + 4, neighbours in the fragment.
template <bool FRAG>
__global__ __launch_bounds__(256) void k_pattn_merge(const float* __restrict__ po, const float* __restrict__ pml,
                                                     float* __restrict__ out, uint32_t* __restrict__ xh,
                                                     float* __restrict__ xsc, int T, int nHq, int nsplit, int rows) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;                               // wave-uniform
    const int t = row / nHq, h = row % nHq;
    const int sl = lane >> 2, d = 8 * sl + (lane & 3);
    float v0 = 0.0f, v1 = 0.0f;
    if (t < T) {
        const float* p = po + (size_t)row * nsplit * HD + d;
        const float* ml = pml + (size_t)row * nsplit * 2;
        const float mi = lane < nsplit ? ml[2 * lane] : MLOW, li = lane < nsplit ? ml[2 * lane + 1] : 0.0f;   // nsplit <= 64
        const float w = __builtin_amdgcn_exp2f(mi - ti_wave_max(mi));
        const float lt = ti_wave_sum(li * w);
        for (int i0 = 0; i0 < nsplit; i0 += 8) {
            float a[8], b[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int i = min(i0 + k, nsplit - 1);
                a[k] = p[(size_t)i * HD];
                b[k] = p[(size_t)i * HD + 4];
            }
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float f = i0 + k < nsplit ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), i0 + k)) : 0.0f;
                v0 = fmaf(a[k], f, v0);
                v1 = fmaf(b[k], f, v1);
            }
        }
        const float inv = 127.0f * lt;
        v0 = v0 / inv;
        v1 = v1 / inv;
    }
    if constexpr (!FRAG) {
        out[(size_t)row * HD + d] = v0;
        out[(size_t)row * HD + d + 4] = v1;
    } else {
        float mx = fmaxf(fabsf(v0), fabsf(v1));
        mx = fmaxf(mx, ti_xor(mx, 1));
        mx = fmaxf(mx, ti_xor(mx, 2));
        mx = fmaxf(mx, ti_xor(mx, 4));
        mx = fmaxf(mx, ti_xor(mx, 8));
        const float scale = mx / 127.0f;
        const float inv = scale > 0.0f ? 1.0f / scale : 0.0f;
        const ti_h2 q = {(_Float16)q8_code(v0, inv), (_Float16)q8_code(v1, inv)};
        const size_t f = (size_t)(t >> 4) * nHq * NG + h * NG + (sl >> 2);
        xh[(f * 64 + 16 * (sl & 3) + (t & 15)) * 4 + (lane & 3)] = __builtin_bit_cast(uint32_t, q);
        if ((lane & 15) == 0) xsc[f * 16 + (t & 15)] = scale;
    }
}

}  // namespace

// 32 rows or fewer would leave half of a workgroup's waves idle: the short kernels keep them
bool ti_pattn_ok(int T, int nHq, int nKv, int hd) { return hd == HD && T > 1 && nHq / nKv * T > 32; }

int ti_pattn_prep_launch(ti_ctx* c, const float* q, const float* k, const float* v, const uint16_t* qw, const uint16_t* kw,
                         const float* rope, float eps, float* qr, uint32_t* kq, float* ks, uint32_t* vq, float* vs, int pos,
                         int T, int nHq, int nKv, int kvs) {
    const int units = T * (nHq + 2 * nKv);
    k_pattn_prep<<<(unsigned)((units + 3) / 4), 256, 0, c->stream>>>(q, k, v, qw, kw, rope, eps, qr, kq, ks, vq, vs, pos, T, nHq, nKv, kvs);
    TI_LAUNCHED("k_pattn_prep");
    return TI_OK;
}

// queries T at contexts S0, S0 + 1, ...: out [T][nHq][128], or (frag) the o projection's fragments
int ti_pattn_launch(ti_ctx* c, const float* qr, const uint32_t* kq, const float* ks, const uint32_t* vq, const float* vs,
                    float* out, const TiFrag* frag, int S0, int T, int nHq, int nKv, int kvs) {
    const int G = nHq / nKv, nrows = G * T, Smax = S0 + T - 1;
    const int nblk = (nrows + 63) / 64;
    const long kb = (Smax + KB - 1) / KB;
    // key ranges: a workgroup a CU, of at least two blocks (the merge reads every range's rows). us at one a CU / two:
    // 16 heads over 8, 256 tokens at 1792 34.1 / 34.1, 64 at 4000 23.7 / 23.0, 100 at 1000 18.7 / 19.3, 20 at 6000
    // 19.0 / 21.6
    const long wg = (long)nKv * nblk;
    long ns = (c->cus + wg - 1) / wg;
    if (ns > (kb + 1) / 2) ns = (kb + 1) / 2;
    // and, up to 16384 keys, of at most 256: the output's running sum rounds three times per 32 keys (256 tokens over
    // 4096 keys in ranges of 512: error 2.7e-7 and 51.5 us, of 256: 2.4e-7 and 54.7; over 16256 in ranges of 2048: 4.7e-7,
    // of 256: 2.7e-7). Past 16384 keys the merge's 64 ranges grow (32256 keys, ranges of 512: 3.2e-7; k_attn_multi_q8
    // 4.6e-7)
    if (ns < (kb + 3) / 4) ns = (kb + 3) / 4;
    if (ns > 64) ns = 64;
    if (ns * T * nHq > TI_ATTN_ROWSPLITS) ns = TI_ATTN_ROWSPLITS / ((long)T * nHq);
    if (ns < 1) ns = 1;
    const int per = (int)((kb + ns - 1) / ns) * KB;
    const int nsplit = (Smax + per - 1) / per;
    PattnArgs a = {qr, reinterpret_cast<const uint8_t*>(kq), ks, reinterpret_cast<const uint8_t*>(vq), vs, c->attn_po, c->attn_ml,
                   S0, T, nHq, nKv, G, nsplit, per, nblk, kvs};
    const unsigned grid = (unsigned)((long)nKv * nblk * nsplit);
    k_pattn<<<grid, 256, 0, c->stream>>>(a);
    TI_LAUNCHED("k_pattn");
    const int rows = (frag ? (T + 15) / 16 * 16 : T) * nHq;
    if (frag) k_pattn_merge<true><<<(rows + 3) / 4, 256, 0, c->stream>>>(c->attn_po, c->attn_ml, nullptr, frag->xh, frag->sc, T, nHq, nsplit, rows);
    else k_pattn_merge<false><<<(rows + 3) / 4, 256, 0, c->stream>>>(c->attn_po, c->attn_ml, out, nullptr, nullptr, T, nHq, nsplit, rows);
    TI_LAUNCHED("k_pattn_merge");
    return TI_OK;
}
