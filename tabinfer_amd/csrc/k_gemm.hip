// k_gemm.hip — int4 x int8 GEMM of a prompt's tokens on the matrix cores (gemmDP4A,
// models/qwen3.js:1326-1407; per-token activation quant QUANTQ8T :1210-1231; the SwiGLU before
// the down projection): every projection of more than 16 tokens, and those of 2..16 whose K the
// short-batch kernels (k_tgemm.hip) have no instance for.
//
// y[t][n] (+)= sum_g s_w[n,g] * s_x[t,g] * dot_g(t, n), dot_g the exact integer dot of the
// 32-element group g, scaled into an f32 sum as the reference does per group.
//
// What bounds it is the scaling: per token, row and group one multiply of the two scales and one
// fma, 4 cycles each per 64 of them, against 1 cycle of MFMA. The integer MFMA would add a
// conversion of every dot, so the dots are taken with v_mfma_f32_16x16x32_f16, whose f32 result
// is the integer itself: a nibble under the exponent byte 0x64 is the f16 1024 + nibble (a shift
// and an and-or for two), the codes are exact in f16, and -1032 * sum(codes) enters as the C
// operand, itself the MFMA of the codes and a constant -1032, shared by the row tiles. Every
// partial sum is an integer below 2^24 (32 * 127 * 1039 = 4.2e6 on top of C's 4.2e6), so exact.
//
// The activation comes in fragment order (k_quant_frag, k_norm_frag, the gate/up epilogue): for a
// tile of 16 tokens and a group, lane (m, j)'s 16 bytes are the codes of token m, elements 8j..8j+7
// in the order the weight word's nibbles leave the mask (0 4 1 5 2 6 3 7), so that an A operand is
// one contiguous 1 KB load of the wave, without LDS; a wave reads each for all its NT row tiles.
//
// Weights: lane (m, j) loads the 16-byte group g0 + j of row m, and a 4 x 4 transpose over the lane
// rows (tr4_rows) makes that the B operands of four groups. A wave takes 4-group steps of its
// workgroup's 16 NT rows x 16 MT tokens, every W-th one; the W sums meet in LDS. At 6144 x 2048 x 77
// (with the quantizer) 42.9 -> 13 us, at 4096 x 2048 x 256 160 -> 14.
#include "ti_dev.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int GMAX = 512;       // K <= 16384: the fragments of TI_ACT_TMAX tokens fit the context's activation scratch
static_assert(GMAX * 32 * 2 <= TI_ACT_CAP && GMAX * 4 <= TI_ACT_CAP / 32 * 4, "fragments in act_q, scales in act_s");

struct GemmArgs {
    const uint4* pack[3];
    const uint16_t* sc[3];
    float* y[3];
    int n[3];
    int blk0[3];                // first workgroup (grid x) of each matrix
    int nseg;
    int G, T, acc;
    const ti_h8* xh;            // activation fragments [tile][G][64]
    const float* xsc;           // [tile][G][16] scales
    _Float16* yh;               // gate/up: the SwiGLU's fragments [tile][N / 32][64][8]
    float* ysc;
};

// the fragment slot of element e of a group's 8-element slice
__device__ __forceinline__ int frag_slot(int e) { return ((e & 3) << 1) | (e >> 2); }

// as k_tgemm.hip's: in, lane row j holds words 0..3 of group j; out, b[u] in lane row j is word j of group u
__device__ __forceinline__ void tr4_rows(const uint4 w, uint32_t (&b)[4]) {
    const auto p = __builtin_amdgcn_permlane32_swap(w.x, w.z, false, false);
    const auto q = __builtin_amdgcn_permlane32_swap(w.y, w.w, false, false);
    const auto r0 = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    const auto r1 = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    b[0] = r0[0];
    b[1] = r0[1];
    b[2] = r1[0];
    b[3] = r1[1];
}

// GU: tiles 0, 1 are gate rows +0 / +16 of the workgroup's 32-row chunk, 2, 3 the same up rows
template <bool GU, int NT, int MT, int W>
__global__ __launch_bounds__(64 * W, 2) void k_gemm_q4(GemmArgs a) {
    static_assert(!GU || NT == 4, "gate/up: two gate and two up tiles");
    struct WaveBuf {
        float sx[MT][4][16];
        float sw[NT][4][16];
    };
    constexpr int PW = 16 * MT * 17;                       // one wave's sums of a row tile
    constexpr int STAGE = W * (int)sizeof(WaveBuf), SUMS = W * PW * 4, FRAGS = GU ? MT * 1024 : 0;
    __shared__ __align__(16) char s_mem[STAGE > SUMS ? STAGE : SUMS];
    __shared__ __align__(16) char s_frag[FRAGS ? FRAGS : 16];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, j = lane >> 4;
    const int G = a.G, ntile = (a.T + 15) / 16;
    const int b = blockIdx.x, tile0 = blockIdx.y * MT;
    WaveBuf& L = reinterpret_cast<WaveBuf*>(s_mem)[wave];

    const int mi = GU ? 0 : (a.nseg > 1 && b >= a.blk0[1]) + (a.nseg > 2 && b >= a.blk0[2]);
    const int N = mi == 0 ? a.n[0] : (mi == 1 ? a.n[1] : a.n[2]);
    const int row0 = GU ? 32 * b : (b - (mi == 0 ? 0 : (mi == 1 ? a.blk0[1] : a.blk0[2]))) * 16 * NT;
    const uint4* wr[NT];
    const uint16_t* sr[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const int s = GU ? n / 2 : mi;
        const uint4* p = s == 0 ? a.pack[0] : (s == 1 ? a.pack[1] : a.pack[2]);
        const uint16_t* q = s == 0 ? a.sc[0] : (s == 1 ? a.sc[1] : a.sc[2]);
        const size_t row = min(row0 + 16 * (GU ? n % 2 : n) + m, N - 1);
        wr[n] = p + row * G;
        sr[n] = q + row * G;
    }
    size_t tg[MT];                                         // (tile, group 0) of each token tile
#pragma unroll
    for (int t = 0; t < MT; t++) tg[t] = (size_t)min(tile0 + t, ntile - 1) * G;

    uint4 wv[NT];
    uint16_t sw[NT];
    float sx[MT];
    auto load_step = [&](int st) {                         // past the last group: it again, scaled by 0
        const int g = min(4 * st + j, G - 1);
#pragma unroll
        for (int n = 0; n < NT; n++) {
            wv[n] = wr[n][g];
            sw[n] = sr[n][g];
        }
#pragma unroll
        for (int t = 0; t < MT; t++) sx[t] = a.xsc[(tg[t] + g) * 16 + m];
    };
    ti_h8 A[2][MT];
    auto load_a = [&](ti_h8 (&d)[MT], int g) {
        g = min(g, G - 1);
#pragma unroll
        for (int t = 0; t < MT; t++) d[t] = a.xh[(tg[t] + g) * 64 + lane];
    };
    v4f acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[n][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    // opaque: as literals the and and the or would stay two instructions
    uint32_t nib = 0x000F000Fu, magic = 0x64006400u;
    asm("" : "+s"(nib));
    asm("" : "+v"(magic));
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const _Float16 mb = (_Float16)-1032.0f;
    const ti_h8 bias = {mb, mb, mb, mb, mb, mb, mb, mb};
    load_step(wave);
    load_a(A[0], 4 * wave);
    for (int st = wave; 4 * st < G; st += W) {
        uint32_t bw[NT][4];
        ti_wave_lds_fence();                                  // the last step's reads are done
#pragma unroll
        for (int n = 0; n < NT; n++) {
            L.sw[n][j][m] = 4 * st + j < G ? ti_h2f(sw[n]) : 0.0f;
            tr4_rows(wv[n], bw[n]);
        }
#pragma unroll
        for (int t = 0; t < MT; t++) L.sx[t][j][m] = sx[t];
        ti_wave_lds_fence();
        load_step(st + W);
        TI_ISSUE_FENCE();
#pragma unroll
        for (int u = 0; u < 4; u++) {
            load_a(A[(u + 1) & 1], u < 3 ? 4 * st + u + 1 : 4 * (st + W));
            v4f xs4[MT], cr[MT], d[2][MT];
            float s[NT];
#pragma unroll
            for (int t = 0; t < MT; t++) xs4[t] = *reinterpret_cast<const v4f*>(&L.sx[t][u][4 * j]);
#pragma unroll
            for (int n = 0; n < NT; n++) s[n] = L.sw[n][u][m];
#pragma unroll
            for (int t = 0; t < MT; t++) cr[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[u & 1][t], bias, zero, 0, 0, 0);
            // the next row tile's dots are under way while this one's are scaled
            auto dots = [&](int n) {
                const uint32_t w = bw[n][u];
                const uint4 bb = make_uint4((w & nib) | magic, ((w >> 4) & nib) | magic, ((w >> 8) & nib) | magic,
                                            ((w >> 12) & nib) | magic);
                const ti_h8 B = __builtin_bit_cast(ti_h8, bb);
#pragma unroll
                for (int t = 0; t < MT; t++)
                    d[n & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[u & 1][t], B, cr[t], 0, 0, 0);
            };
            dots(0);
#pragma unroll
            for (int n = 0; n < NT; n++) {
                if (n + 1 < NT) dots(n + 1);
                TI_ISSUE_FENCE();
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[n][t][i] = fmaf(d[n & 1][t][i], s[n] * xs4[t][i], acc[n][t][i]);
            }
        }
    }

    // the waves' sums, a row tile at a time: [wave][16 MT tokens][16 rows + 1]
    constexpr int NE = (256 * MT + 64 * W - 1) / (64 * W);   // a thread's (token, row) pairs of a tile
    float* part = reinterpret_cast<float*>(s_mem);
    auto tile_sum = [&](int n, float (&v)[NE]) {
        __syncthreads();                                   // s_mem is free
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) part[wave * PW + (16 * t + 4 * j + i) * 17 + m] = acc[n][t][i];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < NE; r++) {
            const int e = tid + 64 * W * r;
            v[r] = 0.0f;
            if (e < 256 * MT) {
#pragma unroll
                for (int k = 0; k < W; k++) v[r] += part[k * PW + (e >> 4) * 17 + (e & 15)];
            }
        }
    };
    if constexpr (!GU) {
        float* y = mi == 0 ? a.y[0] : (mi == 1 ? a.y[1] : a.y[2]);
        auto at = [&](int n, int r, size_t& o) {
            const int e = tid + 64 * W * r, tok = 16 * tile0 + (e >> 4), row = row0 + 16 * n + (e & 15);
            o = (size_t)tok * N + row;
            return e < 256 * MT && tok < a.T && row < N;
        };
        float old[NT][NE] = {};
        if (a.acc) {
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int r = 0; r < NE; r++) {
                    size_t o;
                    if (at(n, r, o)) old[n][r] = y[o];
                }
        }
#pragma unroll
        for (int n = 0; n < NT; n++) {
            float v[NE];
            tile_sum(n, v);
#pragma unroll
            for (int r = 0; r < NE; r++) {
                size_t o;
                if (at(n, r, o)) y[o] = a.acc ? old[n][r] + v[r] : v[r];
            }
        }
    } else {
        // silu(g) * u and quantQ8 over the chunk's 32 rows, as fragments of the down projection's input
        float v[4][NE];
#pragma unroll
        for (int n = 0; n < 4; n++) tile_sum(n, v[n]);
        _Float16* f = reinterpret_cast<_Float16*>(s_frag);
        const int Gy = N / 32;
#pragma unroll
        for (int r = 0; r < NE; r++) {
            const int e = tid + 64 * W * r, tok = e >> 4, row = e & 15;
            const float v0 = silu_mul(v[0][r], v[2][r]), v1 = silu_mul(v[1][r], v[3][r]);
            float mx = fmaxf(fabsf(v0), fabsf(v1));
            mx = fmaxf(mx, ti_xor(mx, 1));
            mx = fmaxf(mx, ti_xor(mx, 2));
            mx = fmaxf(mx, ti_xor(mx, 4));
            mx = fmaxf(mx, ti_xor(mx, 8));
            const float scale = mx / 127.0f;
            const float inv = scale > 0.0f ? 1.0f / scale : 0.0f;
            const int q0 = q8_code(v0, inv), q1 = q8_code(v1, inv);
            if (e < 256 * MT) {                            // rows 0..15 are slices 0, 1; 16..31 slices 2, 3
                const int base = (tok >> 4) * 512 + (tok & 15) * 8 + (row >> 3) * 128 + frag_slot(row & 7);
                f[base] = (_Float16)q0;
                f[base + 256] = (_Float16)q1;
                const int tile = tile0 + (tok >> 4);
                if (row == 0 && tile < ntile) a.ysc[((size_t)tile * Gy + b) * 16 + (tok & 15)] = scale;
            }
        }
        __syncthreads();
        for (int e = tid; e < 64 * MT; e += 64 * W) {
            const int tile = tile0 + (e >> 6);
            if (tile < ntile)
                reinterpret_cast<ti_h8*>(a.yh)[((size_t)tile * Gy + b) * 64 + (e & 63)] = reinterpret_cast<const ti_h8*>(s_frag)[e];
        }
    }
}

// 8 consecutive elements of a group (lane pair-of-pairs `o1`, `o2` apart hold the group): quantQ8
// (q8_group's arithmetic) as a fragment slice, and the group's scale
__device__ __forceinline__ ti_h8 quant_slice(const float (&v)[8], int o1, int o2, float& scale) {
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[i]));
    mx = fmaxf(mx, ti_xor(mx, o1));
    mx = fmaxf(mx, ti_xor(mx, o2));
    scale = mx / 127.0f;
    const float inv = scale > 0.0f ? 1.0f / scale : 0.0f;
    ti_h8 h;
#pragma unroll
    for (int i = 0; i < 8; i++) h[((i & 3) << 1) | (i >> 2)] = (_Float16)q8_code(v[i], inv);
    return h;
}

// x [T][32 G] -> fragments; a wave per (tile of 16 tokens, group); tokens past T are zero
__global__ __launch_bounds__(256) void k_quant_frag(const float* __restrict__ x, ti_h8* __restrict__ xh,
                                                    float* __restrict__ xsc, int T, int G, int nfrag) {
    const int lane = threadIdx.x & 63, m = lane & 15, j = lane >> 4;
    const int f = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (f >= nfrag) return;                                // wave-uniform
    const int tok = f / G * 16 + m, g = f % G;
    float v[8] = {};
    if (tok < T) {
        const float4* p = reinterpret_cast<const float4*>(x + ((size_t)tok * G + g) * 32 + 8 * j);
        const float4 p0 = p[0], p1 = p[1];
        v[0] = p0.x; v[1] = p0.y; v[2] = p0.z; v[3] = p0.w;
        v[4] = p1.x; v[5] = p1.y; v[6] = p1.z; v[7] = p1.w;
    }
    float scale;
    xh[(size_t)f * 64 + lane] = quant_slice(v, 16, 32, scale);
    if (j == 0) xsc[(size_t)f * 16 + m] = scale;
}

// RMSNorm (the reference's 256 strided partials and tree, as k_rmsnorm) + quantQ8 -> fragments;
// a workgroup per token. KU: H <= 256 KU, every load issued before the first sum waits (2048 wide, 256
// tokens: 6.0 -> 4.9 us); KU = 0: any H. Elements past H are left out of their partial.
template <int KU>
__global__ __launch_bounds__(256) void k_norm_frag(const float* __restrict__ x, const uint16_t* __restrict__ nw, float eps,
                                                   ti_h8* __restrict__ xh, float* __restrict__ xsc, int T, int H) {
    __shared__ float red[256];
    constexpr int NC = KU ? (KU + 7) / 8 : 1;              // 8-element chunks of a thread
    const int tok = blockIdx.x, G = H / 32, t = threadIdx.x;
    const size_t f0 = (size_t)(tok >> 4) * G;
    const int m = tok & 15;
    const bool live = tok < T;                             // the last tile's other tokens are zero
    const float* xr = x + (size_t)min(tok, T - 1) * H;
    float4 p[NC][2];
    uint4 w4[NC];
    auto load = [&](int k, int c) {
        const float4* s = reinterpret_cast<const float4*>(xr + 8 * c);
        p[k][0] = s[0];
        p[k][1] = s[1];
        w4[k] = *reinterpret_cast<const uint4*>(nw + 8 * c);
    };
    float inv_rms;
    if constexpr (KU > 0) {
        float xs[KU];
#pragma unroll
        for (int i = 0; i < KU; i++) xs[i] = xr[min(t + 256 * i, H - 1)];
#pragma unroll
        for (int k = 0; k < NC; k++) load(k, min(t + 256 * k, H / 8 - 1));
        TI_ISSUE_FENCE();
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < KU; i++) {
            const float sq = xs[i] * xs[i];
            s = t + 256 * i < H ? s + sq : s;
        }
        float mean = ti_tree_sum_256(s, red) / (float)H;
        mean = mean + eps;
        inv_rms = 1.0f / sqrtf(mean);
    } else {
        inv_rms = rms_inv_256(xr, H, eps, red);
    }
    auto chunk = [&](int k, int c) {
        const uint32_t w[4] = {w4[k].x, w4[k].y, w4[k].z, w4[k].w};
        float v[8] = {p[k][0].x, p[k][0].y, p[k][0].z, p[k][0].w, p[k][1].x, p[k][1].y, p[k][1].z, p[k][1].w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float n = v[i] * inv_rms;
            const float s = n * ti_h2f((uint16_t)(w[i / 2] >> (16 * (i & 1))));
            v[i] = live ? s : 0.0f;
        }
        float scale;
        const ti_h8 h = quant_slice(v, 1, 2, scale);
        const int g = c >> 2, j = c & 3;
        xh[(f0 + g) * 64 + 16 * j + m] = h;
        if (j == 0) xsc[(f0 + g) * 16 + m] = scale;
    };
    // H / 8 is a multiple of 4: a group's four lanes stay together
    if constexpr (KU > 0) {
#pragma unroll
        for (int k = 0; k < NC; k++)
            if (t + 256 * k < H / 8) chunk(k, t + 256 * k);
    } else {
        for (int c = t; c < H / 8; c += 256) {
            load(0, c);
            chunk(0, c);
        }
    }
}

template <bool GU, int NT, int MT, int W>
void launch(ti_ctx* c, GemmArgs& a) {
    long blocks = 0;
    for (int i = 0; i < 3; i++) {
        a.blk0[i] = (int)blocks;
        if (i < a.nseg) blocks += GU ? a.n[0] / 32 : ((long)a.n[i] + 16 * NT - 1) / (16 * NT);
    }
    const int ntile = (a.T + 15) / 16;
    k_gemm_q4<GU, NT, MT, W><<<dim3((unsigned)blocks, (unsigned)((ntile + MT - 1) / MT)), 64 * W, 0, c->stream>>>(a);
}

// The smallest tile whose workgroups (8 waves) still find a CU each: a second round costs more than
// a larger tile. us at tiles of NT x MT, 8 waves: 4096 rows x 2048 x 32 tokens 1x1 (512 workgroups) 7.2,
// 1x2 (256) 5.0, 2x2 6.7; 2048 x 6144 x 64 1x1 (512) 12.2, 1x2 (256) 9.8, 1x4 12.8; 6144 x 2048 x 77 1x4 (768)
// 14.2, 2x4 (384) 16.0, 2x5 (192) 10.1. Past that, workgroups of 4 waves, two or three on a CU: 4096 x 2048 x 256
// 2x4 in 8 waves 16.6, in 4 waves 13.4; 6144 x 2048 x 256 2x4 (768) 19.7, 4x4 21.4; 8192 x 2048 x 256 2x4 (1024)
// 24.0, 4x4 22.1.
void pick(ti_ctx* c, GemmArgs& a) {
    const long tt = (a.T + 15) / 16;
    auto groups = [&](int nt, int mt) {
        long b = 0;
        for (int i = 0; i < a.nseg; i++) b += ((long)a.n[i] + 16 * nt - 1) / (16 * nt);
        return b * ((tt + mt - 1) / mt);
    };
    auto fits = [&](int nt, int mt) { return groups(nt, mt) <= c->cus; };
    if (fits(1, 1) || (tt == 1 && groups(1, 1) <= 2 * c->cus)) launch<false, 1, 1, 8>(c, a);
    else if (fits(1, 2)) launch<false, 1, 2, 8>(c, a);
    else if (fits(1, 3)) launch<false, 1, 3, 8>(c, a);
    else if (fits(1, 4)) launch<false, 1, 4, 8>(c, a);
    else if (fits(2, 2)) launch<false, 2, 2, 8>(c, a);
    else if (fits(2, 3)) launch<false, 2, 3, 8>(c, a);
    else if (fits(2, 4)) launch<false, 2, 4, 8>(c, a);
    else if (fits(2, 5)) launch<false, 2, 5, 8>(c, a);
    else if (groups(2, 4) <= 3 * c->cus) launch<false, 2, 4, 4>(c, a);
    else launch<false, 4, 4, 4>(c, a);
}

// The same for gate/up (one 32-row chunk a workgroup). us at 6144 x 2048: 17 tokens MT 1 16.0, 2 11.5, 4 14.8;
// 64 tokens MT 4 14.7, 2 20.2; 256 tokens MT 4 in 8 waves 39.9, in 4 waves 32.6.
void pick_gateup(ti_ctx* c, GemmArgs& a) {
    const long tt = (a.T + 15) / 16, chunks = a.n[0] / 32;
    auto fits = [&](int mt) { return chunks * ((tt + mt - 1) / mt) <= c->cus; };
    if (fits(1)) launch<true, 4, 1, 8>(c, a);
    else if (fits(2)) launch<true, 4, 2, 8>(c, a);
    else if (fits(3)) launch<true, 4, 3, 8>(c, a);
    else if (fits(4)) launch<true, 4, 4, 8>(c, a);
    else launch<true, 4, 4, 4>(c, a);
}

}  // namespace

bool ti_gemm_ok(int K) { return K % 32 == 0 && K / 32 <= GMAX; }
size_t ti_frag_words(int T, int K) { return (size_t)((T + 15) / 16) * (K / 32) * 256; }   // 32-bit words of TiFrag::xh
size_t ti_frag_scales(int T, int K) { return (size_t)((T + 15) / 16) * (K / 32) * 16; }   // floats of TiFrag::sc

int ti_quant_frag_launch(ti_ctx* c, const float* x, const TiFrag& f, int T, int K) {
    const int G = K / 32, nfrag = (T + 15) / 16 * G;
    k_quant_frag<<<(unsigned)((nfrag + 3) / 4), 256, 0, c->stream>>>(x, reinterpret_cast<ti_h8*>(f.xh), f.sc, T, G, nfrag);
    TI_LAUNCHED("k_quant_frag");
    return TI_OK;
}

int ti_norm_frag_launch(ti_ctx* c, const float* x, const uint16_t* w, float eps, const TiFrag& f, int T, int H) {
    const unsigned grid = (unsigned)((T + 15) / 16 * 16);
    ti_h8* xh = reinterpret_cast<ti_h8*>(f.xh);
    if (H <= 1024) k_norm_frag<4><<<grid, 256, 0, c->stream>>>(x, w, eps, xh, f.sc, T, H);
    else if (H <= 2048) k_norm_frag<8><<<grid, 256, 0, c->stream>>>(x, w, eps, xh, f.sc, T, H);
    else if (H <= 4096) k_norm_frag<16><<<grid, 256, 0, c->stream>>>(x, w, eps, xh, f.sc, T, H);
    else k_norm_frag<0><<<grid, 256, 0, c->stream>>>(x, w, eps, xh, f.sc, T, H);
    TI_LAUNCHED("k_norm_frag");
    return TI_OK;
}

// y_s[t][:] (+)= W_s a_t for up to three matrices sharing the activation f
int ti_gemm_q4_launch(ti_ctx* c, const TiFrag& f, int nseg, const uint32_t* const* packs, const uint16_t* const* scs,
                      float* const* ys, const int* Ns, int T, int K, int acc) {
    if (!ti_gemm_ok(K)) return ti_fail(TI_ERR_INVALID, "int4 GEMM: K=%d must be a multiple of 32, <= %d", K, GMAX * 32);
    GemmArgs a = {};
    for (int i = 0; i < 3; i++) {
        const int s = i < nseg ? i : nseg - 1;
        if (T <= 0 || Ns[s] <= 0) return ti_fail(TI_ERR_INVALID, "int4 GEMM: T=%d N=%d", T, Ns[s]);
        a.pack[i] = reinterpret_cast<const uint4*>(packs[s]);
        a.sc[i] = scs[s];
        a.y[i] = ys[s];
        a.n[i] = Ns[s];
    }
    a.nseg = nseg;
    a.G = K / 32;
    a.T = T;
    a.acc = acc;
    a.xh = reinterpret_cast<const ti_h8*>(f.xh);
    a.xsc = f.sc;
    pick(c, a);
    TI_LAUNCHED("k_gemm_q4");
    return TI_OK;
}

// out = quantQ8(silu(Wg a_t) * (Wu a_t)) as fragments; I a multiple of 32
int ti_gemm_gateup_launch(ti_ctx* c, const TiFrag& f, const uint32_t* gpack, const uint16_t* gsc, const uint32_t* upack,
                          const uint16_t* usc, int I, int H, int T, const TiFrag& out) {
    if (!ti_gemm_ok(H) || I % 32 || T <= 0 || I <= 0) return ti_fail(TI_ERR_INVALID, "int4 gate/up GEMM: T=%d H=%d I=%d", T, H, I);
    GemmArgs a = {};
    for (int i = 0; i < 3; i++) {
        a.pack[i] = reinterpret_cast<const uint4*>(i ? upack : gpack);
        a.sc[i] = i ? usc : gsc;
        a.n[i] = I;
    }
    a.nseg = 1;
    a.G = H / 32;
    a.T = T;
    a.xh = reinterpret_cast<const ti_h8*>(f.xh);
    a.xsc = f.sc;
    a.yh = reinterpret_cast<_Float16*>(out.xh);
    a.ysc = out.sc;
    pick_gateup(c, a);
    TI_LAUNCHED("k_gemm_q4 (gate/up)");
    return TI_OK;
}
