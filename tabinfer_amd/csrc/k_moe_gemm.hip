// k_moe_gemm.hip — the int3 experts of a prompt's tokens on the matrix cores (moeSort + moeGemm3,
// models/lfm25.js:1503-1647; quantAct8 :1487-1494; swiglu :1831-1847): one workgroup per (rows,
// expert) lists the expert's (token, expert) pairs and multiplies its rows with all of them.
//
//   y[pair, n] = sum_g s_w[n,g] * s_x[pair,g] * dot_g,  dot_g the exact integer dot of 32 codes
//
// dot_g is one v_mfma_f32_16x16x32_f16 for 16 pairs x 16 rows: codes of +-127 and weights of -4..3
// are exact in f16 and every partial sum is an integer below 2^24. Of a weight's f16 only the high
// byte is not zero, so v_perm_b32 looks it up from the 3-bit code (q3_f16).
//
// Lane (m, j) loads the whole group g0 + j of row m (12 bytes and a scale), gathers its planes to
// code nibbles (q3_nibs), and a 4 x 4 transpose over the lane rows hands lane row j the word j of four
// groups: elements j, j+4, j+8, ... The activation rows are written in that order (moe_slot), so
// that lane (pair, j) reads its A operand with one 16-byte load.
//
// What bounds it at 16 pairs an expert is VALU work, 16 operations a (16 rows, group) to expand and
// 8 a (16 rows, 16 pairs, group) to scale, beside the weights' way from HBM: the next step's weights are
// asked for at the start of one (loads return in order, so the wait for the second group's A operands, asked
// for behind them, is a wait for them too), and three workgroups share a CU. The block of 128 tokens x
// top-4 of 32 experts (2048 x 1792) takes 120 us on the same inputs again and 125 to 138 on others each time (78 + 41
// of them here in a trace), against 186 to 190 with the kernel before (dot4 in registers, a reduction over the lanes
// per pair).
#include "ti_dev.h"
#include "ti_moe.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
struct Planes {                    // a group's three bitplanes
    uint32_t b[3];
};

constexpr int W = 4;               // waves of a workgroup: every fourth 4-group step each

struct MoeGemm {
    const ti_h8* xh;               // activation rows [row][G][4][8]
    const float* xs;               // [row][G]
    const uint32_t* p3[2];         // w (GU: w1, w3), all experts' rows
    const uint16_t* s3[2];
    const int32_t* ridx;           // expert of each pair
    float* y[2];                   // [pair][N] (GU: gate, up)
    float* act;                    // GU: silu(gate) * up [pair][N], and quantized
    _Float16* yh;
    float* ys;
    int P, N, G, src_div;
};

__device__ __forceinline__ void tr4(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t (&o)[4]) {
    const auto p = __builtin_amdgcn_permlane32_swap(a, c, false, false);
    const auto q = __builtin_amdgcn_permlane32_swap(b, d, false, false);
    const auto r0 = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    const auto r1 = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    o[0] = r0[0];
    o[1] = r0[1];
    o[2] = r1[0];
    o[3] = r1[1];
}

// eight 3-bit codes in nibbles -> the weights (code - 4) in f16, nibbles 0 4 2 6 | 1 5 3 7
__device__ __forceinline__ ti_h8 q3_f16(uint32_t x) {
    // high bytes of f16 -4 -3 -2 -1 | 0 1 2 3
    const uint32_t h0 = __builtin_amdgcn_perm(0x42403C00u, 0xBCC0C2C4u, x & 0x07070707u);
    const uint32_t h1 = __builtin_amdgcn_perm(0x42403C00u, 0xBCC0C2C4u, (x >> 4) & 0x07070707u);
    // selector byte 0x0c: zero
    const uint4 w = make_uint4(__builtin_amdgcn_perm(h0, h0, 0x020C000Cu), h0 & 0xFF00FF00u,
                               __builtin_amdgcn_perm(h1, h1, 0x020C000Cu), h1 & 0xFF00FF00u);
    return __builtin_bit_cast(ti_h8, w);
}

constexpr int SCAN = 1024;         // routing ids listed at a time: a second list would read the weights again
constexpr int MTX = 2;             // 16-pair tiles of one pass, at most

template <int NT>
struct MoeLds {                    // a wave's sums [tile][lane] and scales of one step
    v4f acc[NT * MTX][64];
    float sx[MTX][4][16], sw[NT][4][16];
};

template <int NT>
struct MoeStep {                   // a lane's loads of one step: group 4 st + j of its row in each tile
    Planes p[NT];
    uint16_t s[NT];
};

template <int NT>
struct MoeRows {                   // the workgroup's rows: base of each tile's matrix, this lane's row in it
    const Planes* p[NT];
    const uint16_t* s[NT];
    uint32_t off[NT];              // in groups, from the workgroup's first row
    __device__ __forceinline__ void load(MoeStep<NT>& z, int st, int G) const {
        const int g = min(4 * st + (int)((threadIdx.x & 63) >> 4), G - 1);
#pragma unroll
        for (int n = 0; n < NT; n++) {
            z.p[n] = p[n][off[n] + g];
            z.s[n] = s[n][off[n] + g];
        }
    }
};

// L.acc[NT t + n] = this wave's sums of row tile n with the pairs list[16 t .. 16 t + 15] (past cnt: the last
// again). A step's four groups are summed in registers and added to LDS: chains of 4 and 4 where
// one running sum would be a chain of 16 (an error 1.25 times the row kernels', and the more
// codes of the SwiGLU rounded otherwise), and no registers for the running sums.
template <int NT, int MT>
__device__ __forceinline__ void moe_sums(const MoeGemm& a, const MoeRows<NT>& rows, MoeStep<NT>& z, bool loaded, const int* list, int cnt, MoeLds<NT>& L) {
    const int lane = threadIdx.x & 63, m = lane & 15, j = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = a.G;
    uint32_t x0[MT];                                       // first group of each pair's activation row
#pragma unroll
    for (int t = 0; t < MT; t++) x0[t] = (uint32_t)(list[min(16 * t + m, cnt - 1)] / a.src_div) * G;
    float xn[MT];
    auto load_x = [&](int st) {
        const int g = min(4 * st + j, G - 1);
#pragma unroll
        for (int t = 0; t < MT; t++) xn[t] = a.xs[x0[t] + g];
    };
    ti_h8 A[2][MT];
    auto load_a = [&](ti_h8 (&d)[MT], int g) {
        g = min(g, G - 1);
#pragma unroll
        for (int t = 0; t < MT; t++) d[t] = a.xh[(x0[t] + g) * 4 + j];
    };
    if (!loaded) rows.load(z, wave, G);
    load_x(wave);
    load_a(A[0], 4 * wave);
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    if (4 * wave >= G) {
#pragma unroll
        for (int k = 0; k < NT * MT; k++) L.acc[k][lane] = zero;
    }
    for (int st = wave; 4 * st < G; st += W) {
        uint32_t nib[NT][4];
        v4f sum[NT][MT];
        ti_wave_lds_fence();                                  // the last step's reads are done
#pragma unroll
        for (int t = 0; t < MT; t++) L.sx[t][j][m] = xn[t];
#pragma unroll
        for (int n = 0; n < NT; n++) {
            L.sw[n][j][m] = 4 * st + j < G ? ti_h2f(z.s[n]) : 0.0f;   // past the last group: it again, scaled by 0
            uint32_t x[4];
            q3_nibs(z.p[n].b[0], z.p[n].b[1], z.p[n].b[2], x);
            tr4(x[0], x[1], x[2], x[3], nib[n]);
        }
        ti_wave_lds_fence();
        rows.load(z, st + W, G);
        load_x(st + W);
        TI_ISSUE_FENCE();
#pragma unroll
        for (int u = 0; u < 4; u++) {
            load_a(A[(u + 1) & 1], u < 3 ? 4 * st + u + 1 : 4 * (st + W));
            v4f xs4[MT], d[2][MT];
            float sw[NT];
#pragma unroll
            for (int t = 0; t < MT; t++) xs4[t] = *reinterpret_cast<const v4f*>(&L.sx[t][u][4 * j]);
#pragma unroll
            for (int n = 0; n < NT; n++) sw[n] = L.sw[n][u][m];
            auto dots = [&](int n) {                       // the next tile's are under way while one is scaled
                const ti_h8 B = q3_f16(nib[n][u]);
#pragma unroll
                for (int t = 0; t < MT; t++) d[n & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[u & 1][t], B, zero, 0, 0, 0);
            };
            dots(0);
#pragma unroll
            for (int n = 0; n < NT; n++) {
                if (n + 1 < NT) dots(n + 1);
                TI_ISSUE_FENCE();
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float sc = xs4[t][i] * sw[n];
                        sum[n][t][i] = u ? fmaf(d[n & 1][t][i], sc, sum[n][t][i]) : d[n & 1][t][i] * sc;
                    }
            }
        }
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int n = 0; n < NT; n++) {
                v4f* p = &L.acc[NT * t + n][lane];
                *p = st == wave ? sum[n][t] : *p + sum[n][t];
            }
    }
}

// grid (row blocks, experts). GU: 32 rows of w1 and of w3 (gate tiles 0, 1, up tiles 2, 3), else 16 NT rows of w
template <bool GU, int NT>
__global__ __launch_bounds__(64 * W, 2) void k_moe_gemm(MoeGemm a) {
    static_assert(!GU || NT == 4, "two gate and two up tiles");
    __shared__ int s_list[SCAN];
    __shared__ int s_wcnt[SCAN / 64];
    __shared__ __align__(16) MoeLds<NT> s_lds[W];
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, j = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int e = blockIdx.y, N = a.N, G = a.G;
    const int row0 = blockIdx.x * (GU ? 32 : 16 * NT);
    MoeRows<NT> rows;
    const size_t first = ((size_t)e * N + row0) * G;
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const int s = GU ? n / 2 : 0;
        rows.p[n] = reinterpret_cast<const Planes*>(s ? a.p3[1] : a.p3[0]) + first;
        rows.s[n] = (s ? a.s3[1] : a.s3[0]) + first;
        rows.off[n] = (uint32_t)min(16 * (GU ? n % 2 : n) + m, N - 1 - row0) * G;
    }
    // the first routing ids before the weights (in the compiled code the scan's first wait is for both: the loop's
    // later lists are asked for behind the weights)
    constexpr int NQ = SCAN / (64 * W);
    int rid[NQ];
    auto load_ids = [&](int c0) {
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int p = c0 + 64 * W * q + tid;
            rid[q] = p < a.P ? a.ridx[p] : -1;
        }
    };
    load_ids(0);
    MoeStep<NT> z;
    rows.load(z, wave, G);                                 // (few experts have no pair: k_moe.hip's rule)
    bool fresh = true;                                     // z holds the first step
    for (int c0 = 0; c0 < a.P; c0 += SCAN) {
        if (c0) load_ids(c0);
        uint64_t hits[NQ];
        __syncthreads();                                   // the last list is consumed
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            hits[q] = __ballot(rid[q] == e);
            if (lane == 0) s_wcnt[W * q + wave] = __popcll(hits[q]);
        }
        __syncthreads();
        int tot = 0;
#pragma unroll
        for (int k = 0; k < NQ * W; k++) {
            const int q = k / W;
            if (k % W == wave && rid[q] == e)
                s_list[tot + __popcll(hits[q] & ((1ull << lane) - 1ull))] = c0 + 64 * W * q + tid;
            tot += s_wcnt[k];
        }
        __syncthreads();
        for (int i0 = 0; i0 < tot; i0 += 16 * MTX) {       // workgroup-uniform
            const int cnt = min(tot - i0, 16 * MTX);
            auto pass = [&](auto mtc) {
                constexpr int MT = decltype(mtc)::value;
                moe_sums<NT, MT>(a, rows, z, fresh, s_list + i0, cnt, s_lds[wave]);
                fresh = false;
                __syncthreads();
                // row tile n's sums: thread -> (pair 16 r + tid / 16, row tid % 16)
                auto tile_sum = [&](int n, float (&v)[MT]) {
#pragma unroll
                    for (int r = 0; r < MT; r++) {
                        float q[W];
#pragma unroll
                        for (int w = 0; w < W; w++) q[w] = s_lds[w].acc[NT * r + n][(tid & 15) + 16 * (tid >> 6)][(tid >> 4) & 3];
                        v[r] = (q[0] + q[1]) + (q[2] + q[3]);
                    }
                };
                if constexpr (!GU) {
#pragma unroll
                    for (int n = 0; n < NT; n++) {
                        float v[MT];
                        tile_sum(n, v);
                        const int row = row0 + 16 * n + (tid & 15);
#pragma unroll
                        for (int r = 0; r < MT; r++) {
                            const int k = 16 * r + (tid >> 4);
                            if (k < cnt && row < N) a.y[0][(size_t)s_list[i0 + k] * N + row] = v[r];
                        }
                    }
                } else {
                    float v[4][MT];
#pragma unroll
                    for (int n = 0; n < 4; n++) tile_sum(n, v[n]);
#pragma unroll
                    for (int r = 0; r < MT; r++) {
                        const int k = 16 * r + (tid >> 4), row = tid & 15;
                        const float a0 = v[0][r] / (1.0f + expf(-v[0][r])) * v[2][r];
                        const float a1 = v[1][r] / (1.0f + expf(-v[1][r])) * v[3][r];
                        float mx = fmaxf(fabsf(a0), fabsf(a1));   // quantAct8 over the 32 rows
                        mx = fmaxf(mx, ti_xor(mx, 1));
                        mx = fmaxf(mx, ti_xor(mx, 2));
                        mx = fmaxf(mx, ti_xor(mx, 4));
                        mx = fmaxf(mx, ti_xor(mx, 8));
                        const float scale = mx / 127.0f;
                        const float inv = scale > 0.0f ? 1.0f / scale : 0.0f;
                        if (k < cnt) {
                            const size_t pair = s_list[i0 + k];
                            const size_t o = pair * N + row0 + row;
                            a.y[0][o] = v[0][r];
                            a.y[0][o + 16] = v[1][r];
                            a.y[1][o] = v[2][r];
                            a.y[1][o + 16] = v[3][r];
                            a.act[o] = a0;
                            a.act[o + 16] = a1;
                            _Float16* h = a.yh + pair * N + row0;
                            h[moe_slot(row)] = (_Float16)q8_code(a0, inv);
                            h[moe_slot(row + 16)] = (_Float16)q8_code(a1, inv);
                            if (row == 0) a.ys[pair * (N / 32) + blockIdx.x] = scale;
                        }
                    }
                }
            };
            if (cnt <= 16) pass(std::integral_constant<int, 1>{});
            else pass(std::integral_constant<int, 2>{});
            __syncthreads();                               // the sums are read
        }
    }
}

}  // namespace

// x rows as moe_slot-ordered f16 codes xh with scales xs; ridx names each pair's expert, pair p reads row p / src_div
int ti_moe_gemm_launch(ti_ctx* c, const uint16_t* xh, const float* xs, const uint32_t* p3, const uint16_t* s3,
                       const int32_t* ridx, float* y, int P, int N, int K, int src_div, int nE) {
    MoeGemm a = {};
    a.xh = reinterpret_cast<const ti_h8*>(xh);
    a.xs = xs;
    a.p3[0] = a.p3[1] = p3;
    a.s3[0] = a.s3[1] = s3;
    a.ridx = ridx;
    a.y[0] = a.y[1] = y;
    a.P = P;
    a.N = N;
    a.G = K / 32;
    a.src_div = src_div;
    k_moe_gemm<false, 4><<<dim3((unsigned)((N + 63) / 64), (unsigned)nE), 64 * W, 0, c->stream>>>(a);
    TI_LAUNCHED("k_moe_gemm");
    return TI_OK;
}

// gate, up [P][I], act = silu(gate) * up, and act quantized: yh, ys
int ti_moe_gateup_launch(ti_ctx* c, const uint16_t* xh, const float* xs, const uint32_t* w1p, const uint16_t* w1s,
                         const uint32_t* w3p, const uint16_t* w3s, const int32_t* ridx, float* gate, float* up, float* act,
                         uint16_t* yh, float* ys, int P, int I, int H, int src_div, int nE) {
    MoeGemm a = {};
    a.xh = reinterpret_cast<const ti_h8*>(xh);
    a.xs = xs;
    a.p3[0] = w1p;
    a.p3[1] = w3p;
    a.s3[0] = w1s;
    a.s3[1] = w3s;
    a.ridx = ridx;
    a.y[0] = gate;
    a.y[1] = up;
    a.act = act;
    a.yh = reinterpret_cast<_Float16*>(yh);
    a.ys = ys;
    a.P = P;
    a.N = I;
    a.G = H / 32;
    a.src_div = src_div;
    k_moe_gemm<true, 4><<<dim3((unsigned)(I / 32), (unsigned)nE), 64 * W, 0, c->stream>>>(a);
    TI_LAUNCHED("k_moe_gemm (gate/up)");
    return TI_OK;
}
