// k_tern_gemm.hip — ternary (Q2_0_g64) GEMM of several activation rows on the matrix cores
// (gemm_tern_b4, cpu/kernel/src/lib.rs:331-367, and the per-token gemv_tern of a prompt,
// native/crates/n2-kernels/src/tern.rs:79-119).
//
// out[t][n] = sum_b s[n,b] * (dot_b(t, n) - xsum[t,b]): one v_mfma_i32_16x16x64_i8 forms the
// exact int32 dots of one 64-code block for 16 tokens x 16 rows, with -xsum as its C operand,
// and each result is scaled into an f32 sum with one fma. The scalar kernel keeps sum s*dot
// and sum s*xsum apart and subtracts them at the end, which cancels two sums some 100 times
// the result; this form has no such cancellation and one rounding a block instead of four.
//
// Operands: lane l feeds row/column l%16 and the 16 K slots of group j = l/16: plane j of the
// block, codes 16j..16j+15 (the weights' 16 bytes shifted by 2j and masked) against the
// activations' 16 bytes at 16j. In that layout neighbouring lanes are in different rows, and a
// version that loaded its operands so from memory was bound by the scattered loads (14 us at
// 2048 x 6144 x 50, 40 at 8192 x 6144 x 128; this one 6.4 and 26.7). So each wave loads whole 64- and
// 256-byte runs, parks them in its own part of LDS and reads the operands from there; LDS
// serves a wave in order, so there is no barrier in the loop.
#include "ti_internal.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr uint32_t M2 = 0x03030303u;
struct GemmMats {
    const ti_v4u* codes[3];
    const float* scales[3];
    float* out[3];
    long stride[3];
    int N[3];
    int blk0[3];                   // first workgroup (grid x) of each matrix
    int nmat;
};

// One wave's part of LDS: a step is four blocks (256 codes) of 16 NT rows and 16 MT tokens.
template <int NT, int MT>
struct WaveBuf {
    ti_v4u act[16 * MT][17];        // 256 bytes a token; the 17th piece spreads the rows over the banks
    ti_v4u codes[16 * NT][5];       // 64 bytes a row, padded likewise
    v4f scale[16 * NT];
    v4i xsum[4][4 * MT];          // [block][token / 4]: -xsum
};

// Workgroup: a tile of 16 NT rows by 16 MT tokens (grid x: rows of the matrices in turn, y:
// tokens); its 4 waves take every fourth step and their sums meet in LDS. A wave holds two steps' registers, but
// the compiler sinks the odd step's loads behind the test for the last step, to where they are used. Issued where
// they are written (the odd step unconditional, issue fences) both steps are in flight and nothing is gained: 2048 x
// 6144 x 50 6.4 us either way, 8192 x 6144 x 128 26.7 against 26.9.
template <int NT, int MT>
__global__ __launch_bounds__(256, 2) void k_tern_gemm(GemmMats m, const int8_t* __restrict__ act,
                                                      const int32_t* __restrict__ xsum, int K, int B) {
    __shared__ WaveBuf<NT, MT> s_wave[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, j = lane >> 4;
    const int nb = K / 64;
    const int b = blockIdx.x;
    const int mi = (m.nmat > 1 && b >= m.blk0[1]) + (m.nmat > 2 && b >= m.blk0[2]);
    const ti_v4u* codes = mi == 0 ? m.codes[0] : (mi == 1 ? m.codes[1] : m.codes[2]);
    const float* scales = mi == 0 ? m.scales[0] : (mi == 1 ? m.scales[1] : m.scales[2]);
    float* out = mi == 0 ? m.out[0] : (mi == 1 ? m.out[1] : m.out[2]);
    const long stride = mi == 0 ? m.stride[0] : (mi == 1 ? m.stride[1] : m.stride[2]);
    const int N = mi == 0 ? m.N[0] : (mi == 1 ? m.N[1] : m.N[2]);
    const int row0 = (b - (mi == 0 ? 0 : (mi == 1 ? m.blk0[1] : m.blk0[2]))) * 16 * NT;
    const int t0 = blockIdx.y * 16 * MT;
    WaveBuf<NT, MT>& L = s_wave[wave];

    // loads: 4 lanes a row and step for codes, scales and xsum; 16 lanes a token for activations
    const int l4 = lane >> 2, p4 = lane & 3;
    const ti_v4u* crow[NT];
    const float* srow[NT];
    const int32_t* xrow[MT];
    const ti_v4u* arow[4 * MT];
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const size_t row = min(row0 + 16 * n + l4, N - 1);
        crow[n] = codes + row * nb;
        srow[n] = scales + row * nb;
    }
#pragma unroll
    for (int t = 0; t < MT; t++) xrow[t] = xsum + (size_t)min(t0 + 16 * t + l4, B - 1) * nb;
#pragma unroll
    for (int q = 0; q < 4 * MT; q++) arow[q] = reinterpret_cast<const ti_v4u*>(act + (size_t)min(t0 + 4 * q + j, B - 1) * K);

    struct Step {
        ti_v4u cw[NT], av[4 * MT];
        float sc[NT];
        int xs[MT];
    };
    const int ns = (nb + 3) / 4;
    auto load = [&](Step& s, int st) {             // past the last block: it again, scaled by 0
        const int b0 = 4 * min(st, ns - 1);
        const int blk = min(b0 + p4, nb - 1), piece = 4 * min(b0 + (r >> 2), nb - 1) + (r & 3);
#pragma unroll
        for (int q = 0; q < 4 * MT; q++) s.av[q] = arow[q][piece];
#pragma unroll
        for (int n = 0; n < NT; n++) {
            s.cw[n] = crow[n][blk];
            s.sc[n] = srow[n][blk];
        }
#pragma unroll
        for (int t = 0; t < MT; t++) s.xs[t] = xrow[t][blk];
    };
    float acc[NT][MT][4] = {};
    auto step = [&](const Step& s, int st) {
        ti_wave_lds_fence();                       // the last step's reads are done
#pragma unroll
        for (int q = 0; q < 4 * MT; q++) L.act[4 * q + j][r] = s.av[q];
#pragma unroll
        for (int n = 0; n < NT; n++) {
            L.codes[16 * n + l4][p4] = s.cw[n];
            reinterpret_cast<float*>(L.scale)[64 * n + lane] = 4 * st + p4 < nb ? s.sc[n] : 0.0f;
        }
#pragma unroll
        for (int t = 0; t < MT; t++) reinterpret_cast<int*>(L.xsum)[p4 * 16 * MT + 16 * t + l4] = -s.xs[t];
        ti_wave_lds_fence();
        v4f sc[NT];
#pragma unroll
        for (int n = 0; n < NT; n++) sc[n] = L.scale[16 * n + r];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            v4i A[MT], C[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) {
                A[t] = __builtin_bit_cast(v4i, L.act[16 * t + r][4 * u + j]);
                C[t] = L.xsum[u][4 * t + j];
            }
#pragma unroll
            for (int n = 0; n < NT; n++) {
                const ti_v4u w = (L.codes[16 * n + r][u] >> (uint32_t)(2 * j)) & M2;
                const v4i Bv = __builtin_bit_cast(v4i, w);
                const float s4 = sc[n][u];
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    const v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[t], Bv, C[t], 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[n][t][i] = fmaf(s4, (float)d[i], acc[n][t][i]);
                }
            }
        }
    };
    Step s0, s1;
    load(s0, wave);
    load(s1, wave + 4);
    for (int st = wave; st < ns; st += 8) {
        step(s0, st);
        load(s0, st + 8);
        if (st + 4 >= ns) break;
        step(s1, st + 4);
        load(s1, st + 12);
    }
    constexpr int PR = 16 * NT + 1, PW = 16 * MT * PR;   // [wave][16 MT tokens][16 NT rows + 1]
    static_assert(4 * PW * 4 <= (int)sizeof(s_wave), "the sums fit the waves' buffers");
    float* part = reinterpret_cast<float*>(s_wave);
    __syncthreads();                                   // every wave has read its last step
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) part[wave * PW + (16 * t + 4 * j + i) * PR + 16 * n + r] = acc[n][t][i];
    __syncthreads();
#pragma unroll
    for (int e = tid; e < 256 * NT * MT; e += 256) {
        const int n = e % (16 * NT), t = e / (16 * NT);
        const float* p = part + t * PR + n;
        if (row0 + n < N && t0 + t < B) out[(size_t)(t0 + t) * stride + row0 + n] = (p[0] + p[PW]) + (p[2 * PW] + p[3 * PW]);
    }
}

template <int NT, int MT>
void launch(ti_ctx* c, GemmMats& m, const int8_t* act, const int32_t* xsum, int K, int B) {
    long blocks = 0;
    for (int i = 0; i < 3; i++) {
        m.blk0[i] = (int)blocks;
        if (i < m.nmat) blocks += ((long)m.N[i] + 16 * NT - 1) / (16 * NT);
    }
    const dim3 grid((unsigned)blocks, (unsigned)((B + 16 * MT - 1) / (16 * MT)));
    k_tern_gemm<NT, MT><<<grid, 256, 0, c->stream>>>(m, act, xsum, K, B);
}

}  // namespace

bool ti_tern_gemm_mfma_ok(int N, int K, int B) {
    return K % 64 == 0 && B <= 16 * 65535 && N <= (1 << 30);
}

// rows t of outs[i] start at outs[i] + t * strides[i]; act [B][K] (16-byte aligned), xsum [B][K/64]
int ti_tern_gemm_mfma(ti_ctx* c, const int8_t* act, const int32_t* xsum, int K, int B, int nmat, const uint8_t* const* codes,
                      const float* const* scales, float* const* outs, const long* strides, const int* Ns) {
    GemmMats m = {};
    long tiles = 0;
    for (int i = 0; i < 3; i++) {
        const int s = i < nmat ? i : nmat - 1;
        TI_REQUIRE(ti_tern_gemm_mfma_ok(Ns[s], K, B), "ternary GEMM: N=%d K=%d B=%d", Ns[s], K, B);
        m.codes[i] = reinterpret_cast<const ti_v4u*>(codes[s]);
        m.scales[i] = scales[s];
        m.out[i] = outs[s];
        m.stride[i] = strides[s];
        m.N[i] = Ns[s];
        if (i < nmat) tiles += (long)((Ns[s] + 15) / 16) * ((B + 15) / 16);
    }
    m.nmat = nmat;
    // Few tiles: one 16 x 16 tile a workgroup (its four waves split K), so that more CUs have
    // one; many: larger tiles, whose operands are read from LDS once for several products. us at
    // 16 x 16, 32 x 16, 32 x 32 (rows x tokens; 256 CUs): 2048 x 6144 x 50 (512 tiles) 7.5 / 7.5 / 10.9;
    // 8192 x 2048 x 48 (1536) 7.4 / 6.5 / 7.1; 8192 x 6144 x 128 (4096) 36.6 / 27.2 / 26.5. The lines: four
    // workgroups of the smallest tile a CU, and six of the next.
    if (tiles < 4L * c->cus) launch<1, 1>(c, m, act, xsum, K, B);
    else if (tiles < 12L * c->cus) launch<2, 1>(c, m, act, xsum, K, B);
    else launch<2, 2>(c, m, act, xsum, K, B);
    TI_LAUNCHED("k_tern_gemm");
    return TI_OK;
}
