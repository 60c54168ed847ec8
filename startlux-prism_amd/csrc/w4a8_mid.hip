// W4A8 GEMM for batches between the decode kernels (up to 16 rows) and the 128 x 128 tile kernels: Q4_K and Q6_K
// weights in the packed layouts of w4a8.hip, the same arithmetic and bits.
//
// A 128 x 128 tile per workgroup leaves most CUs idle on one projection (13824 x 5120 is 108 tiles, 5120 x 17408 forty),
// and its 128 rows are computed whatever the batch.  Here a workgroup owns TG adjacent 16-row weight tiles and MT 16-row
// activation tiles, and its NW waves take the super-blocks in turn: wave w computes super-block r NW + w of round r, the
// two-plane int8 products of all its TG x MT blocks (the scale planes made once for the MT blocks), and stores the terms
// t to LDS.  After one barrier per round the workgroup's threads add the round's terms, y = fma(a[b, m], t, y), in
// super-block order as every other kernel does: the chain is only K / 256 long, and one round's exchange is 1 KB per
// block and wave against 2.25 or 4.3 KB of weights.  The weights of the next two super-blocks of a wave are in flight
// in registers; an activation piece's registers are requested again for the next super-block once its MFMAs are issued.
#include "w4a8_mid.h"

#include "w4a8_common.h"

namespace prism {

template <bool Q6>
struct MidW {                                          // one tile's super-block as a lane holds it
    v4u w[2];                                          // Q4_K: its bytes of the two halves
    v4u meta;                                          // row lm's 16 meta bytes (Q6_K: its 16 scales)
};
template <>
struct MidW<true> {
    v2u w[4][2];                                       // pair p: inputs 64 p + 16 q .. + 7, .. + 15 of row lm
    v4u meta;
    uint32_t d;
};

// The rounds' term buffers: two (one barrier per round), or one where two would leave room for one workgroup per CU.
constexpr int mid_bufs(int TG, int MT) { return TG * MT >= 8 ? 1 : 2; }
constexpr size_t mid_lds(int NW, int TG, int MT) {
    return (size_t)mid_bufs(TG, MT) * NW * (TG * MT * 256 + MT * 16) * 4 + (size_t)NW * MT * 1024;
}

template <bool Q6, int NW, int TG, int MT, int EPI>
__global__ __launch_bounds__(NW * 64, 2) void w4_mid_kernel(const int8_t* __restrict__ xq, const float* __restrict__ a,
                                                            int64_t a_sb, const int8_t* __restrict__ xs,
                                                            const uint8_t* __restrict__ qv,
                                                            const uint8_t* __restrict__ meta, void* __restrict__ out,
                                                            int64_t ldo, const int32_t* __restrict__ n_rows, int M,
                                                            int N, int K, int gy) {
    constexpr int MR = 16 * MT, TERMS = TG * MR * 16;  // one super-block's terms [tile][m][n]
    constexpr int BUFS = mid_bufs(TG, MT);
    extern __shared__ __attribute__((aligned(16))) float tl[];  // [BUFS][NW][TERMS], a [BUFS][NW][MR], scratch [NW][MT] KB
    float* al = tl + BUFS * NW * TERMS;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 15, q = lane >> 4;
    // the row groups of one tile group run on one XCD next to each other, so its weights come from HBM once
    const int j8 = blockIdx.x >> 3, tg0 = (j8 / gy) * 8 + (blockIdx.x & 7), nt0 = tg0 * TG, m0 = (j8 % gy) * MR;
    const int NB = K / 256, nr = (NB + NW - 1) / NW;
    if (nt0 * 16 >= N) return;
    if (m0 > 0 && m0 >= __ldg(n_rows)) return;         // the first rows' group reads the count only at its end

    constexpr int WB = Q6 ? 4096 : 2048, MB = Q6 ? Q6_META : 256;
    const auto wr = buf_rsrc(qv + (int64_t)nt0 * NB * WB);
    const auto mr = buf_rsrc(meta + (int64_t)nt0 * NB * MB);
    const auto xr = buf_rsrc(xq + (int64_t)m0 * K);
    // activations: four consecutive lanes load a row's 64 bytes of a pair, and the wave turns them in LDS (lds_turn)
    const auto sr = buf_rsrc(Q6 ? (const int8_t*)nullptr : xs + (int64_t)m0 * 16);
    uint32_t xv[MT], xsv[MT];
#pragma unroll
    for (int j = 0; j < MT; j++) {
        xsv[j] = (min(m0 + 16 * j + lm, M - 1) - m0) * 16;
        xv[j] = (uint32_t)(min(m0 + 16 * j + (lane >> 2), M - 1) - m0) * K + 16 * ((lane & 3) ^ lds_turn(lane >> 4));
    }
    int8_t* xw = reinterpret_cast<int8_t*>(al + BUFS * NW * MR) + wv * MT * 1024;
    const int xrd = lm * 64 + 16 * (q ^ lds_turn(lm >> 2));
    const uint32_t wv6 = (32 * (q & 1) + lm) * 16 + 8 * (q >> 1);

    auto load_w = [&](int b, MidW<Q6>* c) {            // past the end: the last super-block again
        b = min(b, NB - 1);
#pragma unroll
        for (int g = 0; g < TG; g++) {
            if constexpr (Q6) {
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    c[g].w[p][0] = buf_load8(wr, wv6, (g * NB + b) * WB + p * 1024);
                    c[g].w[p][1] = buf_load8(wr, wv6 + 256, (g * NB + b) * WB + p * 1024);
                }
                c[g].d = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(mr, lm * 2 + 256, (g * NB + b) * MB, 0);
            } else {
#pragma unroll
                for (int h = 0; h < 2; h++)
                    c[g].w[h] = __builtin_bit_cast(v4u, buf_load16<kBufNT>(wr, lane * 16, (g * NB + b) * WB + h * 1024));
            }
            c[g].meta = __builtin_bit_cast(v4u, buf_load16(mr, lm * 16, (g * NB + b) * MB));
        }
    };
    v4i x[4][MT], s[MT];
    float av;
    auto load_x2 = [&](int b, int p) {
        b = min(b, NB - 1);
#pragma unroll
        for (int j = 0; j < MT; j++) {
            x[p][j] = buf_load16(xr, xv[j], b * 256 + p * 64);
            x[p + 1][j] = buf_load16(xr, xv[j], b * 256 + p * 64 + 64);
        }
    };
    auto load_s = [&](int b) {
        b = min(b, NB - 1);
        if (!Q6) {
#pragma unroll
            for (int j = 0; j < MT; j++) s[j] = buf_load16(sr, xsv[j], b * M * 16);
        }
        av = a[(int64_t)b * a_sb + min(m0 + min(lane, MR - 1), M - 1)];
    };
    auto round = [&](int r, MidW<Q6>* c) {
        const int b = r * NW + wv;
        v4i lo[TG][MT], hi[TG][MT];
#pragma unroll
        for (int g = 0; g < TG; g++)
#pragma unroll
            for (int j = 0; j < MT; j++) lo[g][j] = hi[g][j] = v4i{0, 0, 0, 0};
        uint32_t sp[TG][4];
#pragma unroll
        for (int g = 0; g < TG; g++) {
            if constexpr (Q6) {
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const uint32_t sc = (uint32_t)__builtin_amdgcn_sbfe((int)c[g].meta[p], 8 * q, 8) & 0xffffu;
                    sp[g][p] = sc | (sc << 16);
                }
            } else {
                q4k_lane_splits(c[g].meta, q >> 1, sp[g]);
            }
        }
        // a pair's pieces to LDS and back as MFMA operands: the wave's LDS operations run in order, so the next pair's
        // stores follow this pair's reads with no wait
        v4i xf_[2][MT];
        auto turn = [&](int p) {
#pragma unroll
            for (int j = 0; j < MT; j++) *reinterpret_cast<v4i*>(xw + j * 1024 + lane * 16) = x[p][j];
#pragma unroll
            for (int j = 0; j < MT; j++) xf_[p & 1][j] = *reinterpret_cast<const v4i*>(xw + j * 1024 + xrd);
        };
        turn(0);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            if (p < 3) turn(p + 1);
            if (p == 0 || p == 2) load_x2(b + NW, p);  // both pairs of these rows' 128-byte lines are in LDS
#pragma unroll
            for (int g = 0; g < TG; g++) {
                v4i wl, wh;
                if constexpr (Q6) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        uint32_t l, h;
                        q6_planes(c[g].w[p][i >> 1][i & 1], sp[g][p], l, h);
                        wl[i] = (int)l, wh[i] = (int)h;
                    }
                } else {
                    two_plane(c[g].w[p >> 1][2 * (p & 1)], c[g].w[p >> 1][2 * (p & 1) + 1], sp[g][p], wl, wh);
                }
#pragma unroll
                for (int j = 0; j < MT; j++) {
                    lo[g][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wl, xf_[p & 1][j], lo[g][j], 0, 0, 0);
                    hi[g][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wh, xf_[p & 1][j], hi[g][j], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        float* tb = tl + ((r % BUFS) * NW + wv) * TERMS + lm * 16 + 4 * q;
#pragma unroll
        for (int g = 0; g < TG; g++) {
            // the lane holds row lm's d (and dmin); its outputs are rows 4 q + e
            const float d = f16_to_f32(Q6 ? reinterpret_cast<const uint32_t&>(reinterpret_cast<const MidW<true>&>(c[g]).d)
                                          : c[g].meta[0] & 0xffffu);
            const float dm = Q6 ? 0.f : f16_to_f32(c[g].meta[0] >> 16);
            float de[4], dme[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                de[e] = __shfl(d, 4 * q + e, kWave);
                dme[e] = Q6 ? 0.f : __shfl(dm, 4 * q + e, kWave);
            }
            const int64_t mn8 = !Q6 && q == 0 ? q4k_mins8(c[g].meta) : 0;
#pragma unroll
            for (int j = 0; j < MT; j++) {
                v4f t;
                if constexpr (Q6) {
#pragma unroll
                    for (int e = 0; e < 4; e++) t[e] = mul_rn(de[e], (float)(lo[g][j][e] + 64 * hi[g][j][e]));
                } else {
                    // lanes q > 0 carry zero mins, so their split sums are not masked
                    const v4i mins = mins_mfma(mn8, (int64_t)(uint32_t)s[j][0] | ((int64_t)s[j][1] << 32),
                                               (int64_t)(uint32_t)s[j][2] | ((int64_t)s[j][3] << 32));
#pragma unroll
                    for (int e = 0; e < 4; e++) t[e] = q4k_term(de[e], dme[e], lo[g][j][e] + 8 * hi[g][j][e], mins[e]);
                }
                if (b < NB) *reinterpret_cast<v4f*>(tb + (g * MR + 16 * j) * 16) = t;
            }
        }
        if (lane < MR) al[((r % BUFS) * NW + wv) * MR + lane] = av;
        load_w(b + 2 * NW, c);
        load_s(b + NW);
    };

    // thread -> outputs 4 (tid + i NW 64) .. + 3 of [tile][m][n]
    constexpr int OV = (TERMS / 4 + NW * 64 - 1) / (NW * 64);
    v4f y[OV];
#pragma unroll
    for (int i = 0; i < OV; i++) y[i] = v4f{0.f, 0.f, 0.f, 0.f};
    auto fold = [&](int r) {
        const int nb = min(NW, NB - r * NW);
        const float* tb = tl + (r % BUFS) * NW * TERMS;
        const float* ab = al + (r % BUFS) * NW * MR;
#pragma unroll
        for (int w = 0; w < NW; w++)
            if (w < nb) {
#pragma unroll
                for (int i = 0; i < OV; i++) {
                    const int o = min(tid + i * NW * 64, TERMS / 4 - 1);
                    const v4f t = *reinterpret_cast<const v4f*>(tb + w * TERMS + 4 * o);
                    const float am = ab[w * MR + (o >> 2) % MR];
#pragma unroll
                    for (int e = 0; e < 4; e++) y[i][e] = fmaf(am, t[e], y[i][e]);
                }
            }
    };
    MidW<Q6> c0[TG], c1[TG];
    load_w(wv, c0);
    load_x2(wv, 0);
    load_x2(wv, 2);
    load_s(wv);
    load_w(wv + NW, c1);
    for (int r = 0; r < nr; r += 2) {
        round(r, c0);
        lds_barrier();
        fold(r);
        if (BUFS == 1) lds_barrier();
        if (r + 1 < nr) {
            round(r + 1, c1);
            lds_barrier();
            fold(r + 1);
            if (BUFS == 1) lds_barrier();
        }
    }
    const int live = min(M, __ldg(n_rows));
#pragma unroll
    for (int i = 0; i < OV; i++) {
        const int o = tid + i * NW * 64;
        const int m = m0 + (o >> 2) % MR, n = 16 * (nt0 + (o >> 2) / MR) + 4 * (o & 3);
        if (o >= TERMS / 4 || m >= live || n >= N) continue;
        if (EPI == 0) {
            const uint32_t lo = f32_to_bf16(y[i][0]) | (f32_to_bf16(y[i][1]) << 16);
            const uint32_t hi = f32_to_bf16(y[i][2]) | (f32_to_bf16(y[i][3]) << 16);
            uint16_t* op = reinterpret_cast<uint16_t*>(out) + (int64_t)m * ldo + n;
            if ((((uintptr_t)op) & 7) == 0) {
                *reinterpret_cast<v2u*>(op) = v2u{lo, hi};
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) op[e] = (uint16_t)f32_to_bf16(y[i][e]);
            }
        } else {
            float* op = reinterpret_cast<float*>(out) + (int64_t)m * ldo + n;
#pragma unroll
            for (int e = 0; e < 4; e++) op[e] = add_rn(op[e], y[i][e]);
        }
    }
}

template <bool Q6, int NW, int TG, int MT, int EPI>
static void mid_go(const int8_t* xq, const float* a, int64_t a_sb, const int8_t* xs, const uint8_t* qv,
                   const uint8_t* meta, void* out, int64_t ldo, const int32_t* n_rows, int M, int N, int K, int gy,
                   hipStream_t st) {
    constexpr size_t lds = mid_lds(NW, TG, MT);
    const int groups = (N / 16 + TG - 1) / TG;
    allow_lds(w4_mid_kernel<Q6, NW, TG, MT, EPI>, lds);
    hipLaunchKernelGGL((w4_mid_kernel<Q6, NW, TG, MT, EPI>), dim3((groups + 7) / 8 * 8 * gy), dim3(NW * 64), lds, st, xq, a,
                       a_sb, xs, qv, meta, out, ldo, n_rows, M, N, K, gy);
}

#define MID_ARGS xq, a, a_sb, xs, qv, meta, out, ldo, n_rows, M, N, K, gy, st
template <bool Q6, int NW, int TG>
static void mid_mt(int mt, int epi, const int8_t* xq, const float* a, int64_t a_sb, const int8_t* xs,
                   const uint8_t* qv, const uint8_t* meta, void* out, int64_t ldo, const int32_t* n_rows, int M, int N,
                   int K, int gy, hipStream_t st) {
    // (two tiles, four row tiles: the Q4_K form of four waves only; the others would take the rows in more groups)
    constexpr int M4 = TG == 2 && (Q6 || NW == 8) ? 3 : 4;
    if (mt > M4) gy = ((M + 15) / 16 + M4 - 1) / M4;
    if (mt <= 2) epi == 0 ? mid_go<Q6, NW, TG, 2, 0>(MID_ARGS) : mid_go<Q6, NW, TG, 2, 1>(MID_ARGS);
    else if (mt == 3) epi == 0 ? mid_go<Q6, NW, TG, 3, 0>(MID_ARGS) : mid_go<Q6, NW, TG, 3, 1>(MID_ARGS);
    else epi == 0 ? mid_go<Q6, NW, TG, M4, 0>(MID_ARGS) : mid_go<Q6, NW, TG, M4, 1>(MID_ARGS);
}

void w4_mid_launch(const int8_t* xq, const float* a, int64_t a_sb, const int8_t* xs, const uint8_t* qv,
                   const uint8_t* meta, void* out, int64_t ldo, const int32_t* n_rows, int M, int N, int K, int epi,
                   hipStream_t st) {
    const int gy = (M + 63) / 64, mt = ((M + 15) / 16 + gy - 1) / gy;
    // Measured at 37 rows of Q4_K, us, with NW x TG = 4 x 1 / 4 x 2 / 8 x 2: 13824 x 5120 26 / 22 / 27; 5120 x 17408 36 / 38
    // / 31; two tiles share each activation piece where the grid still fills the chip, and eight waves where it would not.
    // At four row tiles per workgroup (49-64 rows) two tiles fit the registers on Q4_K only, and pay on wide projections:
    // 64 x 13824 x 5120 30 against 33; 100 x 5120 x 17408 77 against 67.
    const bool wide = N > 8192;
    if (xs) {
        if (N % 32 || (mt == 4 && !wide)) mid_mt<false, 4, 1>(mt, epi, MID_ARGS);
        else if (wide) mid_mt<false, 4, 2>(mt, epi, MID_ARGS);
        else mid_mt<false, 8, 2>(mt, epi, MID_ARGS);
    } else {
        if (N % 32 || mt == 4 || !wide) mid_mt<true, 4, 1>(mt, epi, MID_ARGS);
        else mid_mt<true, 4, 2>(mt, epi, MID_ARGS);
    }
}
#undef MID_ARGS

// Measured at K = 5120 (both sides go with K): the mid kernel takes about 3 us and 8.7 ns (Q4_K) or 10 ns (Q6_K) per 16 x 16
// outputs, the tile kernel 45 us for each round of one 128 x 128 tile per CU, whatever the rows in it: 64 x 13824 30
// against 45 us, 100 x 13824 51 against 47, 128 x 5120 25 against 44.
bool w4_mid_faster(bool q6k, int64_t M, int64_t N, int64_t K) {
    if (!w4_mid_fits(M, K)) return false;
    const int64_t blocks = (M + 15) / 16 * (N / 16), tiles = (M + 127) / 128 * ((N + 127) / 128);
    return 30000 + (q6k ? 100 : 87) * blocks < (tiles + 255) / 256 * 450000;
}

}  // namespace prism
