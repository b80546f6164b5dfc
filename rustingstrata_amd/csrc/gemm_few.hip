// GEMM on int8 MFMA for few positions (gemm_dense of a short prompt or a batch of decoding sequences; the expert tiles
// of a short prompt): the same products and the same bits as gemm_kernel (gemm.hip).
//
// With a few dozen positions a 128-row block of gemm_kernel leaves most CUs without an item and runs a row's
// super-blocks one after the other (24 positions of 5120 x 2048 Q6_K: 40 blocks, 8 steps, 29 us for 9 MB). Here a
// wave's unit is one super-block of 16 weight rows against up to 16 positions:
//   * KSP: a block's 8 waves split an item's super-blocks (pair mode: 4 waves the gate rows, 4 the up rows), leave the
//     super-blocks' float terms in LDS and add them in super-block order, as the CPU does, so a row's super-blocks run
//     side by side and the sum keeps its bits;
//   * otherwise (rows of few super-blocks, many items) every wave walks its own item's super-blocks with the sum in
//     registers, and no wave waits for another.
// (16 positions a unit: 32 or 64, with the weights decoded once for them, measure slower, 5120 x 2048 Q6_K: 24 positions
// 13.4 against 10.1 us, 64 positions 17.8 against 14.7. At 16 the block form of Q6_K spills 3 registers, the others none; a
// spill's loads and stores can only make wait_vm<NXL> wait for more than the raw rows, which are older than they are.)
// X fragments come straight from global memory (the whole X is a few KB to a few hundred: L2), raw weight rows through
// a wave's own LDS region, reloaded for its next unit as soon as the current one is decoded. Two blocks fit a CU.
#include <algorithm>

#include "dsa.h"
#include "gemm_dev.h"
#include "../../include/strata_hip.h"

namespace strata {

typedef int v2i __attribute__((ext_vector_type(2)));

namespace {
constexpr int FW = 8;    // waves per block
constexpr int FTS = 8;   // super-blocks whose terms the LDS holds at once
constexpr int FPM = 16;  // positions of a unit
constexpr int FPP = FPM + 4;  // floats of a term row (16-byte pad: rows start in spread banks)

// Where this form is taken, by what both sides measured (us, gemm_kernel or gemm_small_kernel -> this one).
// Dense, by items (16 rows x 16 positions; gemm_kernel needs a 128-row block's whole super-block chain whatever the
// items): Q6_K 5120 x 2048: 5 positions 28.4 -> 7.2, 24 29.6 -> 9.9, 64 (1280 items) 32.1 -> 15.0, 256 (5120) 32.4 ->
// 36.7; Q4_K 5120 x 2048: 64 27.8 -> 15.7, 100 (2240) 27.8 -> 23.9, 200 28.4 -> 42.7; 2048 x 2048, 256 positions
// (2048): Q6_K 31.8 -> 16.2, Q4_K 27.8 -> 20.5. One unit of positions, whatever the rows: 151936 x 2048, 16 positions
// (9496): Q6_K 128 -> 69, Q4_K 95 -> 92, Q2_K 82 -> 54 (32 positions: 134 -> 128, 103 -> 179, 87 -> 103). A block an item up
// to 1280 items: 64 positions of 5120 x 2048 15.0 against 16.1 a wave an item (Q4_K 15.7 / 20.1), 256 of 2048 x 2048 22.2 /
// 16.2 (23.2 / 20.5).
constexpr long long FEW_DENSE_BLOCK_ITEMS = 1280, FEW_DENSE_ITEMS = 2048;
long long few_dense_items(int rows, int n) { return (long long)((rows + 15) / 16) * ((n + FPM - 1) / FPM); }
// Tile lists with SMALL_TILES, gemm_small_kernel -> this form.
// Gate/up, by the tokens gathered from (128 experts, top 8, 2048 x 768; us at 27 / 100 / 200 tokens): Q3_K 81 -> 65 / 120 ->
// 110 / 122 -> 138, IQ2_XXS 69 -> 57 / 103 -> 95 / 105 -> 119, Q2_K 48 -> 42 / 67 -> 67 / 69 -> 92 (48: 57 -> 55, 64: 58 ->
// 62); the scale-after types, whose close is heavier per tile, only up to 32 tokens: Q5_K 64 -> 53 / 94 -> 103, Q4_K 59 ->
// 51 / 86 -> 94, IQ4_XS 72 -> 54 / 102 -> 98 (64 tokens: 82 -> 87). This form's time over the other's, for even and
// Zipf-skewed loads, with 128 experts top 8 / 64 top 6 / 32 top 4 (1024 columns) / 8 top 2: Q3_K 100 tokens 0.92 1.02 / 0.92
// 1.17 / 0.99 0.95 / 0.66 0.73, 128 tokens 0.92 1.19 / 1.03 1.24 / 0.98 0.88 / 0.77 0.91 (IQ2_XXS alike); Q6_K 64 tokens 0.79
// 0.81 / 0.76 0.84 / 0.78 0.90 / 0.71 0.67, 100 tokens 0.79 0.88 / 0.77 0.95 / 1.08 1.05 / 0.72 0.79, 128 tokens 0.81 0.98 /
// 0.87 1.00 / 1.09 0.91 / 0.84 0.99; 32 tokens, the others, at most 0.96.
// Down, by the rows of X (128 experts; 216 / 512 / 800): Q3_K 43 -> 37 / 52 -> 51 / 57 -> 61, IQ2_XXS 46 -> 38 / 58 -> 54 /
// 63 -> 64, Q2_K 27 -> 24 / 32 -> 35 / 35 -> 44 (384: 31 -> 31), Q6_K 50 -> 35 / - / 72 -> 61 (1600: 72 -> 62); IQ4_XS 40 ->
// 37 (320: 47 -> 42, 512: 50 -> 54), IQ3_S 47 -> 39; Q4_K 128: 25 -> 23, 216: 33 -> 37, Q5_K 27 -> 24, 36 -> 38.
// And by the rows a tile slot, because every 16 positions of a tile decode its weights again: over the other form's time, even
// and skewed, at 3 rows an expert (128 experts / 64): Q4_K 0.87 1.03 / 0.90 1.09, IQ4_XS 0.71 0.89 / 0.74 0.93, at 4 and 4.5
// IQ4_XS 0.74 1.10 / 0.77 1.17, IQ3_S 0.67 0.99 / 0.69 1.03, Q2_K 0.75 1.17 / 0.70 1.07, at 6 Q2_K 0.79 1.15 / 0.79 1.30, Q3_K
// 0.77 0.98 / 0.75 1.10, Q6_K at 8 and 12 0.64 0.84 / 0.89 0.98. With less than an item a wave, where a tile's chunks run
// side by side: 32 experts of 1024 x 512 at 6 / 8 / 12.5 rows an expert Q6_K 0.60 0.76 / 0.60 0.79 / 0.82 1.29, Q4_K 0.80 0.72
// / 0.82 0.99 / 1.03 1.73 (one after the other, 0.57 1.15 and 0.77 1.40 at 6); 8 experts of 2048 x 1024 at 12 / 16: Q6_K
// 0.59 0.59 / 0.59 0.81, Q4_K 0.89 0.90 / 0.89 1.01, IQ4_XS 0.86 0.86 / 0.87 1.05.
int few_gathered(int ty, int cols) {
    switch (ty) {
    case Q6_K: return cols < 1536 ? 64 : 128;
    case Q3_K: case IQ2_XXS: return 100;
    case Q2_K: return 48;
    default: return 32;
    }
}
// Most rows of X, and most quarter rows a tile slot where every wave has an item.
struct FewRows {
    int rows, slot4;
};
FewRows few_rows(int ty) {
    switch (ty) {
    case Q6_K: return {1024, 48};
    case Q3_K: case IQ2_XXS: return {512, 26};
    case Q2_K: return {384, 18};
    case IQ3_S: return {320, 16};
    case IQ4_XS: return {320, 12};
    default: return {128, 10};
    }
}
constexpr int FEW_WAVES = 256 * 2 * FW;  // waves resident at once
}  // namespace

template <int T> struct FewFmt : GemmPlanes<T> {
    static constexpr int WI = (16 * GemmPlanes<T>::NCH + 63) / 64;  // weight load instructions per unit
    static constexpr int WREG = 64 * WI * 16;                        // LDS bytes of a wave's raw rows
};
template <int T> static constexpr size_t few_smem(bool ksp, bool pair) {
    size_t b = (size_t)FW * FewFmt<T>::WREG;
    if (ksp) b += (size_t)(pair ? 2 : 1) * FTS * 16 * FPP * 4;
    if (T == IQ2_XXS || T == IQ3_S) b += sizeof(IqTables);
    return b;
}

template <int T, bool KSP>
__global__ __launch_bounds__(64 * FW, 4) void gemm_few_kernel(GemmArgs a) {
    using F = FewFmt<T>;
    constexpr int NP = F::NP, SBB = sb_bytes(T), NCH = F::NCH, RAWP = F::RAWP, WI = F::WI, WREG = F::WREG;
    constexpr int P_HI = 0, P_LO = F::HI ? 1 : 0, P_M = F::HI ? 2 : 1;
    constexpr bool IQ = T == IQ2_XXS || T == IQ3_S, SA = Dsa<T>::ON;
    constexpr int NXL = (SA ? 8 : 4) + 1;  // X and scale loads of a unit
    extern __shared__ __align__(16) uint8_t smem[];
    // LDS: [raw rows: FW x WREG][IqTables][terms: (pair: 2 x) FTS x 16 x FPP floats]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    uint8_t* raw = smem + wave * WREG;
    IqTables* tab = (IqTables*)(smem + FW * WREG);
    float* terms = (float*)(smem + FW * WREG + (IQ ? sizeof(IqTables) : 0));
    const int cols = a.cols, nsb = cols / 256, l16 = lane & 15, kl = lane >> 4;
    const int ntiles = a.tiles ? (a.n_tiles_dev ? min(sload(a.n_tiles_dev), a.max_tiles) : a.max_tiles) : a.max_tiles;
    const bool pair = KSP && a.pair != 0;
    // an item is a tile's 16 rows and every (1 << cs)-th of its chunks of 16 positions, the first chunks' items first
    const int nrb = (a.rows + 15) / 16, nit = nrb * ntiles, cs = KSP ? 0 : a.few_cs, total = nit << cs;
    // this wave's super-blocks s0, s0 + KS, .. of an item, of the second matrix (pair) for waves 4..7
    const int mat = pair ? wave >> 2 : 0, KS = !KSP ? 1 : pair ? 4 : 8, s0 = !KSP ? 0 : pair ? wave & 3 : wave;
    const uint64_t w2 = mat ? (uint64_t)a.w2 : 0;
    const int ibeg = KSP ? blockIdx.x : blockIdx.x * FW + wave, istep = KSP ? gridDim.x : gridDim.x * FW;

    struct Item {
        uint64_t w;
        int m0, cnt, n0, rest;  // cnt 0: no item; rest > 0: the item has a chunk after this one
    };
    auto item_at = [&](int id, int pc) __attribute__((always_inline)) {
        Item it;
        int c = pc << cs;
        if (cs) {  // (at most 4 chunks side by side)
            const int q = (id >= nit) + (id >= 2 * nit) + (id >= 3 * nit);
            c += q;
            id -= q * nit;
        }
        const int tile = id / nrb;
        it.n0 = 16 * (id - tile * nrb);
        int cnt;
        if (a.tiles) {
            const uint64_t t0 = sload(a.tiles + 2 * tile), t1 = sload(a.tiles + 2 * tile + 1);
            it.w = t0;
            it.m0 = (int)(uint32_t)t1 + FPM * c;
            cnt = min(256, (int)(t1 >> 32)) - FPM * c;
        } else {
            it.w = (uint64_t)a.dense_w;
            it.m0 = FPM * tile;
            cnt = min(FPM, a.dense_n - it.m0);
        }
        it.cnt = max(0, min(FPM, cnt));
        it.rest = cnt - (FPM << cs);
        return it;
    };
    // the next chunk with positions: the next of the same item, else the first of the next item that has any
    auto next_item = [&](int& id, int& pc, const Item& prev) __attribute__((always_inline)) {
        if (prev.rest > 0) return item_at(id, ++pc);
        Item it{0, 0, 0, 0, 0};
        pc = 0;
        for (id += istep; id < total; id += istep) {
            it = item_at(id, 0);
            if (it.cnt > 0) break;
        }
        return it;
    };
    if constexpr (IQ) {
        load_iq_tables(tab);
        __syncthreads();
    }

    // raw rows of super-block s of an item: chunk c = 64 i + lane is chunk c % NCH of row c / NCH (the 16-byte cover of
    // the row's super-block; rows past the matrix read its last row)
    auto load_w = [&](const Item& it, int s) __attribute__((always_inline)) {
        const uint64_t beg = it.w + w2 + (uint64_t)s * SBB, base = beg & ~(uint64_t)15;
        const uint32_t b15 = (uint32_t)(beg & 15);
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int c = 64 * i + lane, r = c / NCH;
            const uint32_t t = b15 + __umul24((uint32_t)min(it.n0 + r, a.rows - 1), (uint32_t)a.rb);
            const uint32_t o = (t & ~15u) + 16 * (uint32_t)(c - r * NCH);
            if (r < 16 && o < t + SBB) load_lds16_so(base, o, raw + 16 * 64 * i);
        }
    };
    // the X row of this lane's position l16 of an item (positions past cnt: its first one)
    auto row_of = [&](const Item& it) __attribute__((always_inline)) {
        const int m = it.m0 + (l16 < it.cnt ? l16 : 0);
        return it.cnt == 0 ? 0 : a.xrow ? a.xrow[m] : m;
    };

    int id = ibeg - istep, pc = 0;
    Item cur = next_item(id, pc, Item{0, 0, 0, 0, 0});
    if (cur.cnt == 0) return;  // (KSP: the whole block)
    int xr = row_of(cur);
    if (s0 < nsb) load_w(cur, s0);
    Item nxt = next_item(id, pc, cur);

    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    // KSP: threads 0..255 add up output (row, position) of the first matrix, 256..511 (pair) of the second
    const int orow = tid & 15, opos = (tid >> 4) & 15;
    const bool adds = tid < (pair ? 512 : 256);
    float sum = 0.0f;

    // y[m, n0 + row] (op) v
    auto put = [&](float* yp, float v) __attribute__((always_inline)) {
        if (a.act == STRATA_ACT_STORE) *yp = v;
        else if (a.act == STRATA_ACT_SWIGLU) *yp = silu_dev(*yp) * v;
        else *yp += v;
    };

    while (true) {
        const int xrn = row_of(nxt);
        for (int sb = 0; sb < nsb; sb += KSP ? FTS : nsb) {
            const int se = KSP ? min(sb + FTS, nsb) : nsb;  // the super-blocks of this round
            for (int s = sb + s0; s < se; s += KS) {
                // X fragments and scale of the unit
                v4i xf[4];
                const uint64_t xb = (uint64_t)a.xq + (uint32_t)xr * (uint32_t)cols + 256u * (uint32_t)s;
                if constexpr (SA) {
#pragma unroll
                    for (int g = 0; g < 8; g++) {
                        const v2i v = *gptr<v2i>(xb + 32 * g + 8 * kl);
                        xf[g >> 1][2 * (g & 1)] = v[0];
                        xf[g >> 1][2 * (g & 1) + 1] = v[1];
                    }
                } else {
#pragma unroll
                    for (int kk = 0; kk < 4; kk++) xf[kk] = *gptr<v4i>(xb + 64 * kk + 16 * kl);
                }
                const float dxv = *gptr<float>((uint64_t)(a.xd + (uint32_t)xr * (uint32_t)(cols / 32) + 8 * s));
                // the unit's raw rows (older than its X loads, none of which may move past this wait)
                asm volatile("" : : : "memory");
                __builtin_amdgcn_sched_barrier(0);
                wait_vm<NXL>();
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("" : : : "memory");
                const uint64_t ra = cur.w + w2;
                const uint8_t* b = raw + l16 * RAWP +
                                   (((uint32_t)(ra & 15) + __umul24((uint32_t)min(cur.n0 + l16, a.rows - 1), (uint32_t)a.rb) +
                                     (uint32_t)s * SBB) & 15);
                v4i B[4][NP];
                uint32_t Bq[8][2], Bm[8];
                int scg[8];
                float D, M;
                if constexpr (SA) {
                    using DS = Dsa<T>;
                    const auto r = DS::row(b, kl);
#pragma unroll
                    for (int g = 0; g < 8; g++) {
                        int m;
                        DS::run(b, r, g, kl, tab, Bq[g], scg[g], m);
                        if constexpr (DS::MIN) Bm[g] = (uint32_t)m * 0x01010101u;
                        if (g % 2 == 1) __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
#pragma unroll
                    for (int kk = 0; kk < 4; kk++) {
                        uint32_t hi[4], lo[4];
                        int m;
                        Dec<T>::run(b, 4 * kk + kl, tab, hi, lo, m);
                        if constexpr (F::HI) B[kk][P_HI] = (v4i){(int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
                        B[kk][P_LO] = (v4i){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3]};
                        if constexpr (F::MIN) {
                            const int mw = (int)((uint32_t)m * 0x01010101u);
                            B[kk][P_M] = (v4i){mw, mw, mw, mw};
                        }
                        __builtin_amdgcn_sched_barrier(0);  // a K step at a time: registers
                    }
                }
                Dec<T>::scales(b, D, M);
                // the raw rows are decoded and X is here: the raw region takes the next unit's rows, which fly while
                // this unit's products and sums run
                wait_lds();
                wait_vm<0>();
                asm volatile("" : : : "memory");
                if (s + KS < nsb) load_w(cur, s + KS);
                else if (nxt.cnt && s0 < nsb) load_w(nxt, s0);
                v4i c[NP], mn = (v4i){0, 0, 0, 0};
                int iv[4] = {0, 0, 0, 0};
                if constexpr (SA) {
#pragma unroll
                    for (int h = 0; h < 8; h += 4) {  // four groups at a time: registers
                        v4i d[4];
#pragma unroll
                        for (int g = h; g < h + 4; g++) {
                            const long af = (long)(((uint64_t)(uint32_t)xf[g >> 1][2 * (g & 1) + 1] << 32) |
                                                   (uint32_t)xf[g >> 1][2 * (g & 1)]);
                            const long bq = (long)(((uint64_t)Bq[g][1] << 32) | Bq[g][0]);
                            d[g - h] = __builtin_amdgcn_mfma_i32_16x16x32_i8(af, bq, (v4i){0, 0, 0, 0}, 0, 0, 0);
                            if constexpr (F::MIN) {
                                const long bm = (long)(((uint64_t)Bm[g] << 32) | Bm[g]);
                                mn = __builtin_amdgcn_mfma_i32_16x16x32_i8(af, bm, mn, 0, 0, 0);
                            }
                        }
#pragma unroll
                        for (int g = h; g < h + 4; g++)
#pragma unroll
                            for (int q = 0; q < 4; q++) iv[q] += __mul24(scg[g], d[g - h][q]);
                    }
                } else {
#pragma unroll
                    for (int kk = 0; kk < 4; kk++)
#pragma unroll
                        for (int pl = 0; pl < NP; pl++)
                            c[pl] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xf[kk], B[kk][pl],
                                                                          kk ? c[pl] : (v4i){0, 0, 0, 0}, 0, 0, 0);
                    if constexpr (F::MIN) mn = c[P_M];
#pragma unroll
                    for (int q = 0; q < 4; q++) iv[q] = F::HI ? (c[P_HI][q] << 8) + c[P_LO][q] : c[P_LO][q];
                }
                // the reference's float steps, rounded one by one (src/cpu_moe.rs:327-377): sum += (D dx) s - (M dx) m
                float f[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float dq = __shfl(dxv, 4 * kl + q, 64);
                    f[q] = (D * dq) * (float)iv[q];
                    if constexpr (F::MIN) f[q] = f[q] - (M * dq) * (float)mn[q];
                }
                if constexpr (KSP) {
                    *(float4*)&terms[((mat * FTS + s - sb) * 16 + l16) * FPP + 4 * kl] = make_float4(f[0], f[1], f[2], f[3]);
                } else {
#pragma unroll
                    for (int q = 0; q < 4; q++) acc[q] = acc[q] + f[q];
                }
            }
            if constexpr (KSP) {
                lds_barrier();  // the round's terms are there
                if (adds && opos < cur.cnt) {
                    const float* tp = terms + ((tid >> 8) * FTS * 16 + orow) * FPP + opos;
                    for (int j = 0; j < se - sb; j++) sum = sum + tp[j * 16 * FPP];
                }
                lds_barrier();  // and read: the next round or item may write its own
            }
        }
        if constexpr (KSP) {
            float* yp = a.y + (int64_t)(cur.m0 + opos) * a.y_stride + cur.n0 + orow;
            const bool mine = adds && opos < cur.cnt && cur.n0 + orow < a.rows;
            if (pair) {
                // the up sums reach the gate sums' threads through the terms' first rows
                if (tid >= 256) terms[tid - 256] = sum;
                lds_barrier();
                if (tid < 256 && mine) *yp = silu_dev(sum) * terms[tid];
                lds_barrier();
            } else if (mine) {
                put(yp, sum);
            }
            sum = 0.0f;
        } else {
            if (cur.n0 + l16 < a.rows) {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (4 * kl + q < cur.cnt) put(a.y + (int64_t)(cur.m0 + 4 * kl + q) * a.y_stride + cur.n0 + l16, acc[q]);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) acc[q] = 0.0f;
        }
        if (nxt.cnt == 0) break;
        cur = nxt;
        xr = xrn;
        nxt = next_item(id, pc, cur);
    }
}

template <int T, bool KSP>
static hipError_t few_launch(const GemmArgs& a, hipStream_t s) {
    const size_t smem = few_smem<T>(KSP, a.pair != 0);
    static bool attr = false;
    if (!attr) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_few_kernel<T, KSP>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)few_smem<T>(KSP, true));
        if (e != hipSuccess) return e;
        attr = true;
    }
    static int ncu = 0;
    if (!ncu) {
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) return e;
    }
    const long long total = ((long long)((a.rows + 15) / 16) * a.max_tiles) << a.few_cs;
    if (total >= (1ll << 31)) return hipErrorInvalidValue;
    const long long want = KSP ? total : (total + FW - 1) / FW;
    const long long grid = std::max<long long>(std::min<long long>(want, 2ll * ncu), 1);  // persistent: two blocks per CU
    gemm_few_kernel<T, KSP><<<dim3((unsigned)grid), 64 * FW, smem, s>>>(a);
    return hipGetLastError();
}

template <int T>
static hipError_t few_t(const GemmLaunch& g, hipStream_t s) {
    GemmArgs a{};
    a.tiles = g.tiles; a.n_tiles_dev = g.n_tiles_dev; a.dense_w = g.dense_w; a.dense_n = g.dense_n;
    a.xq = (const int8_t*)g.xq; a.xd = (const float*)(g.xq + (uint64_t)g.n_x * g.cols);
    a.xrow = g.xrow; a.y = g.y; a.y_stride = g.y_stride; a.rows = g.rows; a.cols = g.cols; a.act = g.act;
    a.pair = g.pair ? 1 : 0;
    a.w2 = g.w2;
    a.rb = row_bytes(T, g.cols);
    a.max_tiles = g.n_tiles;
    // a block for each item while the items are few (dense) or a row has super-blocks for its waves; else a wave each
    bool ksp = g.pair || g.cols >= 1536;
    if (!g.tiles) {
        a.max_tiles = (g.dense_n + FPM - 1) / FPM;
        ksp = few_dense_items(g.rows, g.dense_n) <= FEW_DENSE_BLOCK_ITEMS;
    }
    // with less than an item a wave, a tile's chunks side by side: the largest expert's would otherwise set the time
    if (g.tiles && !ksp && (long long)((g.rows + 15) / 16) * g.n_tiles < FEW_WAVES) a.few_cs = 2;
    return ksp ? few_launch<T, true>(a, s) : few_launch<T, false>(a, s);
}

hipError_t launch_gemv_few(const GemvLaunch& g, hipStream_t s) {
    if (g.ty == Q8_0 || g.numerics != STRATA_NUM_Q8K || !g.xq || g.ids || g.pair || g.cols % 256 ||
        (uint64_t)g.rows * row_bytes(g.ty, g.cols) >= (1ull << 32) || g.rows > (1 << 24) ||
        row_bytes(g.ty, g.cols) >= (1u << 24))
        return hipErrorNotSupported;
    GemmLaunch m;
    m.ty = g.ty; m.rows = g.rows; m.cols = g.cols;
    m.dense_w = g.w; m.dense_n = g.nt; m.n_tiles = 1;
    m.xq = (const uint8_t*)g.xq; m.n_x = g.n_xrows;
    m.y = g.y; m.y_stride = g.y_stride; m.act = STRATA_ACT_STORE;
    return launch_gemm_few(m, s);
}

bool gemm_few_takes_tiles(int ty, int rows, int cols, int n_tiles, bool gathered, int n_x) {
    const long long items = (long long)((rows + 15) / 16) * n_tiles;
    if (ty == Q8_0 || items >= (1ll << 31)) return false;
    if (gathered) return n_x <= few_gathered(ty, cols);
    const FewRows f = few_rows(ty);
    const int slot4 = items < FEW_WAVES / 2 ? 48 : items < FEW_WAVES ? 32 : f.slot4;
    return n_x <= f.rows && 4ll * n_x <= (long long)slot4 * n_tiles;
}

bool gemm_few_takes(const GemmLaunch& g) {
    if (g.ty == Q8_0) return false;
    if (!g.tiles) return g.dense_n <= FPM || few_dense_items(g.rows, g.dense_n) <= FEW_DENSE_ITEMS;
    return g.small && gemm_few_takes_tiles(g.ty, g.rows, g.cols, g.n_tiles, g.xrow != nullptr, g.n_x);
}

hipError_t launch_gemm_few(const GemmLaunch& g, hipStream_t s) {
    switch (g.ty) {
    case Q2_K: return few_t<Q2_K>(g, s);
    case Q3_K: return few_t<Q3_K>(g, s);
    case Q4_K: return few_t<Q4_K>(g, s);
    case Q5_K: return few_t<Q5_K>(g, s);
    case Q6_K: return few_t<Q6_K>(g, s);
    case IQ2_XXS: return few_t<IQ2_XXS>(g, s);
    case IQ3_S: return few_t<IQ3_S>(g, s);
    case IQ4_XS: return few_t<IQ4_XS>(g, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace strata
