// MLA chunked prefill, step 1: expand the cached latents of the sequences in
// the call into per-head keys and values (the decompressed form costs 5.9
// TFLOP on config 4 against 16.4 TFLOP for the absorbed form, because here
// every query row of a head reuses the same expanded K/V tile).
//
//   K_c[h][t][d] = sum_c C[t][c] W_UK[c][h*D+d]     (row-major per head)
//   V^T[h][d][t] = sum_c C[t][c] W_UV[c][h*D+d]     (dim-major per head: the
//                                                    A-operand order of P.V)
//
// C rows come straight from the paged latent pool.  MFMA needs the contracted
// index (c) contiguous per lane in both operands, so W is first packed into
// W^T fragments.  The K_c launch puts features on the MFMA M side (a lane ends
// with consecutive dims of one token: row-major K_c); the V^T launch puts
// tokens there (consecutive tokens of one dim: dim-major V^T).  The GEMM
// itself is mla_expand_kernel below.
#include "rlx_common.h"

#include <algorithm>

namespace rlx {

// W [dc][H*D] -> W^T of H*DP features x 512 channels in 1 KB MFMA fragments,
// element (f, c) at ((f/16 * 16 + c/32) * 16 + f%16) * 32 + c%32, zeros for
// dims d >= D of every head and channels c >= dc (the expansion then writes
// exact zeros for the padded dims, and the zero-padded channels of the latent
// rows meet zero weights).  Thread = 8 channels x 8 features (D a multiple of
// 8), turned in registers: 16-byte loads (by elements where w is not aligned
// for them: the caller's weights may start at any element) and stores.  Bound:
// memory; 16384 features 12 us (17 by 2-byte accesses through LDS).
template <bool VEC>
__global__ __launch_bounds__(256) void mla_wt_kernel(const uint16_t *__restrict__ w,
                                                     uint16_t *__restrict__ wt, int dc, int H, int D,
                                                     int DP) {
    const int f = (blockIdx.x * 256 + threadIdx.x) * 8, c = blockIdx.y * 8;
    if (f >= H * DP) return;
    const int h = f / DP, d = f - h * DP;
    u32x4 r[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        r[k] = u32x4{0, 0, 0, 0};
        if (c + k >= dc || d >= D) continue;
        const uint16_t *p = w + (int64_t)(c + k) * H * D + h * D + d;
        if constexpr (VEC) {
            r[k] = *(const u32x4 *)p;
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) r[k][j] = (uint32_t)p[2 * j] | ((uint32_t)p[2 * j + 1] << 16);
        }
    }
    uint16_t *o = wt + (((int64_t)(f >> 4) * (kMlaDc / 32) + (c >> 5)) * 16 + (f & 15)) * 32 + (c & 31);
#pragma unroll
    for (int e = 0; e < 8; e++) {
        u32x4 v;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t lo = r[2 * j][e >> 1] >> (16 * (e & 1)), hi = r[2 * j + 1][e >> 1] >> (16 * (e & 1));
            v[j] = (lo & 0xFFFFu) | (hi << 16);
        }
        *(u32x4 *)(o + e * 32) = v;
    }
}

// Expansion GEMM.  Work-group = 4 waves, 128 tokens x 4 WF features, c in 8
// steps of 64; wave w holds the sums of all 128 tokens for its WF features, so
// the W^T fragments go from L2 to the registers of the one wave that
// multiplies them, and only the latents pass through LDS (rows of 64 c,
// 16-byte chunk k of row r at slot k ^ ((r >> 1) & 7): no bank conflicts).
// Bound: matrix cores (2 x 512 flop per 2-byte output) and, for the 1 GB a
// launch writes at 32768 tokens x 128 heads, the stores (450 us without
// them).  There K_c takes 596 us (920 TFLOP/s) and V^T 534: 728 and 777 with
// both operands read from LDS by 64 x 64 waves (all of its 128 B a cycle at
// the matrix cores' rate) and one persistent work-group per CU whose stores
// nothing covered; 690 and 700 with 64-byte stores kept in L2, 607 and 555
// with the same non-temporal.
//
// Pipeline per step t: the loads of step t + 1 are issued, step t is
// multiplied, step t + 1's latents go from registers to the other LDS stage,
// one barrier that leaves global loads in flight.
//
// Work order: work-group b runs on XCD b mod 8; each XCD keeps an eighth of
// the feature tiles (2 MB of W^T at 128 heads: its L2) and walks the token
// tiles with them.
constexpr int kXThreads = 256;
constexpr int kXN = 128;               // tokens per tile
constexpr int kXSteps = kMlaDc / 64;

template <int OUT_V, int WF>
__global__ __launch_bounds__(kXThreads, 2) void mla_expand_kernel(
    const uint16_t *__restrict__ pool, const int32_t *__restrict__ table,
    const AttRow *__restrict__ rows, const int2 *__restrict__ work, int n_work,
    const uint16_t *__restrict__ wt, int NT, int n_ft, int H, int P, int dps, uint16_t *__restrict__ dst) {
    constexpr int MI = kXN / 16, NI = WF / 16, XJ = kXN / 32;
    constexpr int kStage = kXN * 128;  // bytes of one step's latents
    constexpr int kLds = 4 * kXN * WF * 2 > 2 * kStage ? 4 * kXN * WF * 2 : 2 * kStage;
    __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, grp = lane >> 4;
    int ft, tt;
    if (n_ft >= 8) {
        const int x = blockIdx.x & 7, i = blockIdx.x >> 3, nf = (n_ft - x + 7) >> 3;
        tt = i / nf;
        ft = x + 8 * (i - tt * nf);
    } else {
        tt = blockIdx.x / n_ft;
        ft = blockIdx.x - tt * n_ft;
    }
    if (tt >= n_work) return;
    const int f0 = (ft * 4 + wave) * NI;  // this wave's first 16-feature fragment
    const int2 wk = work[tt];
    const AttRow R = rows[wk.x];

    // Latents: thread = 16-byte chunk tid % 8 of tokens tid / 8 + 32 j (past
    // the live length: the last live one).
    const int t_hi = min(wk.y + kXN, R.len) - 1;
    const uint16_t *xp[XJ];
#pragma unroll
    for (int j = 0; j < XJ; j++) {
        const int tok = min(wk.y + (tid >> 3) + 32 * j, t_hi);
        xp[j] = pool + ((int64_t)table[R.tab + tok / P] * P + tok % P) * kMlaRow + (tid & 7) * 8;
    }
    struct XRegs {
        u32x4 v[XJ];
    };
    auto load_x = [&](XRegs &r, int t) {
#pragma unroll
        for (int j = 0; j < XJ; j++) r.v[j] = *(const u32x4 *)(xp[j] + min(t, kXSteps - 1) * 64);
    };
    unsigned char *const xw = lds + (tid >> 3) * 128 + (((tid & 7) ^ ((tid >> 4) & 7)) << 4);
    auto store_x = [&](const XRegs &r, int stage) {
#pragma unroll
        for (int j = 0; j < XJ; j++) *(u32x4 *)(xw + stage * kStage + j * 4096) = r.v[j];
    };
    const uint16_t *wb[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ni++) wb[ni] = wt + (int64_t)min(f0 + ni, NT - 1) * (kMlaDc / 32) * 512;
    const uint32_t wl = (uint32_t)(col * 32 + grp * 8);
    struct WRegs {
        u32x4 v[2][NI];
    };
    auto load_w = [&](WRegs &r, int t) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
                r.v[s][ni] = *(const u32x4 *)(wb[ni] + (2 * min(t, kXSteps - 1) + s) * 512 + wl);
    };
    fl4 acc[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++) acc[mi][ni] = fl4{0.f, 0.f, 0.f, 0.f};
    const unsigned char *const xr0 = lds + col * 128 + ((grp ^ ((col >> 1) & 7)) << 4);
    const unsigned char *const xr1 = lds + col * 128 + (((4 + grp) ^ ((col >> 1) & 7)) << 4);
    auto mul = [&](const WRegs &w, int s, int stage) {
        const unsigned char *xr = (s ? xr1 : xr0) + stage * kStage;
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            const bf16x8 x = __builtin_bit_cast(bf16x8, *(const u32x4 *)(xr + mi * 2048));
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                const bf16x8 f = __builtin_bit_cast(bf16x8, w.v[s][ni]);
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(OUT_V ? x : f, OUT_V ? f : x, acc[mi][ni], 0, 0, 0);
            }
        }
    };
    XRegs xg;
    WRegs wg[2];
    load_x(xg, 0);
    load_w(wg[0], 0);
    store_x(xg, 0);
    ring_barrier();
#pragma unroll
    for (int t = 0; t < kXSteps; t++) {
        load_x(xg, t + 1);
        load_w(wg[(t + 1) & 1], t + 1);
        mul(wg[t & 1], 0, t & 1);
        mul(wg[t & 1], 1, t & 1);
        if (t + 1 < kXSteps) {
            store_x(xg, (t + 1) & 1);
            ring_barrier();
        }
    }

    // acc[mi][ni][e]: K_c feature 16 ni + 4 grp + e of token 16 mi + col, V^T
    // token 16 mi + 4 grp + e of feature 16 ni + col.  Two sub-tiles along the
    // contiguous index are paired with one row swap (v_permlane16_swap: odd
    // 16-lane rows of the first operand <-> even rows of the second), after
    // which lane (col, grp) holds its 8 consecutive elements 8 (grp >> 1) + 16
    // (grp & 1) .. + 7.
    const int mo = 8 * (grp >> 1) + 16 * (grp & 1);
    const int Tp = R.nsplit, DP = 1 << dps;  // padded head dim: feature f is dim f % DP of head f / DP
    uint16_t *db = dst + (int64_t)R.part * H * DP;
    auto pair = [&](const fl4 &a, const fl4 &b) {
        const uint32_t x[2] = {pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3])};
        const uint32_t y[2] = {pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
        u32x4 w;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const auto sw = __builtin_amdgcn_permlane16_swap(x[h], y[h], false, false);
            w[h] = sw[0];
            w[2 + h] = sw[1];
        }
        return w;
    };
    // Through the wave's LDS region (K_c [128 tokens][WF], V^T [WF][128 tokens],
    // 16-byte chunks swizzled by row), so that every store instruction writes
    // whole rows of the tile: non-temporal, as the attention kernel reads them
    // back after the launch's gigabyte has passed through the caches.
    if (f0 >= NT) return;
    const int live = min(NI, NT - f0) * 16;  // features of this wave
    ring_barrier();                          // (every wave is done with the stages)
    unsigned char *const mine = lds + wave * (kXN * WF * 2);
    constexpr int CK = WF / 8;  // chunks of a K_c row
    auto kc_at = [&](int tok, int c) { return mine + (tok * CK + (c ^ ((tok / (16 / CK)) & (CK - 1)))) * 16; };
    auto vt_at = [&](int f, int c) { return mine + (f * 16 + (c ^ (f & 15))) * 16; };
#pragma unroll
    for (int ni = 0; ni < NI; ni += OUT_V ? 1 : 2)
#pragma unroll
        for (int mi = 0; mi < MI; mi += OUT_V ? 2 : 1) {
            if constexpr (OUT_V)
                *(u32x4 *)vt_at(16 * ni + col, 2 * mi + mo / 8) = pair(acc[mi][ni], acc[mi + 1][ni]);
            else
                *(u32x4 *)kc_at(16 * mi + col, 2 * ni + mo / 8) = pair(acc[mi][ni], acc[mi][ni + 1]);
        }
#pragma unroll
    for (int i = 0; i < kXN * WF / 512; i++) {
        const int e = i * 64 + lane;
        if constexpr (OUT_V) {
            const int f = e >> 4, c = e & 15;
            if (f < live)
                __builtin_nontemporal_store(*(const u32x4 *)vt_at(f, c),
                                            (u32x4 *)(db + (int64_t)(f0 * 16 + f) * Tp + wk.y + 8 * c));
        } else {
            const int tok = e / CK, c = e % CK, f = f0 * 16 + 8 * c;
            if (8 * c < live)
                __builtin_nontemporal_store(
                    *(const u32x4 *)kc_at(tok, c),
                    (u32x4 *)(db + ((int64_t)(f >> dps) * Tp + wk.y + tok) * DP + (f & (DP - 1))));
        }
    }
}

hipError_t launch_mla_wt(hipStream_t s, const uint16_t *w_uk, const uint16_t *w_uv, int H, int D,
                         int dc, int DP, uint16_t *wt_k, uint16_t *wt_v) {
    if (D > DP || D % 8 != 0 || DP % 64 != 0 || dc > kMlaDc) return hipErrorInvalidValue;
    const dim3 g((H * DP / 8 + 255) / 256, kMlaDc / 8);
    auto pack = [&](const uint16_t *w, uint16_t *wt) {
        if (((uintptr_t)w & 15) == 0)
            mla_wt_kernel<true><<<g, 256, 0, s>>>(w, wt, dc, H, D, DP);
        else
            mla_wt_kernel<false><<<g, 256, 0, s>>>(w, wt, dc, H, D, DP);
    };
    pack(w_uk, wt_k);
    pack(w_uv, wt_v);
    return hipGetLastError();
}

// Rope keys of the call, kr[part + t][0 .. 64) = latent row t's k^R (the
// last 64 entries of the stored row), zero for padding rows t >= len.  One
// block per expansion work item (sequence, 128 tokens); 16-byte chunks.  The
// FA2 kernel then reads each 64-key block's rope keys as one contiguous 8 KB
// region through a running pointer, like K_c.
__global__ __launch_bounds__(256) void mla_rope_gather_kernel(const uint16_t *__restrict__ pool,
                                                              const int32_t *__restrict__ table,
                                                              const AttRow *__restrict__ rows,
                                                              const int2 *__restrict__ work, int P,
                                                              uint16_t *__restrict__ kr) {
    const int2 wk = work[blockIdx.x];
    const AttRow R = rows[wk.x];
    for (int e = threadIdx.x; e < 128 * (kMlaDr / 8); e += blockDim.x) {
        const int t = wk.y + e / (kMlaDr / 8), ch = e % (kMlaDr / 8);
        u32x4 v = u32x4{0, 0, 0, 0};
        if (t < R.len) {
            const int page = table[R.tab + t / P];
            v = *(const u32x4 *)(pool + ((int64_t)page * P + t % P) * kMlaRow + kMlaDc + ch * 8);
        }
        *(u32x4 *)(kr + ((int64_t)R.part + t) * kMlaDr + ch * 8) = v;
    }
}

hipError_t launch_mla_rope_gather(hipStream_t s, const uint16_t *pool, const int32_t *table,
                                  const AttRow *rows, const int2 *work, int n_work, int P,
                                  uint16_t *kr) {
    if (n_work <= 0) return hipSuccess;
    mla_rope_gather_kernel<<<n_work, 256, 0, s>>>(pool, table, rows, work, P, kr);
    return hipGetLastError();
}

hipError_t launch_mla_expand(hipStream_t s, const uint16_t *pool, const int32_t *table,
                             const AttRow *rows, const int2 *work, int n_work, int H, int DP, int P,
                             const uint16_t *wt_k, const uint16_t *wt_v, uint16_t *kc, uint16_t *vt,
                             int cus) {
    if (DP != 128 && DP != 256) return hipErrorInvalidValue;
    const int dps = DP == 128 ? 7 : 8;
    if (n_work <= 0) return hipSuccess;
    // 256 features a work-group where the tiles fill the chip twice, else 128.
    const int NT = H * DP / 16;
    const bool wide = (int64_t)((NT + 15) / 16) * n_work >= 2 * cus;
    const int n_ft = wide ? (NT + 15) / 16 : (NT + 7) / 8;
    // (work-groups of the XCD with the most feature tiles, times 8)
    const int grid = n_ft >= 8 ? (n_ft + 7) / 8 * n_work * 8 : n_ft * n_work;
#define RLX_EXPAND(V, WF, W, D) \
    mla_expand_kernel<V, WF><<<grid, kXThreads, 0, s>>>(pool, table, rows, work, n_work, W, NT, n_ft, H, P, dps, D)
    if (wide) {
        RLX_EXPAND(0, 64, wt_k, kc);
        RLX_EXPAND(1, 64, wt_v, vt);
    } else {
        RLX_EXPAND(0, 32, wt_k, kc);
        RLX_EXPAND(1, 32, wt_v, vt);
    }
#undef RLX_EXPAND
    return hipGetLastError();
}

}  // namespace rlx
