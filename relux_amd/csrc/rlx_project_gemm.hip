// The projections of rlx_project.hip at prefill sizes (proj_use_gemm):
// one MFMA GEMM over all rows with the same epilogues --
// RoPE, the paged append, the q outputs; or out = x.W (+ residual).
//
// Bound: matrix cores (2 * rows * N * K flop over 2 * (rows + N) * K bytes:
// at 1531 rows of a 4096-wide layer 1 100 flop/B).  The decode-size kernels
// stream the whole weight matrix for every 64 rows instead.  Measured, 1531
// bf16 rows at d_model 4096: Q/K/V projection, RoPE and append (N 6144) 24
// launches and 980 us -> 121 us (640 TFLOP/s); W_O + residual (N 4096) 574 ->
// 73 us.  At 8192 rows of N 6144 the tiles alone reach 960 TFLOP/s.
//
// Work-group = 4 waves, a tile of BM rows x 4 * WF features; wave w holds
// the sums of all BM rows for its WF features, so the packed weights -- 1 KB
// MFMA fragments in memory -- go straight from L2 to the registers of the
// one wave that multiplies them, and only the activations pass through LDS
// (rows of 64 k, 16-byte chunk c of row r at slot c ^ ((r >> 1) & 7): any 16
// consecutive lanes of a 16-byte read or write touch distinct slots of the
// 64 banks).  Weights are the MFMA A operand and activations the B operand:
// a result lane then holds 4 consecutive features of one row, so a RoPE pair
// is in one lane, a row's placement is read once per row tile, and q, K and
// latent rows are written 4 elements at a time.
//
// Pipeline per 64-wide k-step t: the loads of step t + PF are issued, step t
// is multiplied, step t + 1's activations go from registers to the other LDS
// stage, one barrier that leaves global loads in flight.  f32 activations
// are split into hi + lo bf16 pairs on their way to LDS (proj_split2) and
// both are multiplied, as the decode-size kernels do.
//
// Work order: work-group b runs on XCD b mod 8; each XCD takes a contiguous
// run of tiles, row tiles fastest, so that its work-groups read the same
// weight fragments at the same time.
#include "rlx_project.h"

namespace rlx {

constexpr int kPgThreads = 256;
constexpr int kPgGroup = 16;  // row tiles of one run of feature tiles

template <bool XBF16, int MODEL, int BM, int WF, int PF, int UN>
__global__ __launch_bounds__(kPgThreads, 2) void proj_gemm_kernel(
    const Patch *__restrict__ patches, int n_patch, const AppendTok *__restrict__ toks,
    const int32_t *__restrict__ pos_dev, int rows, const void *__restrict__ x, int K,
    const uint16_t *__restrict__ wp, int NT, int tiles_m, int tiles_n, const ProjDims pd,
    const float *__restrict__ rcos, const float *__restrict__ rsin, void *__restrict__ q_out,
    void *__restrict__ q_out2, int q_bf16, int vec, int rope2, uint16_t *__restrict__ kpool,
    uint16_t *__restrict__ vpool, int32_t *__restrict__ table, int P) {
    constexpr int MI = BM / 16, NI = WF / 16, XJ = BM / 32;
    constexpr int XH = XBF16 ? 1 : 2;           // bf16 images of the activations (hi, lo)
    constexpr int kStage = BM * 128;            // bytes of one image of one k-step
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * XH * kStage];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, grp = lane >> 4;
    if (blockIdx.x == 0) {
        for (int i = tid; i < n_patch; i += kPgThreads) {
            const Patch pt = patches[i];
            table[pt.idx] = pt.val;
        }
    }
    const int total = tiles_m * tiles_n, per = (total + 7) >> 3;
    const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (id >= total) return;
    const int g0 = id / (kPgGroup * tiles_n) * kPgGroup;
    const int gm = min(kPgGroup, tiles_m - g0), rem = id - g0 * tiles_n;
    const int m0 = (g0 + rem % gm) * BM;
    const int f0 = rem / gm * (4 * NI) + wave * NI;  // this wave's first 16-feature fragment
    const int KS = K >> 5, steps = (KS + 1) >> 1;

    // Activations: thread = 16-byte chunk c of rows (tid / 8) + 32 j.
    const int c = tid & 7;
    const int esz = XBF16 ? 2 : 4;
    const char *xbase = (const char *)x + (int64_t)m0 * K * esz;
    uint32_t xrow[XJ];
#pragma unroll
    for (int j = 0; j < XJ; j++) xrow[j] = (uint32_t)min((tid >> 3) + 32 * j, rows - 1 - m0) * (uint32_t)(K * esz);
    struct XRegs {
        u32x4 v[XJ * (XBF16 ? 1 : 2)];
    };
    auto load_x = [&](XRegs &r, int t) {
        // (past the last k: the last whole chunk, in bounds; never multiplied)
        const uint32_t ko = (uint32_t)min(min(t, steps - 1) * 64 + c * 8, K - 8) * esz;
#pragma unroll
        for (int j = 0; j < XJ; j++) {
            if constexpr (XBF16) {
                r.v[j] = *(const u32x4 *)(xbase + xrow[j] + ko);
            } else {
                r.v[2 * j] = *(const u32x4 *)(xbase + xrow[j] + ko);
                r.v[2 * j + 1] = *(const u32x4 *)(xbase + xrow[j] + ko + 16);
            }
        }
    };
    unsigned char *const xw = lds + (tid >> 3) * 128 + ((c ^ ((tid >> 4) & 7)) << 4);
    auto store_x = [&](const XRegs &r, int stage) {
        unsigned char *w = xw + stage * XH * kStage;
#pragma unroll
        for (int j = 0; j < XJ; j++) {
            if constexpr (XBF16) {
                *(u32x4 *)(w + j * 4096) = r.v[j];
            } else {
                const float4 a = __builtin_bit_cast(float4, r.v[2 * j]);
                const float4 b = __builtin_bit_cast(float4, r.v[2 * j + 1]);
                const u32x2 p0 = proj_split2(a.x, a.y), p1 = proj_split2(a.z, a.w);
                const u32x2 p2 = proj_split2(b.x, b.y), p3 = proj_split2(b.z, b.w);
                *(u32x4 *)(w + j * 4096) = u32x4{p0[0], p1[0], p2[0], p3[0]};
                *(u32x4 *)(w + kStage + j * 4096) = u32x4{p0[1], p1[1], p2[1], p3[1]};
            }
        }
    };
    // Weights: fragment ni of this wave, k-step ks: 1 KB at wb[ni] + ks KB
    // (fragments past the last read the last one; their sums are dropped).
    const uint16_t *wb[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ni++) wb[ni] = wp + (int64_t)min(f0 + ni, NT - 1) * KS * 512;
    const uint32_t wl = (uint32_t)(col * 32 + grp * 8);
    struct WRegs {
        u32x4 v[2][NI];
    };
    auto load_w = [&](WRegs &r, int t) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
                r.v[s][ni] = *(const u32x4 *)(wb[ni] + (int64_t)min(2 * t + s, KS - 1) * 512 + wl);
    };
    // A chain of at most 12 k-steps and a quarter of them (acc), and the sum
    // of the chains: one chain over all of k would round more often than the
    // decode-size kernels' k-split over 4 waves does (K 4096, f32 output,
    // relative error against f64: chains 1.6e-7, decode-size kernels 1.9e-7).
    const int chain = min(12, (steps + 15) >> 4 << 2);
    fl4 acc[MI][NI], sum[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++) acc[mi][ni] = sum[mi][ni] = fl4{0.f, 0.f, 0.f, 0.f};
    auto flush = [&]() {
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                sum[mi][ni] += acc[mi][ni];
                acc[mi][ni] = fl4{0.f, 0.f, 0.f, 0.f};
            }
    };
    const unsigned char *const xr0 = lds + col * 128 + ((grp ^ ((col >> 1) & 7)) << 4);
    const unsigned char *const xr1 = lds + col * 128 + (((4 + grp) ^ ((col >> 1) & 7)) << 4);
    auto mul = [&](const WRegs &w, int s, int stage) {
        const unsigned char *xr = (s ? xr1 : xr0) + stage * XH * kStage;
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int e = 0; e < XH; e++) {
                const u32x4 v = *(const u32x4 *)(xr + e * kStage + mi * 2048);
#pragma unroll
                for (int ni = 0; ni < NI; ni++)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, w.v[s][ni]), __builtin_bit_cast(bf16x8, v), acc[mi][ni], 0, 0, 0);
            }
    };
    XRegs xg[PF];
    WRegs wg[PF + 1];
#pragma unroll
    for (int t = 0; t < PF; t++) {
        load_x(xg[t], t);
        load_w(wg[t], t);
    }
    store_x(xg[0], 0);
    ring_barrier();
    // Step t: x(t) is in LDS stage t & 1; x(t + 1 .. t + PF - 1) and
    // w(t .. t + PF - 1) are in flight or in registers.
    for (int t0 = 0; t0 < steps; t0 += UN) {
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const int t = t0 + u;
            if (t >= steps) break;
            if (u % 4 == 0 && t % chain == 0) flush();
            load_x(xg[u % PF], t + PF);
            load_w(wg[(u + PF) % (PF + 1)], t + PF);
            const int stage = t & 1;
            mul(wg[u % (PF + 1)], 0, stage);
            if (2 * t + 1 < KS) mul(wg[u % (PF + 1)], 1, stage);
            store_x(xg[(u + 1) % PF], stage ^ 1);
            ring_barrier();
        }
    }
    flush();

    // ---- output: lane = features n .. n + 3 of rows m0 + 16 mi + col --------
    const int r0 = m0 + col;
    int pos[MI], page[MI], slot[MI];
    if constexpr (MODEL != kProjOut) {
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            const int rr = min(r0 + mi * 16, rows - 1);
            pos[mi] = pos_dev[rr];
            const int2 tk = *(const int2 *)(toks + rr);
            page[mi] = tk.x;
            slot[mi] = tk.y;
        }
    }
    auto pack4 = [](const fl4 &v) {
        return u32x2{(uint32_t)bf16_rne(v[0]) | ((uint32_t)bf16_rne(v[1]) << 16),
                     (uint32_t)bf16_rne(v[2]) | ((uint32_t)bf16_rne(v[3]) << 16)};
    };
    // The first cnt of 4 consecutive elements of a q / out buffer.
    auto put = [&](void *dst, int64_t off, const fl4 &v, int cnt) {
        if (vec && cnt >= 4) {
            if (q_bf16)
                *(u32x2 *)((uint16_t *)dst + off) = pack4(v);
            else
                *(fl4 *)((float *)dst + off) = v;
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (i < cnt) {
                if (q_bf16)
                    ((uint16_t *)dst)[off + i] = bf16_rne(v[i]);
                else
                    ((float *)dst)[off + i] = v[i];
            }
    };
#pragma unroll
    for (int ni = 0; ni < NI; ni++) {
        if (f0 + ni >= NT) break;
        const int n0 = (f0 + ni) * 16;
        if constexpr (MODEL == kProjOut) {
            const int n = n0 + grp * 4, cnt = pd.D - n;
#pragma unroll
            for (int mi = 0; mi < MI; mi++) {
                const int r = r0 + mi * 16;
                if (r >= rows) continue;
                const int64_t off = (int64_t)r * pd.D + n;
                fl4 v = sum[mi][ni];
                if (q_out2) {
                    if (vec && cnt >= 4) {
                        if (q_bf16) {
                            const u32x2 a = *(const u32x2 *)((const uint16_t *)q_out2 + off);
                            v += fl4{bf16_lo(a[0]), bf16_hi(a[0]), bf16_lo(a[1]), bf16_hi(a[1])};
                        } else {
                            v += *(const fl4 *)((const float *)q_out2 + off);
                        }
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (i < cnt)
                                v[i] += q_bf16 ? bf16_f32(((const uint16_t *)q_out2)[off + i])
                                               : ((const float *)q_out2)[off + i];
                    }
                }
                put(q_out, off, v, cnt);
            }
        } else {
            // Part, heads and dims: uniform per fragment when a head is whole
            // 16-feature fragments, else (narrow heads packed unpadded) per lane.
            int part, nn0, hw, tw;
            proj_part<MODEL>(pd, n0, part, nn0, hw, tw);
            const int nn = nn0 + grp * 4;
            if (hw) {
                // RoPE: (x0, x1) -> (x0 c - x1 s, x1 c + x0 s), products
                // rounded separately as in rope.go.
                auto turn = [&](fl4 &v, int i, float cs, float sn) {
                    const float x0 = v[i], x1 = v[i + 1];
                    v[i] = __fsub_rn(__fmul_rn(x0, cs), __fmul_rn(x1, sn));
                    v[i + 1] = __fadd_rn(__fmul_rn(x1, cs), __fmul_rn(x0, sn));
                };
                if (rope2 && (hw & 15) == 0) {  // both pairs of the lane in one load
                    const int dr = nn0 % hw + grp * 4;
#pragma unroll
                    for (int mi = 0; mi < MI; mi++) {
                        if (pos[mi] < 0 || dr >= tw) continue;
                        const int64_t at = (int64_t)pos[mi] * (tw >> 1) + (dr >> 1);
                        const float2 cs = *(const float2 *)(rcos + at), sn = *(const float2 *)(rsin + at);
                        turn(sum[mi][ni], 0, cs.x, sn.x);
                        turn(sum[mi][ni], 2, cs.y, sn.y);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i += 2) {
                        const int dr = (nn + i) % hw;
#pragma unroll
                        for (int mi = 0; mi < MI; mi++) {
                            if (pos[mi] < 0 || dr >= tw) continue;
                            const int64_t at = (int64_t)pos[mi] * (tw >> 1) + (dr >> 1);
                            turn(sum[mi][ni], i, rcos[at], rsin[at]);
                        }
                    }
                }
            }
            const bool qr = MODEL == kProjMLA && part == 1;
            const bool to_q = (MODEL == kProjGQA) ? part == 0 : part < 2;
            const int hdim = qr ? pd.DRP : pd.DW;  // packed features of a head
            const int width = qr ? pd.DR : pd.D;   // stored dims of a head
            // Elements 4 at a time when the stored dims are a multiple of 4
            // (a lane's features are then in one head, all stored or none),
            // else one by one.
            if (MODEL == kProjMLA && !to_q) {
                // latent c^KV dims < DC, k^R dims < DR (the row's padding is zeroed apart)
                const int cnt = (part == 2 ? pd.DC : pd.DR) - nn;
#pragma unroll
                for (int mi = 0; mi < MI; mi++) {
                    if (r0 + mi * 16 >= rows) continue;
                    uint16_t *dst = kpool + ((int64_t)page[mi] * P + slot[mi]) * kMlaRow +
                                    (part == 2 ? 0 : kMlaDc) + nn;
                    const u32x2 pk = pack4(sum[mi][ni]);
                    if (cnt >= 4) {
                        *(u32x2 *)dst = pk;
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (i < cnt) dst[i] = (uint16_t)(pk[i >> 1] >> (16 * (i & 1)));
                    }
                }
            } else if ((width & 3) == 0 && (to_q || part == 1)) {
                const int head = (hdim & 15) ? nn / hdim : nn0 / hdim;
                const int d = (hdim & 15) ? nn % hdim : nn0 % hdim + grp * 4;
#pragma unroll
                for (int mi = 0; mi < MI; mi++) {
                    const int r = r0 + mi * 16;
                    if (r >= rows || d >= width) continue;
                    if (to_q)
                        put(qr ? q_out2 : q_out, ((int64_t)r * pd.H + head) * width + d, sum[mi][ni], 4);
                    else
                        *(u32x2 *)(kpool + ((int64_t)page[mi] * pd.KVH + head) * P * pd.DS +
                                   k_page_off(slot[mi], d, pd.DS)) = pack4(sum[mi][ni]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int head = (hdim & 15) ? (nn + i) / hdim : nn0 / hdim;
                    const int d = (hdim & 15) ? (nn + i) % hdim : nn0 % hdim + grp * 4 + i;
#pragma unroll
                    for (int mi = 0; mi < MI; mi++) {
                        const int r = r0 + mi * 16;
                        if (r >= rows || d >= width) continue;
                        const float v = sum[mi][ni][i];
                        const int64_t hb = (int64_t)page[mi] * pd.KVH + head;
                        if (to_q) {
                            const int64_t off = ((int64_t)r * pd.H + head) * width + d;
                            if (q_bf16)
                                ((uint16_t *)(qr ? q_out2 : q_out))[off] = bf16_rne(v);
                            else
                                ((float *)(qr ? q_out2 : q_out))[off] = v;
                        } else if (part == 1) {
                            kpool[hb * P * pd.DS + k_page_off(slot[mi], d, pd.DS)] = bf16_rne(v);
                        } else {  // (16 lanes: 16 rows, consecutive slots of a dim)
                            vpool[(hb * pd.DS + d) * P + slot[mi]] = bf16_rne(v);
                        }
                    }
                }
            }
        }
    }
}

hipError_t launch_proj_gemm(hipStream_t s, int model, const Patch *patches, int n_patch,
                            const AppendTok *toks, const int32_t *pos, int rows, const void *x,
                            int x_bf16, int K, const uint16_t *wp, const ProjDims &pd,
                            const float *rcos, const float *rsin, void *q_out, void *q_out2,
                            int q_bf16, uint16_t *kpool, uint16_t *vpool, int32_t *table, int P,
                            int cus, hipEvent_t e0, hipEvent_t e1) {
    const int N = proj_features(model, pd);
    if (rows <= 0 || K <= 0 || K % 32 != 0 || N % 16 != 0) return hipErrorInvalidValue;
    const int NT = N / 16;
    // 4-element q / out / residual accesses: rows of a multiple of 4
    // elements (checked per part in the kernel; here kProjOut's) on bases
    // aligned to one access.
    const uintptr_t am = q_bf16 ? 7 : 15;
    const int vec = (((uintptr_t)q_out | (uintptr_t)q_out2) & am) == 0 &&
                    (model != kProjOut || pd.D % 4 == 0);
    // (cos, sin) of two pairs in one access: rotated widths of a multiple of
    // 4 on tables aligned to 8 bytes.
    const int tw = model == kProjModelMLA ? pd.DR : pd.D;
    const int rope2 = tw % 4 == 0 && (((uintptr_t)rcos | (uintptr_t)rsin) & 7) == 0;
    // Tile shape: the least time for the most tiles one CU runs (n), from
    // the time of 1, 2 and each of 3 or more tiles a CU in us at K = 4096
    // (every shape's time is proportional to K).  Measured, N = 4096 and
    // 6144, 65 to 8192 rows: a lone tile is bound by its chain of k-steps
    // (so small tiles win until every CU has one), many by the matrix cores
    // and LDS, where the large one is 1.6 times as fast per output.
    struct Shape {
        int bm, wf;
        float us[2][3];  // bf16, f32 activations
    };
    static const Shape shapes[] = {{128, 32, {{43.5f, 70.f, 37.f}, {107.f, 162.f, 83.f}}},
                                   {64, 32, {{25.5f, 46.f, 23.8f}, {59.f, 98.f, 46.f}}},
                                   {64, 16, {{21.f, 29.5f, 15.1f}, {53.f, 72.f, 33.5f}}}};
    const char *forced = getenv("RLX_PROJ_GEMM");  // override: tile shape 0 to 2 (tests; read per call)
    int best = forced ? atoi(forced) : -1;
    if (best < 0 || best > 2) {
        float cost = 0.f;
        for (int i = 0; i < 3; i++) {
            const int64_t tiles = (int64_t)((rows + shapes[i].bm - 1) / shapes[i].bm) *
                                  ((NT + shapes[i].wf / 4 - 1) / (shapes[i].wf / 4));
            const int64_t n = (tiles + cus - 1) / cus;
            const float *us = shapes[i].us[x_bf16 ? 0 : 1];
            const float c = n <= 2 ? us[n - 1] : us[2] * (float)n;
            if (i == 0 || c < cost) {
                cost = c;
                best = i;
            }
        }
    }
    const int tm = (rows + shapes[best].bm - 1) / shapes[best].bm;
    const int tn = (NT + shapes[best].wf / 4 - 1) / (shapes[best].wf / 4);
    const dim3 grid((unsigned)((tm * tn + 7) / 8 * 8)), block(kPgThreads);
#define RLX_PG(XB, MODELV, BMV, WFV, PFV, UNV)                                                            \
    return launch_timed(proj_gemm_kernel<XB, MODELV, BMV, WFV, PFV, UNV>, grid, block, s, e0, e1, patches, \
                        n_patch, toks, pos, rows, x, K, wp, NT, tm, tn, pd, rcos, rsin, q_out, q_out2, \
                        q_bf16, vec, rope2, kpool, vpool, table, P)
#define RLX_PG_SHAPE(XB, MODELV)                  \
    if (best == 0) RLX_PG(XB, MODELV, 128, 32, 1, 4); \
    if (best == 1) RLX_PG(XB, MODELV, 64, 32, 2, 12); \
    RLX_PG(XB, MODELV, 64, 16, 2, 12);
#define RLX_PG_MODEL(MODELV)           \
    if (x_bf16) {                      \
        RLX_PG_SHAPE(true, MODELV)     \
    } else {                           \
        RLX_PG_SHAPE(false, MODELV)    \
    }
    if (model == kProjGQA) {
        RLX_PG_MODEL(kProjGQA)
    } else if (model == kProjMLA) {
        RLX_PG_MODEL(kProjMLA)
    } else {
        RLX_PG_MODEL(kProjOut)
    }
#undef RLX_PG_MODEL
#undef RLX_PG_SHAPE
#undef RLX_PG
}

}  // namespace rlx
