// Whole-prompt prefill kernels for gfx950 (omega_gpu_pf_*): the activation quantiser, the grouped
// W8A8 GEMM over a tile table, the router logits in the packed layout, the MoE weighted combine,
// and the session memory the prefill driver allocates.
//
// Boundary: crates/aien-omega-pf/src/lib.rs:384-456 (the extern "C" blocks) with the semantics of
// its host mirrors: build_tiles (:122-160, the tile table), router_logits_ref (:505-517, the
// sequential f32 router sum from -0.0 over the packed layout of pack_router, :466-478),
// moe_combine_ref (:519-539, the slot-order combine from +0.0) and the quantiser of
// crates/aien-inference-abi/src/qwen3_moe_omega_prefill/fake_quant.rs:31-104 (power-of-two block
// scale, e4m3 round-to-nearest-even saturating to 448), whose golden table is pq_golden.txt.
// The driver that calls them is qwen3_moe_omega_prefill.rs:483-760 (WholePromptPrefill::run).
//
// Every entry is synchronous: it returns after the chip finished, with the chip nanoseconds of
// its launches (HIP events on the library stream) in *ns, also added to the module's counters.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <type_traits>
#include <utility>
#include <vector>

#include <pthread.h>

#include "device.hpp"
#include "kernels.hpp"
#include "mfma.hpp"
#include "runtime.hpp"

namespace omega {

// One tile-table entry, byte for byte the reference's Tile (aien-omega-pf/src/lib.rs:83-93).
typedef OmegaGpuPfTile PfTile;

constexpr uint32_t kPfBm = 64;  // activation rows per tile
constexpr uint32_t kPfLayoutPlain = 0, kPfLayoutSwiglu = 2;

// ------------------------------------------------------------------ quantiser
struct PfQuantArgs {
    uint32_t k = 0, rows = 0;
    const void *x = nullptr;
    uint8_t *q = nullptr;  // [rows][k]
    float *s = nullptr;    // [rows][k / 128]
};

// e4m3 codes of two values already scaled into +-448 (beyond it, and NaN: the largest code of the
// value's sign), round to nearest even
template <bool HI>
__device__ __forceinline__ int e4m3_pair(float a, float b, int old) {
    auto sat = [](float f) {
        const uint32_t u = __float_as_uint(f);
        return __uint_as_float((u & 0x80000000u) | min(u & 0x7fffffffu, 0x43e00000u));
    };
    return __builtin_amdgcn_cvt_pk_fp8_f32(sat(a), sat(b), old, HI);
}

// A 128-block per 128 / V lanes, V consecutive values a lane; the blocks of all rows are one list.
// V 8 (16 lanes, 16-byte loads, 8-byte stores, the block maximum inside a 16-lane row) is the form
// for 16-byte aligned rows, V 2 (one wavefront a block) for other addresses. Bound by its bytes
// through HBM and L2. Launch times, V 2 for everything before: 16000 rows of 768 bf16 values 22.8 ->
// 8.7 us (4.2 TB/s), 2000 rows of 2048 f32 values 10.3 -> 6.6 us, an empty launch being 6.
template <bool BF16, int V>
__global__ __launch_bounds__(256) void k_pf_quant(const PfQuantArgs a) {
    constexpr uint32_t kLanes = 128 / V;
    const uint64_t item = (uint64_t)blockIdx.x * (256 / kLanes) + threadIdx.x / kLanes;
    if (item >= (uint64_t)a.rows * (a.k / 128)) return;
    const uint32_t l = threadIdx.x % kLanes;
    const size_t at = (size_t)item * 128 + V * l;
    float v[V];
    if constexpr (BF16) {
        uint32_t w[V / 2];
        const uint16_t *x = static_cast<const uint16_t *>(a.x) + at;
        if constexpr (V == 8) {
            const u32x4 t = *as_global(x);
            w[0] = t.x, w[1] = t.y, w[2] = t.z, w[3] = t.w;
        } else {
            w[0] = *as_global_u32(x);
        }
#pragma unroll
        for (int i = 0; i < V / 2; ++i) {
            v[2 * i] = __uint_as_float(w[i] << 16);
            v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
    } else {
        const float *x = static_cast<const float *>(a.x) + at;
        if constexpr (V == 8) {
            const f32x4 t = *as_global_f32x4(x), u = *as_global_f32x4(x + 4);
            v[0] = t.x, v[1] = t.y, v[2] = t.z, v[3] = t.w, v[4] = u.x, v[5] = u.y, v[6] = u.z, v[7] = u.w;
        } else {
            const u32x2 t = *as_global_u32x2(x);
            v[0] = __uint_as_float(t.x), v[1] = __uint_as_float(t.y);
        }
    }
    float m = fabsf(v[0]);
#pragma unroll
    for (int i = 1; i < V; ++i) m = fmaxf(m, fabsf(v[i]));
    m = row16_max(m);
    if constexpr (V == 2)
        m = fmaxf(fmaxf(readlane_f32(m, 0), readlane_f32(m, 16)), fmaxf(readlane_f32(m, 32), readlane_f32(m, 48)));
    m = fmaxf(m, 7.888609052210118e-31f);  // 2^-100
    // scale 2^(E - 8), or 2^(E - 7) when the mantissa is above 1.75 (E the exponent of m)
    const uint32_t mb = __float_as_uint(m), e = mb >> 23, c = ((mb & 0x7fffffu) + 0x1fffffu) >> 23;
    const float scale = __uint_as_float((e + c - 8u) << 23), inv = __uint_as_float((262u - e - c) << 23);
    if constexpr (V == 8) {
        u32x2 q;
        q.x = (uint32_t)e4m3_pair<true>(v[2] * inv, v[3] * inv, e4m3_pair<false>(v[0] * inv, v[1] * inv, 0));
        q.y = (uint32_t)e4m3_pair<true>(v[6] * inv, v[7] * inv, e4m3_pair<false>(v[4] * inv, v[5] * inv, 0));
        *reinterpret_cast<u32x2 *>(a.q + at) = q;
    } else {
        *reinterpret_cast<uint16_t *>(a.q + at) = (uint16_t)e4m3_pair<false>(v[0] * inv, v[1] * inv, 0);
    }
    if (l == 0) a.s[item] = scale;
}

// ------------------------------------------------------------------ grouped W8A8 GEMM
// Workgroup = 64 RW weight rows (PLAIN: output columns 64 RW x ..; SWIGLU: gate rows 32 RW x .. and
// the up rows of the same act columns) x one tile of up to 64 activation rows, RW x 2 wavefronts of
// 64 weight rows x half of the activation rows each. RW 2 (three workgroups a CU) is the general
// form. The paired form (RW 4, PLAIN) also takes two consecutive tiles of one expert at once; the
// second tile's workgroup then leaves.
//
// What bounds it is the traffic into the CUs (about 20 bytes a clock each, L2 included) and, for
// small tiles, the weights from HBM. So a load instruction of a wavefront reads 8 rows x one whole
// 128-byte line (operand-shaped loads, 16 rows x 64 bytes, left the streams a third slower), rows
// past the tile's count repeat its last row (an L1 hit), and XCDs own ranges of tiles or spans.
// Both operands go through LDS, one 128-column k-block at a time: a thread loads 16-byte pieces in
// registers two k-blocks ahead, writes them to the buffer that the previous step read, and one
// barrier per k-block hands it over. Piece c of row r sits at slot c ^ (r % 8) of the row, so the
// 16 rows that a matrix-core operand read touches fall on distinct banks without padding. Per
// k-block, the e4m3 products run with the activation block scale as the B operand's E8M0 scale (a
// power of two, so the products stay exact) and the f32 block sum is multiplied by the weight block
// scale into the accumulator.
//
// Measured (launch times; the form with the weights loaded straight into operand registers and one
// 64 x 128 tile per workgroup before): q|k|v 5120 x 2048 at 512 rows 31 -> 24 us, 4096 rows 170 ->
// 93 us; o 2048 x 4096 at 4096 rows 135 -> 57 us; 128 experts at 2000 tokens gate|up 299 -> 151 us,
// down 162 -> 110 us; at 100 tokens 108 -> 76 and 61 -> 38 us.
// Tiles of up to 32 rows stage, read and multiply 32 (BT 1), not 64: 128 experts of 64 tokens gate|up
// 68.8 -> 61.8 us, down 35.2 -> 30.1; of 200 tokens 82.6 -> 79.0 and 41.4 -> 39.1, of 517 95.1 -> 92.1
// and 51.6 -> 49.9.
struct PfGemmArgs {
    uint32_t n = 0, k = 0, layout = 0, ntiles = 0;
    uint32_t by_cols = 0;  // an XCD takes a range of column spans (else a range of tiles)
    uint32_t per = 0;      // workgroups of an XCD's range
    const PfTile *tiles = nullptr;
    const uint32_t *rowidx = nullptr;  // nullptr: output row r reads activation row r
    const uint8_t *xq = nullptr;       // [rows][k] e4m3
    const float *xs = nullptr;         // [rows][k / 128]
    void *y = nullptr;                 // PLAIN f32 [rows][n]; SWIGLU bf16 [rows][n / 2]
};

constexpr uint32_t kPfMaxKb = 32768 / 128;

template <int AROWS, int BROWS>
struct PfLds {
    uint8_t a[2][AROWS * 128];
    uint8_t b[2][BROWS * 128];
    int sb[2][BROWS];        // E8M0 exponents of the rows' block scales
    float ws[2][kPfMaxKb];   // weight block scales of the two halves of the weight rows
};

// the two 16-byte pieces of a lane's operand: row n of the 16 rows at `t`, pieces g and g + 4
__device__ __forceinline__ i32x8 pf_frag(const uint8_t *t, uint32_t off) {
    const u32x4 lo = *reinterpret_cast<const u32x4 *>(t + off), hi = *reinterpret_cast<const u32x4 *>(t + (off ^ 64));
    return i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
}

// RW x 2 wavefronts: 64 RW weight rows; BT: 16-row B tiles per wavefront (1: a tile of up to 32 rows,
// 2: one of up to 64, 4: two)
template <int LAYOUT, int RW, int BT, class Lds>
__device__ __forceinline__ void pf_qgemm_wg(const PfGemmArgs &a, Lds &L, uint64_t w_va, uint64_t s_va, uint32_t x,
                                            uint32_t row0, uint32_t cnt) {
    const uint32_t tid = threadIdx.x, lane = lane_id(), w = tid >> 6, g = lane >> 4, n = lane & 15;
    const uint32_t KB = a.k / 128, wr = w >> 1, wc = w & 1;
    // first weight row of the two halves
    constexpr bool kSwiglu = LAYOUT == kPfLayoutSwiglu;
    constexpr uint32_t kThreads = 128 * RW, kHalf = 32 * RW, kPass = 16 * RW, NB = 2 * BT / RW;
    const uint32_t h0 = kSwiglu ? kHalf * x : 2 * kHalf * x;
    const uint32_t h1 = kSwiglu ? a.n / 2 + h0 : h0 + kHalf;
    const uint8_t *wt = reinterpret_cast<const uint8_t *>(w_va);
    const float *ws = reinterpret_cast<const float *>(s_va);
    for (uint32_t i = tid; i < KB; i += kThreads) {
        L.ws[0][i] = *as_global_f32(ws + (size_t)(h0 >> 7) * KB + i);
        L.ws[1][i] = *as_global_f32(ws + (size_t)(h1 >> 7) * KB + i);
    }
    // staging: thread t takes pieces of rows t / 8 + kPass i, slot t % 8
    const uint32_t sr = tid >> 3, piece = ((tid & 7) ^ (sr & 7)) * 16;
    const uint32_t woff = sr * a.k + piece;
    const uint8_t *xp[NB];
    const float *xsp[NB];
#pragma unroll
    for (uint32_t i = 0; i < NB; ++i) {
        const uint32_t r = row0 + min(sr + kPass * i, cnt - 1), src = a.rowidx ? *as_global_u32(a.rowidx + r) : r;
        xp[i] = a.xq + (size_t)src * a.k + piece;
        xsp[i] = a.xs + (size_t)src * KB;
    }
    struct Set {
        u32x4 a[4], b[NB];
        float s[NB];
    };
    auto load = [&](Set &S, uint32_t kb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) S.a[i] = *as_global(wt + ((size_t)((i < 2 ? h0 : h1) + kPass * (i & 1)) * a.k + 128 * kb) + woff);
#pragma unroll
        for (uint32_t i = 0; i < NB; ++i) S.b[i] = *as_global(xp[i] + 128 * kb);
#pragma unroll
        for (uint32_t i = 0; i < NB; ++i) S.s[i] = *as_global_f32(xsp[i] + kb);
    };
    auto stage = [&](const Set &S, int u) {
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4 *>(L.a[u] + 16 * tid + 16 * kThreads * i) = S.a[i];
#pragma unroll
        for (uint32_t i = 0; i < NB; ++i) *reinterpret_cast<u32x4 *>(L.b[u] + 16 * tid + 16 * kThreads * i) = S.b[i];
        if ((tid & 7) == 0)
#pragma unroll
            for (uint32_t i = 0; i < NB; ++i) L.sb[u][sr + kPass * i] = e8m0_of(S.s[i]);
    };
    f32x4 tot[4][BT];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < BT; ++j) tot[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t off = n * 128 + ((g ^ (n & 7)) << 4);
    // 16-row A tiles of the wavefront: PLAIN 4 wr .. 4 wr + 3; SWIGLU gate tiles 2 wr, 2 wr + 1 and
    // the up tiles of the same columns
    const uint32_t at0 = kSwiglu ? 2 * wr : 4 * wr;
    const uint32_t at2 = kSwiglu ? 2 * RW + 2 * wr : 4 * wr + 2;
    auto multiply = [&](uint32_t kb, int u) {
        const uint8_t *la = L.a[u], *lb = L.b[u] + 16 * BT * wc * 128;
        const i32x8 A[4] = {pf_frag(la + 2048 * at0, off), pf_frag(la + 2048 * at0 + 2048, off),
                            pf_frag(la + 2048 * at2, off), pf_frag(la + 2048 * at2 + 2048, off)};
        // PLAIN: a wavefront's rows lie in one 128-row block of scales
        const float w0 = L.ws[kSwiglu ? 0 : 2 * wr / RW][kb], w1 = kSwiglu ? L.ws[1][kb] : w0;
#pragma unroll
        for (int bt = 0; bt < BT; ++bt) {
            const i32x8 B = pf_frag(lb + 2048 * bt, off);
            const int sb = L.sb[u][16 * BT * wc + 16 * bt + n];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const f32x4 c = mfma_fp8_sb(A[t], B, f32x4{0.f, 0.f, 0.f, 0.f}, sb);
#pragma unroll
                for (int i = 0; i < 4; ++i) tot[t][bt][i] = fmaf(c[i], t < 2 ? w0 : w1, tot[t][bt][i]);
            }
        }
    };
    // the sets' loads stay in issue order (a wait counts the loads issued after the one it needs)
    Set P, Q;
    const uint32_t last = KB - 1;
    load(P, 0);
    __builtin_amdgcn_sched_barrier(0);
    load(Q, min(1u, last));
    __builtin_amdgcn_sched_barrier(0);
    stage(P, 0);
    __builtin_amdgcn_sched_barrier(0);
    load(P, min(2u, last));
    __builtin_amdgcn_sched_barrier(0);
    lds_sync();
    uint32_t kb = 0;
    for (; kb + 2 <= KB; kb += 2) {
        stage(Q, 1);
        load(Q, min(kb + 3, last));
        multiply(kb, 0);
        lds_sync();
        stage(P, 0);
        load(P, min(kb + 4, last));
        multiply(kb + 1, 1);
        lds_sync();
    }
    if (kb < KB) multiply(kb, 0);  // an odd number of k-blocks
    // epilogue: accumulator lane (g, n) of (A tile t, B tile bt) holds rows 4 g .. 4 g + 3 of A tile
    // t for activation row 16 bt + n of the wavefront's half
#pragma unroll
    for (int bt = 0; bt < BT; ++bt) {
        const uint32_t r = 16 * BT * wc + 16 * bt + n;
        if (r >= cnt) continue;
        if (kSwiglu) {
            uint16_t *yr = static_cast<uint16_t *>(a.y) + (size_t)(row0 + r) * (a.n / 2) + h0 + 32 * wr + 4 * g;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                uint16_t o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float gg = tot[t][bt][i], uu = tot[t + 2][bt][i];
                    o[i] = bf16_rne(gg / (1.0f + expf(-gg)) * uu);
                }
                *reinterpret_cast<u32x2 *>(yr + 16 * t) = u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16),
                                                                (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
            }
        } else {
            float *yr = static_cast<float *>(a.y) + (size_t)(row0 + r) * a.n + h0 + 64 * wr + 4 * g;
#pragma unroll
            for (int t = 0; t < 4; ++t) *reinterpret_cast<f32x4 *>(yr + 16 * t) = tot[t][bt];
        }
    }
}

// Grid: at least 8 x ceil(column spans x tiles / 8) workgroups, in rows of at most kPfGridX (a multiple
// of 8; the threads of a grid's row must stay below 2^32); workgroup b of all of them runs on XCD
// b % 8, and each XCD takes one contiguous range of the (tile, span) list, ordered so that what its
// workgroups share stays in its L2: by tile, an expert's weights and a tile's activation rows are read
// into one L2 only; by span, a span's weights.
constexpr uint32_t kPfGridX = 1u << 20;

template <int LAYOUT, bool PAIR>
__global__ __launch_bounds__(PAIR ? 512 : 256, PAIR ? 2 : 3) void k_pf_qgemm(const PfGemmArgs a) {
    constexpr int RW = PAIR ? 4 : 2;
    __shared__ __align__(16) PfLds<64 * RW, PAIR ? 128 : 64> L;
    const uint32_t nx = a.n / (64 * RW);
    const uint32_t total = nx * a.ntiles, wg = blockIdx.y * kPfGridX + blockIdx.x, id = (wg & 7) * a.per + (wg >> 3);
    if (id >= total) return;
    const uint32_t x = a.by_cols ? id / a.ntiles : id % nx, t = a.by_cols ? id % a.ntiles : id / nx;
    const cu32 *tw = as_const_u32(a.tiles + t);
    const uint64_t w_va = (uint64_t)tw[0] | ((uint64_t)tw[1] << 32);
    const uint64_t s_va = (uint64_t)tw[2] | ((uint64_t)tw[3] << 32);
    const uint32_t row0 = tw[4], cnt = tw[5];
    if constexpr (PAIR) {
        // tile j of a run (consecutive tiles of the same weights and contiguous rows): j even takes
        // tile j + 1 along, j odd is taken by its neighbour
        const uint32_t lane = lane_id();
        uint32_t back = 0;
        for (uint32_t b0 = 1;; b0 += 64) {
            const uint32_t d = b0 + lane;
            bool same = d <= t;
            if (same) {
                const PfTile *p = a.tiles + (t - d);
                same = p->w_va == w_va && p->s_va == s_va && p->row0 + 64 * d == row0 && p->cnt == 64;
            }
            const uint64_t miss = ~__ballot(same);
            if (miss) {
                back += (uint32_t)__builtin_ctzll(miss);
                break;
            }
            back += 64;
        }
        if (back & 1) return;
        if (cnt == 64 && t + 1 < a.ntiles) {
            const cu32 *nw = as_const_u32(a.tiles + t + 1);
            if (((uint64_t)nw[0] | ((uint64_t)nw[1] << 32)) == w_va && ((uint64_t)nw[2] | ((uint64_t)nw[3] << 32)) == s_va &&
                nw[4] == row0 + 64) {
                pf_qgemm_wg<LAYOUT, RW, 4>(a, L, w_va, s_va, x, row0, 64 + nw[5]);
                return;
            }
        }
    }
    if (!PAIR && cnt <= 32) {  // a short tile: half the activation rows
        pf_qgemm_wg<LAYOUT, 2, 1>(a, L, w_va, s_va, x, row0, cnt);
        return;
    }
    pf_qgemm_wg<LAYOUT, RW, 2>(a, L, w_va, s_va, x, row0, cnt);
}

// ------------------------------------------------------------------ router logits
// logits[r][ex] = (((-0.0 + w[ex][0] x[r][0]) + w[ex][1] x[r][1]) + ...): each product rounded to
// f32, then added in index order (no fused multiply-add), the reference's sequential f32 sum. The
// sum cannot be split along k, so the parallelism is (row, expert): one lane per expert, R rows
// per lane as R independent chains. Rows come in tiles of kPfRouterRows (the buffers hold whole
// tiles): 16, the reference engine's rows per CTA that the reference's own tests expect of
// router_rows() (aien-omega-pf/src/lib.rs:1300).
//
// A workgroup is 64 experts x 4 wavefronts of R rows each. The packed layout
// wq[g][ex][q] = w[ex][4 g + q] gives 64 experts one contiguous KiB per group of 4 columns; the
// weights come in passes of kPfRouterG groups, loaded by all four wavefronts into registers
// kPfRouterAhead passes ahead and handed over through two LDS buffers with one barrier a pass. What
// bounds it otherwise is the weight stream into the CUs (about 20 bytes a clock each): a wavefront
// that reads the weights by itself takes 4 times as many. The x values of a pass
// sit in registers, 16 columns each in every 16-lane row, and reach the product as its DPP row
// broadcast, so they cost no LDS reads and no instructions. What is left is the chain: a product and
// a sum per column, 25 us for 2048 columns with one wavefront a SIMD and one row a lane.
// Launch times against a wavefront that reads weights and x values by itself, 128 experts: 17 rows
// 27.8 -> 24.7 us, 517 rows 31.3 -> 30.5 (behind the layer's other kernels 40.6 -> 29), 1024 rows
// 49.3 -> 35.5, 2048 rows 92.5 -> 54.6, 4096 rows 96.0 -> 84.8 us.
constexpr uint32_t kPfRouterRows = 16;
constexpr uint32_t kPfRouterG = 16;
constexpr uint32_t kPfRouterAhead = 4;

struct PfRouterArgs {
    uint32_t k = 0, e = 0, rows = 0;
    const float *x = nullptr, *wq = nullptr;
    float *logits = nullptr;
};

// the value of lane N of the lane's 16-lane row
template <int N>
__device__ __forceinline__ float pf_row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xF, 0xF, true));
}
template <int... Q, class F>
__device__ __forceinline__ void pf_for_each(std::integer_sequence<int, Q...>, F f) {
    (f(std::integral_constant<int, Q>{}), ...);
}

template <int R>
__global__ __launch_bounds__(256) void k_pf_router(const PfRouterArgs a) {
#pragma clang fp contract(off)  // a multiply then an add, never one fused rounding
    constexpr uint32_t G = kPfRouterG, D = kPfRouterAhead;
    __shared__ f32x4 L[2][G][64];
    const uint32_t tid = threadIdx.x, lane = lane_id(), wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ex = blockIdx.x * 64 + lane, exl = min(ex, a.e - 1);  // lanes past the last expert load its weights
    const uint32_t r0 = (blockIdx.y * 4 + wid) * R;
    const uint32_t ng = a.k / 4, np = (ng + G - 1) / G, last = np - 1;
    struct Set {
        f32x4 w[G / 4];        // groups wid, wid + 4, ... of the pass
        float x[R][G / 4];     // columns 16 i + lane % 16 of the pass
    };
    Set S[D];
    auto load = [&](Set &s, uint32_t p) {
#pragma unroll
        for (uint32_t i = 0; i < G / 4; ++i) {  // past the last group and column: the last one again, unused
            s.w[i] = *as_global_f32x4(a.wq + ((size_t)min(G * p + wid + 4 * i, ng - 1) * a.e + exl) * 4);
#pragma unroll
            for (int j = 0; j < R; ++j)
                s.x[j][i] = *as_global_f32(a.x + (size_t)(r0 + j) * a.k + min(4 * G * p + 16 * i + (lane & 15), a.k - 1));
        }
    };
    float acc[R], xc[R][G / 4];
#pragma unroll
    for (int j = 0; j < R; ++j) acc[j] = -0.0f;
    // the pass's weights to LDS buffer b, its x values to xn
    auto stage = [&](const Set &s, uint32_t b, float (&xn)[R][G / 4]) {
#pragma unroll
        for (uint32_t i = 0; i < G / 4; ++i) {
            L[b][wid + 4 * i][lane] = s.w[i];
#pragma unroll
            for (int j = 0; j < R; ++j) xn[j][i] = s.x[j][i];
        }
    };
    auto group = [&](const f32x4 w, auto qc) {
        constexpr int q = decltype(qc)::value, c = 4 * (q & 3);
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const float x = xc[j][q / 4], p0 = pf_row_bcast<c>(x) * w.x, p1 = pf_row_bcast<c + 1>(x) * w.y;
            const float p2 = pf_row_bcast<c + 2>(x) * w.z, p3 = pf_row_bcast<c + 3>(x) * w.w;
            acc[j] = acc[j] + p0;
            acc[j] = acc[j] + p1;
            acc[j] = acc[j] + p2;
            acc[j] = acc[j] + p3;
        }
    };
    // the first n groups of the pass in buffer b; all its LDS reads go out before the first sum
    auto sums = [&](uint32_t b, uint32_t n, auto full) {
        f32x4 w[G];
#pragma unroll
        for (uint32_t q = 0; q < G; ++q) w[q] = L[b][q][lane];
        __builtin_amdgcn_sched_barrier(0);
        pf_for_each(std::make_integer_sequence<int, (int)G>{}, [&](auto q) {
            if (decltype(full)::value || q < n) group(w[q], q);
        });
    };
#pragma unroll
    for (uint32_t u = 0; u < D; ++u) load(S[u], min(u, last));
    stage(S[0], 0, xc);
    load(S[0], min(D, last));
    lds_sync();
    for (uint32_t p0 = 0; p0 < np; p0 += D) {
#pragma unroll
        for (uint32_t u = 0; u < D; ++u) {
            const uint32_t p = p0 + u;
            if (p >= np) break;  // the same for the whole workgroup
            float xn[R][G / 4];
            Set &s = S[(u + 1) % D];
            stage(s, (u + 1) & 1, xn);
            load(s, min(p + 1 + D, last));
            if (G * (p + 1) <= ng) sums(u & 1, G, std::true_type{});
            else sums(u & 1, ng - G * p, std::false_type{});
            lds_sync();
#pragma unroll
            for (int j = 0; j < R; ++j)
#pragma unroll
                for (uint32_t i = 0; i < G / 4; ++i) xc[j][i] = xn[j][i];
        }
    }
    if (ex < a.e) {
#pragma unroll
        for (int j = 0; j < R; ++j) a.logits[(size_t)(r0 + j) * a.e + ex] = acc[j];
    }
}

// ------------------------------------------------------------------ MoE combine
// out[r][c] = sum over slots in order, from +0.0, of wt[r][slot] * down[inv[r][slot]][c] (each
// product rounded, then added). Bound by the top_k down rows it reads: one thread per row and V
// columns (4 where h and the addresses allow 16-byte loads, else 1), the loads of 8 slots in flight
// before the first is summed. The slots' rows and weights are the same for a whole workgroup and
// come through scalar loads. Launch times, one column a thread and one slot in flight before: 2000
// tokens of 8 x 2048 values 31.5 -> 24.7 us (6 TB/s), 517 tokens 12.4 -> 7.7 us.
struct PfCombineArgs {
    uint32_t h = 0, top_k = 0, rows = 0;
    const float *down = nullptr;
    const uint32_t *inv = nullptr;
    const float *wt = nullptr;
    float *out = nullptr;
};

template <int V>
__global__ __launch_bounds__(256) void k_pf_combine(const PfCombineArgs a) {
#pragma clang fp contract(off)  // a multiply then an add, never one fused rounding
    const uint32_t r = blockIdx.y, c = (blockIdx.x * 256 + threadIdx.x) * V;
    if (c >= a.h) return;
    const cu32 *inv = as_const_u32(a.inv + (size_t)r * a.top_k), *wt = as_const_u32(a.wt + (size_t)r * a.top_k);
    float acc[V] = {};
    uint32_t s = 0;
    auto load = [&](uint32_t slot, float (&d)[V]) {
        const float *p = a.down + (size_t)inv[slot] * a.h + c;
        if constexpr (V == 4) {
            const f32x4 t = *as_global_f32x4(p);
            d[0] = t.x, d[1] = t.y, d[2] = t.z, d[3] = t.w;
        } else {
            d[0] = *as_global_f32(p);
        }
    };
    auto add = [&](uint32_t slot, const float (&d)[V]) {
        const float w = __uint_as_float(wt[slot]);
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] = acc[i] + w * d[i];
    };
    for (; s + 8 <= a.top_k; s += 8) {
        float d[8][V];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) load(s + j, d[j]);
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) add(s + j, d[j]);
    }
    for (; s < a.top_k; ++s) {
        float d[V];
        load(s, d);
        add(s, d);
    }
    float *o = a.out + (size_t)r * a.h + c;
    if constexpr (V == 4) *reinterpret_cast<f32x4 *>(o) = f32x4{acc[0], acc[1], acc[2], acc[3]};
    else o[0] = acc[0];
}

// ------------------------------------------------------------------ residual add + RMSNorm (extension)
// Per row: x += add (when given, in place), then out = x * scale * w with scale = (1 / sqrt(mean
// of squares + eps)) rounded to f32 and the squares summed in f64 (tensor.rs:94-110), so the
// driver's residual stays on the device between the GEMMs.
struct PfNormArgs {
    uint32_t k = 0;
    float *x = nullptr;
    const float *add = nullptr, *w = nullptr;
    float eps = 1e-6f;
    float *out = nullptr;
};

// One workgroup per row, thread t takes columns t, t + 256, ... NV > 0 (rows of up to 256 NV
// columns): all of a thread's columns are loaded before the first is used and stay in registers
// until the normalised row is written. NV 0 (longer rows) walks them one by one and reads the row
// again for the output. The sums have one order in both. Launch times, NV 0 for everything before: 517
// rows of 2048 with an addend 8.8 -> 7.0 us, 2000 rows 14.7 -> 11.6 us (5.6 TB/s).
template <int NV>
__global__ __launch_bounds__(256) void k_pf_resid_norm(const PfNormArgs a) {
#pragma clang fp contract(off)  // x + add and x * scale * w each rounded as written
    __shared__ double red[4];
    const uint32_t r = blockIdx.x, t = threadIdx.x, lane = lane_id(), wid = t >> 6;
    float *xr = a.x + (size_t)r * a.k;
    const float *ar = a.add ? a.add + (size_t)r * a.k : nullptr;
    float *orow = a.out + (size_t)r * a.k;
    float v[NV ? NV : 1], w[NV ? NV : 1], d[NV ? NV : 1];
    double ss = 0.0;
    if constexpr (NV > 0) {
#pragma unroll
        for (uint32_t i = 0; i < NV; ++i) {
            const uint32_t c = min(t + 256 * i, a.k - 1);  // lanes past the end read the last column
            v[i] = *as_global_f32(xr + c);
            w[i] = *as_global_f32(a.w + c);
            d[i] = ar ? *as_global_f32(ar + c) : 0.f;
        }
#pragma unroll
        for (uint32_t i = 0; i < NV; ++i) {
            const uint32_t c = t + 256 * i;
            if (c >= a.k) continue;
            if (ar) {
                v[i] = v[i] + d[i];
                xr[c] = v[i];
            }
            ss += (double)v[i] * (double)v[i];
        }
    } else {
        for (uint32_t c = t; c < a.k; c += 256) {
            float x = xr[c];
            if (ar) {
                x = x + ar[c];
                xr[c] = x;
            }
            ss += (double)x * (double)x;
        }
    }
    ss = wave_sum_f64(ss);
    if (lane == 0) red[wid] = ss;
    __syncthreads();
    const float scale = rms_scale((red[0] + red[1]) + (red[2] + red[3]), a.k, a.eps);
    if constexpr (NV > 0) {
#pragma unroll
        for (uint32_t i = 0; i < NV; ++i)
            if (t + 256 * i < a.k) orow[t + 256 * i] = v[i] * scale * w[i];
    } else {
        for (uint32_t c = t; c < a.k; c += 256) orow[c] = xr[c] * scale * a.w[c];
    }
}

// ------------------------------------------------------------------ host threads for per-token host work
// The MoE plan of a long prompt ranks every token on the host (MoeBatchPlan::from_logits). A few
// threads, started on first use and kept for the process, split such a loop into contiguous
// ranges; the caller takes a range too. One job at a time (the entry points hold the library
// lock). The pool is never destroyed (its threads end with the process, nothing joins them at
// exit), and a child forked from the process has none of its threads: there width() is 1 and
// the caller runs the loop alone. The fork handlers hold the pool's lock across the fork so the
// child does not inherit it taken by a worker.
class HostPool {
  public:
    static HostPool &get() {
        static HostPool *p = new HostPool();
        return *p;
    }
    uint32_t width() const { return forked_ ? 1u : (uint32_t)th_.size() + 1; }
    // fn(part) for part in 0 .. parts - 1, over the pool and the calling thread. The job lives on
    // this frame: a thread takes it under the lock and counts itself in `users`, and run() returns
    // only when every part has finished and no thread still holds the job.
    void run(uint32_t parts, const std::function<void(uint32_t)> &fn) {
        Job job{&fn, parts};
        {
            std::lock_guard<std::mutex> lk(mu_);
            cur_ = &job;
            ++gen_;
        }
        cv_.notify_all();
        work(job);
        std::unique_lock<std::mutex> lk(mu_);
        done_.wait(lk, [&] { return job.finished.load() == parts && job.users == 0; });
        cur_ = nullptr;
    }

  private:
    struct Job {
        const std::function<void(uint32_t)> *fn;
        uint32_t parts;
        std::atomic<uint32_t> next{0}, finished{0};
        uint32_t users = 0;  // guarded by mu_
    };
    HostPool() {
        const unsigned hc = std::thread::hardware_concurrency();
        const unsigned n = std::min(hc ? hc : 1u, 16u);  // a one-GPU share of the host
        pthread_atfork([] { get().mu_.lock(); }, [] { get().mu_.unlock(); },
                       [] {
                           get().forked_ = true;
                           get().mu_.unlock();
                       });
        for (unsigned i = 1; i < n; ++i) th_.emplace_back([this] { loop(); });
    }
    static void work(Job &j) {
        for (uint32_t p; (p = j.next.fetch_add(1)) < j.parts;) {
            (*j.fn)(p);
            j.finished.fetch_add(1);
        }
    }
    void loop() {
        uint64_t seen = 0;
        for (;;) {
            Job *j;
            {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [&] { return cur_ && gen_ != seen; });
                seen = gen_;
                j = cur_;
                ++j->users;
            }
            work(*j);
            {
                std::lock_guard<std::mutex> lk(mu_);
                --j->users;
            }
            done_.notify_all();
        }
    }
    std::mutex mu_;
    std::condition_variable cv_, done_;
    std::vector<std::thread> th_;
    Job *cur_ = nullptr;
    uint64_t gen_ = 0;
    bool forked_ = false;
};

// ------------------------------------------------------------------ session memory and counters
struct PfState {
    std::mutex mu;
    uint64_t chip_ns = 0, launches = 0;
    uint32_t next_index = 1;
};
PfState &pf_state() {
    static PfState s;
    return s;
}

// Times the launches of `enqueue` on the library stream; adds them to the counters.
template <class F>
int pf_timed(Family fam, uint32_t launches, uint64_t *ns, F enqueue) {
    Ctx *c = ctx(fam);
    if (!c) return OMEGA_GPU_CHIP_FAIL;
    OMEGA_HIP(fam, hipEventRecord(c->ev0, c->stream));
    OMEGA_HIP(fam, enqueue(c->stream));
    OMEGA_HIP(fam, hipEventRecord(c->ev1, c->stream));
    OMEGA_HIP(fam, hipEventSynchronize(c->ev1));
    float ms = 0.f;
    OMEGA_HIP(fam, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    const uint64_t t = (uint64_t)((double)ms * 1e6);
    if (ns) *ns = t;
    std::lock_guard<std::mutex> lk(pf_state().mu);
    pf_state().chip_ns += t;
    pf_state().launches += launches;
    return OMEGA_GPU_OK;
}

}  // namespace omega

using namespace omega;

extern "C" {

const char *omega_gpu_pf_rc_name(int rc) { return rc_name(rc); }

static int pf_alloc(size_t bytes, OmegaGpuMem *out, bool host) {
    std::lock_guard<std::recursive_mutex> lk(big_lock());
    clear_error(F_SESSION);
    if (!out || bytes == 0) {
        set_error(F_SESSION, "pf alloc: NULL out or 0 bytes");
        return OMEGA_GPU_BAD_ARGS;
    }
    memset(out, 0, sizeof(*out));
    if (!ctx(F_SESSION)) return OMEGA_GPU_CHIP_FAIL;
    void *p = nullptr, *dp = nullptr;
    if (host) {
        // host-visible, not cached by the GPU: the CPU reads and writes it in place
        OMEGA_HIP(F_SESSION, host_malloc(&p, bytes, hipHostMallocMapped | hipHostMallocCoherent));
        hipError_t e = hipHostGetDevicePointer(&dp, p, 0);
        if (e != hipSuccess) {
            (void)host_free(p);
            set_error(F_SESSION, "pf alloc host: hipHostGetDevicePointer: %s", hipGetErrorString(e));
            return OMEGA_GPU_CHIP_FAIL;
        }
        memset(p, 0, bytes);
    } else {
        OMEGA_HIP(F_SESSION, dev_malloc(&dp, bytes));
        hipError_t e = hipMemset(dp, 0, bytes);
        if (e != hipSuccess) {
            (void)dev_free(dp);
            set_error(F_SESSION, "pf alloc dev: hipMemset: %s", hipGetErrorString(e));
            return OMEGA_GPU_CHIP_FAIL;
        }
    }
    {
        std::lock_guard<std::mutex> sl(pf_state().mu);
        out->handle_index = pf_state().next_index++;
    }
    out->handle_generation = 1;
    out->kind = host ? 1u : 0u;
    out->cpu = p;
    out->va = (uint64_t)(uintptr_t)dp;
    out->size = bytes;
    return OMEGA_GPU_OK;
}

int omega_gpu_pf_alloc_dev(size_t bytes, OmegaGpuMem *out) { return pf_alloc(bytes, out, false); }
int omega_gpu_pf_alloc_host(size_t bytes, OmegaGpuMem *out) { return pf_alloc(bytes, out, true); }

void omega_gpu_pf_free(OmegaGpuMem *m) {
    std::lock_guard<std::recursive_mutex> lk(big_lock());
    if (!m || !m->va) return;
    Ctx *c = ctx(F_SESSION);
    if (c) (void)hipStreamSynchronize(c->stream);
    if (m->kind == 1) (void)host_free(m->cpu);
    else (void)dev_free((void *)(uintptr_t)m->va);
    memset(m, 0, sizeof(*m));
}

int omega_gpu_pf_copy_va(uint64_t dst_va, uint64_t src_va, size_t bytes) {
    std::lock_guard<std::recursive_mutex> lk(big_lock());
    clear_error(F_SESSION);
    if (!dst_va || !src_va || dst_va % 16 || src_va % 16 || bytes % 16) {
        set_error(F_SESSION, "pf copy: addresses and %zu bytes must be non-zero 16-byte multiples", bytes);
        return OMEGA_GPU_BAD_ARGS;
    }
    return pf_timed(F_SESSION, 1, nullptr, [&](hipStream_t st) {
        return hipMemcpyAsync((void *)(uintptr_t)dst_va, (const void *)(uintptr_t)src_va, bytes,
                              hipMemcpyDeviceToDevice, st);
    });
}

void omega_gpu_pf_stats(uint64_t *chip_ns, uint64_t *launches) {
    std::lock_guard<std::mutex> lk(pf_state().mu);
    if (chip_ns) *chip_ns = pf_state().chip_ns;
    if (launches) *launches = pf_state().launches;
}

void omega_gpu_pf_stats_reset(void) {
    std::lock_guard<std::mutex> lk(pf_state().mu);
    pf_state().chip_ns = 0;
    pf_state().launches = 0;
}

int omega_gpu_pf_quant(uint32_t k, uint32_t in_type, uint32_t rows, uint64_t x_va, uint64_t q_va, uint64_t s_va,
                       uint64_t *ns) {
    std::lock_guard<std::recursive_mutex> lk(big_lock());
    clear_error(F_SESSION);
    if (k % 128 || k < 128 || k > 32768 || in_type > 1 || !x_va || !q_va || !s_va) {
        set_error(F_SESSION, "pf quant k=%u in_type=%u refused: k a multiple of 128 in 128..=32768, "
                  "f32 (0) or bf16 (1) input, non-NULL addresses", k, in_type);
        return OMEGA_GPU_BAD_ARGS;
    }
    if (ns) *ns = 0;
    if (rows == 0) return OMEGA_GPU_OK;
    PfQuantArgs a;
    a.k = k;
    a.rows = rows;
    a.x = (const void *)(uintptr_t)x_va;
    a.q = (uint8_t *)(uintptr_t)q_va;
    a.s = (float *)(uintptr_t)s_va;
    const uint64_t waves = (uint64_t)rows * (k / 128);
    if ((waves + 3) / 4 > 0x7fffffffull) {
        set_error(F_SESSION, "pf quant: %u rows of %u too large", rows, k);
        return OMEGA_GPU_TOO_LARGE;
    }
    return pf_timed(F_SESSION, 1, ns, [&](hipStream_t st) {
        const dim3 wg(256), blocks4((uint32_t)((waves + 3) / 4)), blocks16((uint32_t)((waves + 15) / 16));
        if (x_va % 16 || q_va % 8) {
            if (in_type) OMEGA_LAUNCH((k_pf_quant<true, 2>), blocks4, wg, 0, st, a);
            else OMEGA_LAUNCH((k_pf_quant<false, 2>), blocks4, wg, 0, st, a);
        } else if (in_type) OMEGA_LAUNCH((k_pf_quant<true, 8>), blocks16, wg, 0, st, a);
        else OMEGA_LAUNCH((k_pf_quant<false, 8>), blocks16, wg, 0, st, a);
        return hipGetLastError();
    });
}

uint32_t omega_gpu_pf_qgemm_bm(void) { return kPfBm; }

uint32_t omega_gpu_pf_qgemm_tiles_va(uint32_t experts, const uint64_t *w_va, const uint64_t *s_va,
                                     const uint32_t *counts, void *tab, uint32_t max) {
    if (!w_va || !s_va || !counts || !tab || experts == 0) return 0;
    PfTile *t = static_cast<PfTile *>(tab);
    uint32_t n = 0, row = 0;
    for (uint32_t e = 0; e < experts; ++e) {
        for (uint32_t r = 0; r < counts[e];) {
            const uint32_t c = std::min(counts[e] - r, kPfBm);
            if (n >= max) return 0;
            t[n].w_va = w_va[e];
            t[n].s_va = s_va[e];
            t[n].row0 = row + r;
            t[n].cnt = c;
            t[n].pad = 0;
            ++n;
            r += c;
        }
        row += counts[e];
    }
    return n;
}

int omega_gpu_pf_moe_plan(uint32_t tokens, uint32_t experts, uint32_t top_k, const float *logits, uint32_t *topk_ids,
                          float *topk_weights, uint32_t *counts, uint32_t *grouped_token,
                          uint32_t *assignment_to_grouped, uint32_t *grouped_to_assignment) {
    std::lock_guard<std::recursive_mutex> lk(big_lock());  // the session's error slot
    clear_error(F_SESSION);
    if (experts == 0 || experts > 65536 || top_k == 0 || top_k > experts || top_k > 64 ||
        (uint64_t)tokens * top_k > 0xffffffffull || !logits || !topk_ids || !topk_weights || !counts ||
        !grouped_token || !assignment_to_grouped) {
        set_error(F_SESSION, "pf moe plan: experts=%u, top_k=%u (1..=min(experts, 64)), tokens=%u, non-NULL "
                  "buffers", experts, top_k, tokens);
        return OMEGA_GPU_BAD_ARGS;
    }
    // the total order of f32 (f32::total_cmp) as a signed key: negative values count down
    auto key = [](float v) {
        const int32_t b = (int32_t)__builtin_bit_cast(uint32_t, v);
        return b ^ (int32_t)((uint32_t)(b >> 31) >> 1);
    };
    // tokens t0 .. t1 - 1: top_k by (key descending, id ascending), insertion into a sorted list
    // of top_k; returns the first non-finite logit's index (token * experts + expert) or ~0
    auto rank = [&](uint32_t t0, uint32_t t1) -> uint64_t {
        for (uint32_t t = t0; t < t1; ++t) {
            const float *row = logits + (size_t)t * experts;
            uint32_t sel[64];
            int32_t sk[64];
            uint32_t n = 0;
            for (uint32_t e = 0; e < experts; ++e) {
                if (!std::isfinite(row[e])) return (uint64_t)t * experts + e;
                const int32_t k = key(row[e]);
                if (n == top_k && k <= sk[n - 1]) continue;  // a tie goes to the lower id, already held
                uint32_t i = n < top_k ? n++ : n - 1;
                while (i > 0 && sk[i - 1] < k) {
                    sk[i] = sk[i - 1];
                    sel[i] = sel[i - 1];
                    --i;
                }
                sk[i] = k;
                sel[i] = e;
            }
            const float mx = row[sel[0]];
            float prob[64], sum = 0.0f;
            for (uint32_t j = 0; j < top_k; ++j) {
                prob[j] = std::exp(row[sel[j]] - mx);
                sum += prob[j];
            }
            for (uint32_t j = 0; j < top_k; ++j) {
                topk_ids[(size_t)t * top_k + j] = sel[j];
                topk_weights[(size_t)t * top_k + j] = prob[j] / sum;
            }
        }
        return ~0ull;
    };
    // long prompts: contiguous token ranges over the host threads (the results do not depend on
    // the split); the first non-finite logit in row order is the one reported
    constexpr uint32_t kTokensPerPart = 64;
    uint64_t bad = ~0ull;
    HostPool &pool = HostPool::get();
    if (tokens >= 4 * kTokensPerPart && pool.width() > 1) {
        const uint32_t parts = std::min(pool.width() * 4, (tokens + kTokensPerPart - 1) / kTokensPerPart);
        const uint32_t per = (tokens + parts - 1) / parts;
        std::vector<uint64_t> first(parts, ~0ull);
        pool.run(parts, [&](uint32_t p) {
            const uint32_t t0 = std::min(tokens, p * per), t1 = std::min(tokens, t0 + per);
            first[p] = rank(t0, t1);
        });
        for (uint64_t f : first) bad = std::min(bad, f);
    } else {
        bad = rank(0, tokens);
    }
    if (bad != ~0ull) {
        set_error(F_SESSION, "pf moe plan: logit of token %u, expert %u is not finite", (uint32_t)(bad / experts),
                  (uint32_t)(bad % experts));
        return OMEGA_GPU_BAD_ARGS;
    }
    for (uint32_t e = 0; e < experts; ++e) counts[e] = 0;
    for (uint64_t a = 0; a < (uint64_t)tokens * top_k; ++a) ++counts[topk_ids[a]];
    // stable counting sort of the assignments by expert
    std::vector<uint32_t> cursor(experts);
    uint32_t acc = 0;
    for (uint32_t e = 0; e < experts; ++e) {
        cursor[e] = acc;
        acc += counts[e];
    }
    const uint64_t assignments = (uint64_t)tokens * top_k;
    for (uint64_t a = 0; a < assignments; ++a) {
        const uint32_t g = cursor[topk_ids[a]]++;
        assignment_to_grouped[a] = g;
        grouped_token[g] = (uint32_t)(a / top_k);
        if (grouped_to_assignment) grouped_to_assignment[g] = (uint32_t)a;
    }
    return OMEGA_GPU_OK;
}

int omega_gpu_pf_qgemm(uint32_t n, uint32_t k, uint32_t layout, uint64_t tiles_va, uint32_t ntiles,
                       uint64_t rowidx_va, uint64_t xq_va, uint64_t xs_va, uint64_t y_va, uint64_t *ns) {
    std::lock_guard<std::recursive_mutex> lk(big_lock());
    clear_error(F_SESSION);
    const uint64_t row_bytes = layout == kPfLayoutSwiglu ? n : 4ull * n;
    if (k % 128 || k < 128 || k > 32768) {
        set_error(F_SESSION, "pf qgemm k=%u refused: multiple of 128, 128 <= k <= 32768", k);
        return OMEGA_GPU_BAD_ARGS;
    }
    if (n == 0 || n % 128 || row_bytes * kPfBm >= (1ull << 23) || (layout != kPfLayoutPlain && layout != kPfLayoutSwiglu)) {
        set_error(F_SESSION, "pf qgemm n=%u layout=%u refused: positive multiple of 128, row bytes x 64 < 2^23, "
                  "layout PLAIN (0) or SWIGLU_NAT (2)", n, layout);
        return OMEGA_GPU_BAD_ARGS;
    }
    if (layout == kPfLayoutSwiglu && n % 256) {
        set_error(F_SESSION, "pf qgemm SwiGLU n=%u refused: multiple of 256", n);
        return OMEGA_GPU_BAD_ARGS;
    }
    if (ntiles > 65535) {
        set_error(F_SESSION, "pf qgemm %u tiles > 65535", ntiles);
        return OMEGA_GPU_TOO_LARGE;
    }
    if (!tiles_va || !xq_va || !xs_va || !y_va) {
        set_error(F_SESSION, "pf qgemm: null address");
        return OMEGA_GPU_BAD_ARGS;
    }
    if (ns) *ns = 0;
    if (ntiles == 0) return OMEGA_GPU_OK;
    PfGemmArgs a;
    a.n = n;
    a.k = k;
    a.layout = layout;
    a.tiles = reinterpret_cast<const PfTile *>(tiles_va);
    a.rowidx = reinterpret_cast<const uint32_t *>(rowidx_va);
    a.xq = reinterpret_cast<const uint8_t *>(xq_va);
    a.xs = reinterpret_cast<const float *>(xs_va);
    a.y = reinterpret_cast<void *>(y_va);
    a.ntiles = ntiles;
    // fewer activation rows than weight rows of one expert: an XCD that takes column spans reads
    // less (its spans' weights and the rows) than one that takes tiles (q|k|v at 512 rows 24.2 us
    // against 25.8; 4096 rows by tile: 106 against 91 us; experts of 2000 tokens by tile 151
    // against 156 us)
    a.by_cols = 64ull * ntiles < n;
    // the paired form halves the weight reads of a run of tiles but leaves one workgroup a CU, so it
    // takes work for several rounds of 256 (o of 2048 rows, 8192 span-tile-blocks: 50 us against 43;
    // of 2500 rows 52 either way, of 4096 rows 57 against 73; down of 1250 tokens 81 against 85,
    // of 3000 tokens 157 against 170). gate|up gains nothing (2000 tokens 172 against 151 us).
    const bool pair = layout == kPfLayoutPlain && !a.by_cols && n % 256 == 0 &&
                      (uint64_t)(n / 256) * ntiles * (k / 128) >= 10240;
    const uint32_t wgs = (n / (pair ? 256 : 128) * ntiles + 7) / 8 * 8;  // at most 1022 x 65535
    const uint32_t gx = std::min(wgs, kPfGridX), gy = (wgs + gx - 1) / gx;
    a.per = gx * gy / 8;
    return pf_timed(F_SESSION, 1, ns, [&](hipStream_t st) {
        const dim3 grid(gx, gy), block(pair ? 512 : 256);
        if (layout == kPfLayoutSwiglu) OMEGA_LAUNCH((k_pf_qgemm<kPfLayoutSwiglu, false>), grid, block, 0, st, a);
        else if (pair) OMEGA_LAUNCH((k_pf_qgemm<kPfLayoutPlain, true>), grid, block, 0, st, a);
        else OMEGA_LAUNCH((k_pf_qgemm<kPfLayoutPlain, false>), grid, block, 0, st, a);
        return hipGetLastError();
    });
}

uint32_t omega_gpu_pf_router_rows(void) { return kPfRouterRows; }

void omega_gpu_pf_router_pack(uint32_t e, uint32_t k, const float *w, float *wq) {
    if (!w || !wq || k % 4) return;
    for (uint32_t g = 0; g < k / 4; ++g)
        for (uint32_t ex = 0; ex < e; ++ex)
            for (uint32_t q = 0; q < 4; ++q) wq[((size_t)g * e + ex) * 4 + q] = w[(size_t)ex * k + 4 * g + q];
    for (uint32_t i = 0; i < 4 * e; ++i) wq[(size_t)(k / 4) * e * 4 + i] = 0.f;  // the pad group
}

int omega_gpu_pf_router_logits(uint32_t k, uint32_t e, uint32_t rows, uint64_t x_va, uint64_t wq_va,
                               uint64_t logits_va, uint64_t *ns) {
    std::lock_guard<std::recursive_mutex> lk(big_lock());
    clear_error(F_SESSION);
    if (!x_va || !wq_va || !logits_va || k == 0 || k % 4 || e == 0 || e > 1024 || x_va % 16 || wq_va % 16) {
        set_error(F_SESSION, "pf router logits: k=%u (a multiple of 4), e=%u (1..=1024), 16-byte aligned "
                  "non-NULL x and packed weights", k, e);
        return OMEGA_GPU_BAD_ARGS;
    }
    if (ns) *ns = 0;
    if (rows == 0) return OMEGA_GPU_OK;
    PfRouterArgs a;
    a.k = k;
    a.e = e;
    a.rows = (rows + kPfRouterRows - 1) / kPfRouterRows * kPfRouterRows;  // whole tiles
    a.x = reinterpret_cast<const float *>(x_va);
    a.wq = reinterpret_cast<const float *>(wq_va);
    a.logits = reinterpret_cast<float *>(logits_va);
    // R rows per lane when that still gives every CU a workgroup, else fewer: a wavefront's four
    // chains of 2048 columns take 55 us, its one chain 25 us
    const uint32_t gx = (e + 63) / 64;
    const uint64_t wgs = (uint64_t)gx * (a.rows / 4);
    const int r = wgs >= 4 * 256ull ? 4 : wgs >= 2 * 256ull ? 2 : 1;
    const uint32_t max_rows = 32768 * (uint32_t)r;  // grid.y stays within 32768 row groups
    const uint32_t launches = (a.rows + max_rows - 1) / max_rows;
    return pf_timed(F_SESSION, launches, ns, [&](hipStream_t st) {
        for (uint32_t r0 = 0; r0 < a.rows; r0 += max_rows) {
            PfRouterArgs b = a;
            b.rows = a.rows - r0 < max_rows ? a.rows - r0 : max_rows;
            b.x = a.x + (size_t)r0 * k;
            b.logits = a.logits + (size_t)r0 * e;
            const dim3 grid(gx, b.rows / (4 * r));
            if (r == 4)
                OMEGA_LAUNCH(k_pf_router<4>, grid, dim3(256), 0, st, b);
            else if (r == 2)
                OMEGA_LAUNCH(k_pf_router<2>, grid, dim3(256), 0, st, b);
            else
                OMEGA_LAUNCH(k_pf_router<1>, grid, dim3(256), 0, st, b);
            const hipError_t err = hipGetLastError();
            if (err != hipSuccess) return err;
        }
        return hipSuccess;
    });
}

int omega_gpu_pf_moe_combine(uint32_t h, uint32_t top_k, uint32_t rows, uint64_t down_va, uint64_t inv_va,
                             uint64_t wt_va, uint64_t out_va, uint64_t *ns) {
    std::lock_guard<std::recursive_mutex> lk(big_lock());
    clear_error(F_SESSION);
    if (!down_va || !inv_va || !wt_va || !out_va || h == 0 || top_k == 0 || top_k > 64 || rows > 65535) {
        set_error(F_SESSION, "pf moe combine: null address, h=%u, top_k=%u (1..=64) or %u rows (<= 65535)", h,
                  top_k, rows);
        return OMEGA_GPU_BAD_ARGS;
    }
    if (ns) *ns = 0;
    if (rows == 0) return OMEGA_GPU_OK;
    PfCombineArgs a;
    a.h = h;
    a.top_k = top_k;
    a.rows = rows;
    a.down = reinterpret_cast<const float *>(down_va);
    a.inv = reinterpret_cast<const uint32_t *>(inv_va);
    a.wt = reinterpret_cast<const float *>(wt_va);
    a.out = reinterpret_cast<float *>(out_va);
    return pf_timed(F_SESSION, 1, ns, [&](hipStream_t st) {
        if (h % 4 == 0 && down_va % 16 == 0 && out_va % 16 == 0)
            OMEGA_LAUNCH(k_pf_combine<4>, dim3((h + 1023) / 1024, rows), dim3(256), 0, st, a);
        else
            OMEGA_LAUNCH(k_pf_combine<1>, dim3((h + 255) / 256, rows), dim3(256), 0, st, a);
        return hipGetLastError();
    });
}

int omega_gpu_pf_residual_norm(uint32_t k, uint32_t rows, uint64_t x_va, uint64_t add_va, uint64_t w_va, float eps,
                               uint64_t out_va, uint64_t *ns) {
    std::lock_guard<std::recursive_mutex> lk(big_lock());
    clear_error(F_SESSION);
    if (k == 0 || k > 65536 || !x_va || !w_va || !out_va || rows > 0x7fffffffu) {
        set_error(F_SESSION, "pf residual norm: k=%u (1..=65536), non-NULL x, weights and out", k);
        return OMEGA_GPU_BAD_ARGS;
    }
    if (ns) *ns = 0;
    if (rows == 0) return OMEGA_GPU_OK;
    PfNormArgs a;
    a.k = k;
    a.x = reinterpret_cast<float *>(x_va);
    a.add = reinterpret_cast<const float *>(add_va);
    a.w = reinterpret_cast<const float *>(w_va);
    a.eps = eps;
    a.out = reinterpret_cast<float *>(out_va);
    return pf_timed(F_SESSION, 1, ns, [&](hipStream_t st) {
        if (k <= 256 * 8) OMEGA_LAUNCH(k_pf_resid_norm<8>, dim3(rows), dim3(256), 0, st, a);
        else if (k <= 256 * 16) OMEGA_LAUNCH(k_pf_resid_norm<16>, dim3(rows), dim3(256), 0, st, a);
        else OMEGA_LAUNCH(k_pf_resid_norm<0>, dim3(rows), dim3(256), 0, st, a);
        return hipGetLastError();
    });
}

}  // extern "C"
