// Register-resident persistent GRU recurrences for hidden sizes past 256 (to
// 768): four batch rows and 32 hidden units per workgroup, the products of a
// step on the matrix cores (v_mfma_f32_4x4x1_16b_f32).
//
// Workgroup (g, s) owns units [32 s, 32 s + 32) of batch rows [4 g, 4 g + 4);
// the S = ceil(H / 32) workgroups of a group exchange one set of words per
// step (rec_common.h).  Its share of W_hh, 32 x 3H values, lives in VGPRs for
// the whole sequence: 96 per lane up to H = 512, 144 at H = 768 with eight
// wavefronts.  32 units rather than 64, because 64 x 3H values would be 288
// VGPRs per lane at H = 768; four rows, because the 4x4x1 MFMA multiplies four
// and a group of S workgroups then fits the 32 CUs of an XCD for every H.
//
// What bounds a step: the MFMAs (4 x 32 x 3H multiply-adds per workgroup, one
// MFMA of 256 per ~4.1 ns and SIMD: 0.79 us at H = 512, 1.18 us at 768) and
// the chain around them (exchange, reduction, gate math, two barriers).
// Measured on MI355X, per launch, against the LDS-tiled kernels
// (gru_rec_tiled.hip), which hold W_hh in LDS and gather whole rows: B = 64,
// T = 256, H = 512 forward 1448 -> 438 us (1.71 us per step), backward 2688 ->
// 603 us (2.35 us per step); B = 32, T = 256, H = 768 forward 2905 -> 575 us.
#include "rec_common.h"

#include <algorithm>

namespace rka {
namespace {

using rec::NTH;
using rec::NW;

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int WU = 32;  // units per workgroup
constexpr int WR = 4;   // batch rows per workgroup

struct WideParams {
    int B, T, H;
    int G, S;            // groups of four rows, slices of 32 units
    int t_begin, t_end;  // backward: time range processed
    unsigned long long* xcc_words;  // start-up XCD check (nullable)
    unsigned xcc_tag;
    unsigned tag_base;                // added to every step tag
    int spin_limit;                   // poll rounds before a wait gives up
    unsigned long long* abort_count;  // per-device count of aborted launches
    int stall_block;                  // test failure injection (rec::Args::stall_block)
};

// (x of lanes 0-31 + x of lanes 32-63, likewise y): the lower half of the
// wavefront returns x's sum, the upper half y's.
__device__ __forceinline__ float half_sums(float x, float y) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

// ------------------------------------------------------------- forward ---
// Lane l = 32 hf + ul of wavefront w holds W_hh of unit 32 s + ul (MFMA A row
// ul % 4 of block l / 4) at the KP k = (2 w + hf) KP + i of every gate, so one
// MFMA per gate and i multiplies 32 units by two k (one per half) for the
// four rows (B column l % 4, read from LDS).  The two halves' sums are added
// with permlane swaps, the eight wavefronts' meet in LDS, and the owner lane of
// (row, unit) (wavefronts 0 and 1) adds them in a fixed tree, applies the gate
// math and publishes h_t.  Every wavefront polls the h words of its own 2 KP k
// only.  KP = ceil(H / 16) rounded up to a multiple of 8.
template <int KP>
__global__ __launch_bounds__(NTH) void gru_fwd_wide_kernel(
    const float* __restrict__ gx, const float* __restrict__ h0, const float* __restrict__ w_hh,
    const float* __restrict__ b_hh, float* __restrict__ y, float* __restrict__ hn, float* __restrict__ reserve,
    unsigned long long* __restrict__ exch, int* __restrict__ abort_flag, WideParams p) {
    static_assert(KP % 8 == 0, "whole poll registers");
    constexpr int NPR = 8 * KP / 64;   // polled words per lane: 2 KP k of four rows
    constexpr int HRS = 2 * KP + 4;    // LDS row of a wavefront's h values
    // [parity][wave][gate][row][unit]; the same memory holds W_hh's chunks
    // before the loop
    constexpr int kPart = 2 * NW * 3 * WR * WU, kChunk = 16 * (16 * KP + 4);
    __shared__ __attribute__((aligned(16))) float shared0[kPart > kChunk ? kPart : kChunk];
    float (&part)[2][NW][3][WR][WU] = *reinterpret_cast<float (*)[2][NW][3][WR][WU]>(shared0);
    __shared__ __attribute__((aligned(16))) float hrem[NW][WR][HRS];
    __shared__ int s_abort;
    __shared__ int s_local;

    const int B = p.B, T = p.T, H = p.H;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const rec::GroupCoords gc = rec::group_coords(p.S);
    if (gc.g >= p.G) return;  // padding workgroup of a grid rounded up to whole XCDs
    const int s = gc.s;
    const int row0 = gc.g * WR;
    const int hf = lane >> 5, ul = lane & 31, lrow = lane & 3;
    const int u = s * WU + ul;  // the lane's unit, as A row and as owner
    const int k0 = (2 * wave + hf) * KP;

    // W_hh in chunks of one gate's 16 units (half of the slice) and every k,
    // read in whole rows and handed out through LDS: a lane's KP values lie in
    // one row, so its own loads would fetch 64 rows' lines per instruction,
    // each several times (a launch of one step: 23.7 -> 20.8 us at H = 768)
    float wa[3][KP];
    {
        constexpr int NV = KP / 8;  // float4 of a chunk per thread
        constexpr int KT = 16 * KP;
        const bool vec = (H & 3) == 0 && (reinterpret_cast<uintptr_t>(w_hh) & 15u) == 0;
        float4 r[2][NV];
        auto load = [&](int c, float4 (&d)[NV]) {  // chunk c: gate c / 2, units 16 (c % 2) ..
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int x = (int)threadIdx.x + NTH * v;
                const int un = WU * s + 16 * (c % 2) + x / (KT / 4), k = 4 * (x % (KT / 4));
                const float* src = w_hh + ((size_t)(c / 2) * H + un) * H + k;
                if (vec) {
                    const bool in = un < H && k < H;
                    const float4 t = *reinterpret_cast<const float4*>(in ? src : w_hh);
                    d[v] = make_float4(in ? t.x : 0.f, in ? t.y : 0.f, in ? t.z : 0.f, in ? t.w : 0.f);
                } else {
                    float e[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const bool in = un < H && k + q < H;
                        const float t = *(in ? src + q : w_hh);
                        e[q] = in ? t : 0.f;
                    }
                    d[v] = make_float4(e[0], e[1], e[2], e[3]);
                }
            }
        };
        float (&chunk)[16][KT + 4] = *reinterpret_cast<float (*)[16][KT + 4]>(shared0);
        load(0, r[0]);
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            if (c + 1 < 6) load(c + 1, r[(c + 1) & 1]);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const int x = (int)threadIdx.x + NTH * v;
                *reinterpret_cast<float4*>(&chunk[x / (KT / 4)][4 * (x % (KT / 4))]) = r[c & 1][v];
            }
            __syncthreads();
            const bool mine = ul / 16 == c % 2;
#pragma unroll
            for (int i = 0; i < KP; i += 4) {
                const float4 v = *reinterpret_cast<const float4*>(&chunk[ul % 16][k0 + i]);
                float* d = &wa[c / 2][i];
                const bool keep = c % 2 == 1 && !mine;
                d[0] = keep ? d[0] : v.x;
                d[1] = keep ? d[1] : v.y;
                d[2] = keep ? d[2] : v.z;
                d[3] = keep ? d[3] : v.w;
            }
            __syncthreads();
        }
    }

    // owner lane of (row, unit): wavefront 0 rows 0 and 1, wavefront 1 rows 2 and 3
    const int orl = 2 * (wave & 1) + hf;
    const int orow = row0 + orl;
    const bool owner = wave < 2 && u < H && orow < B;
    float h_prev = 0.f, bias_r = 0.f, bias_z = 0.f, bias_n = 0.f;
    float gxs[2][3];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int c = 0; c < 3; ++c) gxs[e][c] = 0.f;
    const float* gx_row = gx + (size_t)orow * T * 3 * H + u;
    auto load_gx = [&](float (&d)[3], int t) {
        const float* gp = gx_row + (unsigned)t * (unsigned)(3 * H);  // 32-bit: B T H < 2^29
        d[0] = gp[0];
        d[1] = gp[H];
        d[2] = gp[2 * H];
    };
    if (owner) {
        h_prev = h0[(size_t)orow * H + u];
        bias_r = b_hh[u];
        bias_z = b_hh[H + u];
        bias_n = b_hh[2 * H + u];
        load_gx(gxs[0], 0);
    }
    if (threadIdx.x == 0) s_abort = 0;
    const rec::WaitCtl wc{abort_flag, p.abort_count, p.spin_limit};
    const bool xlocal = rec::group_on_one_xcd(p.xcc_words, gc.first, gc.stride, p.S, p.xcc_tag, wc, &s_local);

    // Polled word e = 64 v + lane of the wavefront: row e / 2KP, k = 2 KP w +
    // e % 2KP.  A row past B reads the group's first row, a k past H the last
    // unit's word; neither is waited for.
    unsigned poff[NPR];
    bool pval[NPR];
#pragma unroll
    for (int v = 0; v < NPR; ++v) {
        const int e = 64 * v + lane;
        const int r = e / (2 * KP), k = 2 * KP * wave + e % (2 * KP);
        const bool rv = row0 + r < B;
        pval[v] = rv && k < H;
        poff[v] = (unsigned)(rv ? row0 + r : row0) * (unsigned)H + (unsigned)(k < H ? k : H - 1);
    }

    const int pub_flip = (int)blockIdx.x == p.stall_block ? 1 : 0;
    const unsigned slot_words = (unsigned)B * (unsigned)H, my_word = (unsigned)orow * (unsigned)H + (unsigned)u;
    const unsigned pub_off[2] = {(unsigned)pub_flip * slot_words + my_word,
                                 (unsigned)(1 - pub_flip) * slot_words + my_word};
    float o_h = 0.f, o_r = 0.f, o_z = 0.f, o_n = 0.f, o_a = 0.f;
    float* y_row = y + (size_t)orow * T * H + u;
    float* res_row = reserve ? reserve + (size_t)orow * T * 4 * H + 4 * u : nullptr;
    auto store_outputs = [&](int t) {
        y_row[(unsigned)t * (unsigned)H] = o_h;
        if (reserve) *reinterpret_cast<float4*>(res_row + 4 * ((unsigned)t * (unsigned)H)) = make_float4(o_r, o_z, o_n, o_a);
    };

    unsigned long long first_read[NPR];
#pragma unroll
    for (int v = 0; v < NPR; ++v) first_read[v] = 0;

    auto step = [&](int t, const float (&cur)[3], float (&nxt)[3]) -> bool {
        float hx[NPR];
        if (t == 0) {
#pragma unroll
            for (int v = 0; v < NPR; ++v) hx[v] = pval[v] ? h0[poff[v]] : 0.f;
        } else {
            const unsigned long long* src = exch + (size_t)((t - 1) & 1) * slot_words;
            const unsigned long long* pp[NPR];
#pragma unroll
            for (int v = 0; v < NPR; ++v) pp[v] = src + poff[v];
            bool ok = true;
            rec::wait_words<NPR, true>(pp, pval, first_read, p.tag_base + (unsigned)t, wc, ok);
#pragma unroll
            for (int v = 0; v < NPR; ++v) hx[v] = pval[v] ? __uint_as_float((unsigned)first_read[v]) : 0.f;
            if (!ok) s_abort = 1;
        }
#pragma unroll
        for (int v = 0; v < NPR; ++v) {
            const int e = 64 * v + lane;
            hrem[wave][e / (2 * KP)][e % (2 * KP)] = hx[v];
        }
        __builtin_amdgcn_wave_barrier();
        if (owner) {
            if (t > 0) store_outputs(t - 1);
            if (t + 1 < T) load_gx(nxt, t + 1);
        }
        f4 acc[3];
#pragma unroll
        for (int g = 0; g < 3; ++g) acc[g] = f4{0.f, 0.f, 0.f, 0.f};
        const float* hb = &hrem[wave][lrow][hf * KP];
#pragma unroll
        for (int i = 0; i < KP; i += 4) {
            const float4 b = *reinterpret_cast<const float4*>(hb + i);
            const float bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int g = 0; g < 3; ++g)
                    acc[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(wa[g][i + c], bv[c], acc[g], 0, 0, 0);
        }
        // lane l holds units 4 (ul / 4) + 0..3 of row l % 4 (its half's k):
        // the lower half writes all four r and n's first two, the upper half
        // z and n's last two
        {
            float (&pw)[3][WR][WU] = part[t & 1][wave];
            const int ub = ul & ~3;
            const float4 rz = make_float4(half_sums(acc[0][0], acc[1][0]), half_sums(acc[0][1], acc[1][1]),
                                          half_sums(acc[0][2], acc[1][2]), half_sums(acc[0][3], acc[1][3]));
            *reinterpret_cast<float4*>(&pw[hf][lrow][ub]) = rz;
            const float2 nn = make_float2(half_sums(acc[2][0], acc[2][2]), half_sums(acc[2][1], acc[2][3]));
            *reinterpret_cast<float2*>(&pw[2][lrow][ub + 2 * hf]) = nn;
        }
        __syncthreads();
        const bool abort_now = s_abort != 0;
        if (owner) {
            float pq[3][NW];
#pragma unroll
            for (int g = 0; g < 3; ++g)
#pragma unroll
                for (int q = 0; q < NW; ++q) pq[g][q] = part[t & 1][q][g][orl][ul];
            __builtin_amdgcn_sched_barrier(0);
            auto total = [&](int g) { return rec::tree8([&](int q) { return pq[g][q]; }); };
            const float sr = bias_r + total(0);
            const float sz = bias_z + total(1);
            const float sn = bias_n + total(2);
            const float r = rec::sigmoid_f(cur[0] + sr);
            const float z = rec::sigmoid_f(cur[1] + sz);
            const float n = rec::tanh_f(cur[2] + r * sn);
            const float h = n + z * (h_prev - n);
            unsigned off = pub_off[t & 1];
            asm volatile("" : "+v"(off));
            rec::publish_word(exch + off, rec::pack_word(h, p.tag_base + (unsigned)(t + 1)), xlocal);
            o_h = h;
            o_r = r;
            o_z = z;
            o_n = n;
            o_a = sn;
            h_prev = h;
        }
        // keeps the other wavefronts from polling before this workgroup's own
        // words are out (an early poll only costs a second round trip), and
        // s_abort from being set for step t + 1 before every wavefront has
        // read it
        __syncthreads();
        if (t + 1 < T) {
            const unsigned long long* src = exch + (size_t)(t & 1) * slot_words;
#pragma unroll
            for (int v = 0; v < NPR; ++v) first_read[v] = rec::load_word(src + poff[v]);
        }
        return !abort_now;
    };
    // step t stores the outputs of step t - 1: after a step that aborts,
    // rows t_stop .. T-1 were not stored
    int t_stop = T;
    for (int t = 0; t < T; t += 2) {
        if (!step(t, gxs[0], gxs[1])) {
            t_stop = t;
            break;
        }
        if (t + 1 < T && !step(t + 1, gxs[1], gxs[0])) {
            t_stop = t + 1;
            break;
        }
    }
    const bool aborted = t_stop < T;
    if (owner) {
        if (!aborted) {
            store_outputs(T - 1);
        } else {
            o_h = o_r = o_z = o_n = o_a = __builtin_nanf("");
            for (int t = t_stop; t < T; ++t) store_outputs(t);
        }
        hn[(unsigned)(orow * H + u)] = aborted ? __builtin_nanf("") : h_prev;
    }
}

// ------------------------------------------------------------ backward ---
// dh_{t-1} = g z + G_h,t W_hh, with the contraction split over the workgroups
// by its rows: workgroup s multiplies its own 96 gate gradients (three gates
// of its 32 units, four batch rows) by W_hh[those 96 rows][every unit] and
// sends each workgroup c of the group the partial sums of c's 32 units, which
// c adds over the S senders in a fixed order.  A workgroup thus receives
// S x 128 words per step (16 KB at H = 512); exchanging the gate gradients
// themselves, as the kernels for H <= 256 do, would be three times that.
// Wavefront w computes tiles (32 units) w, w + 8, ..: lane l = 32 hf + ul holds
// W_hh[own row 48 hf + i][unit ul of the tile], i < 48, so one MFMA multiplies
// 32 units by two gate gradients for the four rows, and no sum crosses a
// wavefront before it is published.  IT = tiles per wavefront = ceil(S / 8).
template <int IT>
__global__ __launch_bounds__(NTH) void gru_bwd_wide_kernel(
    const float* __restrict__ dy, const float* __restrict__ dhn, const float* __restrict__ reserve,
    const float* __restrict__ h0, const float* __restrict__ y, const float* __restrict__ w_hh,
    float* __restrict__ gout, float* __restrict__ dh0, unsigned long long* __restrict__ exch,
    int* __restrict__ abort_flag, WideParams p) {
    constexpr int NPI = 2 * IT;      // senders polled per lane: ceil(S / 4) at most
    constexpr int GJ = 3 * WU;       // own gate gradients per row
    constexpr int GS = GJ + 4;       // LDS row of them
    constexpr int JH = GJ / 2;       // per wavefront half
    __shared__ __attribute__((aligned(16))) float gl[WR][GS];
    __shared__ float psum[2][4][WR * WU];  // [parity][sender class][row, unit]
    __shared__ int s_abort;
    __shared__ int s_local;

    const int B = p.B, T = p.T, H = p.H, S = p.S;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const rec::GroupCoords gc = rec::group_coords(S);
    if (gc.g >= p.G) return;  // padding workgroup of a grid rounded up to whole XCDs
    const int s = gc.s;
    const int row0 = gc.g * WR;
    const int hf = lane >> 5, ul = lane & 31, lrow = lane & 3;
    const int i0 = T - p.t_end, i1 = T - p.t_begin;  // steps i0 .. i1-1 (t = T-1-i)

    float wl[IT][JH];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int uc = WU * (wave + NW * it) + ul;
#pragma unroll
        for (int i = 0; i < JH; ++i) {
            const int jj = JH * hf + i;
            const int m = WU * s + (jj & 31);
            wl[it][i] = m < H && uc < H ? w_hh[((size_t)(jj >> 5) * H + m) * H + uc] : 0.f;
        }
    }

    // owner lane of (row, unit): wavefront 0 rows 0 and 1, wavefront 1 rows 2 and 3
    const int orl = 2 * (wave & 1) + hf;
    const int orow = row0 + orl;
    const int u = s * WU + ul;
    const bool owner = wave < 2 && u < H && orow < B;
    float dh = 0.f, ddirect = 0.f;
    float o_dan = 0.f, o_drh = 0.f, o_dzh = 0.f, o_dnh = 0.f;
    float ins[2][6];
    const size_t row_el = (size_t)(orow < B ? orow : row0) * T * H;
    const float* dy_r = dy ? dy + row_el : nullptr;
    const float* res_r = reserve + 4 * row_el;
    const float* y_r = y + row_el;
    const float* h0_r = h0 + (size_t)(orow < B ? orow : row0) * H;
    float* g_r = gout + 4 * row_el;
    auto load_inputs = [&](float (&d)[6], int t) {
        const unsigned tH = (unsigned)t * (unsigned)H;  // 32-bit: B T H < 2^29
        d[0] = dy ? dy_r[tH + u] : 0.f;
        const float4 c4 = *reinterpret_cast<const float4*>(res_r + 4 * (tH + u));
        d[1] = c4.x;
        d[2] = c4.y;
        d[3] = c4.z;
        d[4] = c4.w;
        d[5] = t > 0 ? y_r[tH - H + u] : h0_r[u];
    };
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int c = 0; c < 6; ++c) ins[e][c] = 0.f;
    if (owner) {
        if (dhn) dh = dhn[(size_t)orow * H + u];
        load_inputs(ins[0], T - 1 - i0);
        if (i0 + 1 < i1) load_inputs(ins[1], T - 2 - i0);
    }
    if (threadIdx.x == 0) s_abort = 0;
    const rec::WaitCtl wc{abort_flag, p.abort_count, p.spin_limit};
    const bool xlocal = rec::group_on_one_xcd(p.xcc_words, gc.first, gc.stride, S, p.xcc_tag, wc, &s_local);

    // Word of (receiver c, sender q, row, unit) of this group, in each slot:
    // ((g S + c) S + q) 128 + 32 row + unit.  The failure injection publishes
    // into the other slot.
    const unsigned slot_words = (unsigned)p.G * (unsigned)(S * S) * 128u;
    const unsigned group_base = (unsigned)gc.g * (unsigned)(S * S) * 128u;
    const int pub_flip = (int)blockIdx.x == p.stall_block ? 1 : 0;
    // the lane's two published words of tile c: row l % 4, units 4 (ul / 4) +
    // 2 hf + 0, 1
    const unsigned pub_lane = (unsigned)(s * 128 + WU * lrow + (ul & ~3) + 2 * hf);
    // Thread i polls the words of (row, unit) i % 128 from senders i / 128 + 4 v.
    const int pair = threadIdx.x & 127, cls = threadIdx.x >> 7;
    unsigned poff[NPI];
    bool pval[NPI];
#pragma unroll
    for (int v = 0; v < NPI; ++v) {
        const int q = cls + 4 * v;
        pval[v] = q < S;
        poff[v] = group_base + (unsigned)((s * S + (q < S ? q : cls)) * 128 + pair);
    }

    auto pointwise = [&](const float (&cur)[6], float tsum) {
        if (owner) {
            const float cr = cur[1], cz = cur[2], cn = cur[3], ca = cur[4], hp = cur[5];
            const float f_n = (1.0f - cz) * (1.0f - cn * cn);  // dn^ / g
            const float f_r = ca * (cr * (1.0f - cr));         // dr^ / dn^
            const float f_z = (hp - cn) * (cz * (1.0f - cz));  // dz^ / g
            const float gsum = (ddirect + cur[0]) + tsum;      // g = dh_t + dy_t
            o_dnh = gsum * f_n;
            o_dan = o_dnh * cr;
            o_drh = o_dnh * f_r;
            o_dzh = gsum * f_z;
            ddirect = gsum * cz;
        }
        if (wave < 2) {
            gl[orl][ul] = owner ? o_drh : 0.f;
            gl[orl][WU + ul] = owner ? o_dzh : 0.f;
            gl[orl][2 * WU + ul] = owner ? o_dan : 0.f;
        }
    };
    auto step = [&](int i, float (&cur)[6], const float (&nxt)[6]) -> bool {
        const int t = T - 1 - i;
        const unsigned tag = p.tag_base + (unsigned)(i + 1);
        const float* gb = &gl[lrow][JH * hf];
        unsigned long long* pubs = exch + (size_t)((i & 1) ^ pub_flip) * slot_words + group_base + pub_lane;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int c = wave + NW * it;
            f4 acc[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int j = 0; j < JH; j += 4) {
                const float4 b = *reinterpret_cast<const float4*>(gb + j);
                acc[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(wl[it][j], b.x, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(wl[it][j + 1], b.y, acc[1], 0, 0, 0);
                acc[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(wl[it][j + 2], b.z, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(wl[it][j + 3], b.w, acc[1], 0, 0, 0);
            }
            const f4 a = acc[0] + acc[1];
            if (c < S) {  // wave-uniform
                unsigned long long* wp = pubs + (unsigned)(c * S) * 128u;
                unsigned long long* const pp2[2] = {wp, wp + 1};
                const unsigned long long w2[2] = {rec::pack_word(half_sums(a[0], a[2]), tag),
                                                  rec::pack_word(half_sums(a[1], a[3]), tag)};
                rec::publish_words<2>(pp2, w2, xlocal);
            }
        }
        {
            const unsigned long long* slotp = exch + (size_t)(i & 1) * slot_words;
            const unsigned long long* pp[NPI];
            unsigned long long w[NPI];
#pragma unroll
            for (int v = 0; v < NPI; ++v) {
                pp[v] = slotp + poff[v];
                w[v] = rec::load_word(pp[v]);
            }
            bool ok = true;
            rec::wait_words<NPI, true>(pp, pval, w, tag, wc, ok);
            if (!ok) s_abort = 1;
            float sum = 0.f;
#pragma unroll
            for (int v = 0; v < NPI; ++v) sum += pval[v] ? __uint_as_float((unsigned)w[v]) : 0.f;
            psum[i & 1][cls][pair] = sum;
        }
        if (owner) {
            float* op = g_r + 4 * (unsigned)t * (unsigned)H;
            __builtin_nontemporal_store(o_dan, op + u);
            __builtin_nontemporal_store(o_drh, op + H + u);
            __builtin_nontemporal_store(o_dzh, op + 2 * H + u);
            __builtin_nontemporal_store(o_dnh, op + 3 * H + u);
            if (t - 2 >= p.t_begin) load_inputs(cur, t - 2);
        }
        __syncthreads();
        const bool abort_now = s_abort != 0;
        float tsum = 0.f;
        if (owner) {
            const float (&ps)[4][WR * WU] = psum[i & 1];
            const int pr = WU * orl + ul;
            tsum = (ps[0][pr] + ps[1][pr]) + (ps[2][pr] + ps[3][pr]);
            dh = ddirect + tsum;
        }
        if (i + 1 < i1) pointwise(nxt, tsum);
        __syncthreads();
        return !abort_now;
    };
    if (i0 < i1) pointwise(ins[0], dh);  // dh_T = dhn (ddirect is 0)
    __syncthreads();
    // step i stores the G row of step i: after a step that aborts, rows
    // i_stop + 1 .. i1 - 1 were not stored
    int i_stop = i1;
    for (int i = i0; i < i1; i += 2) {
        if (!step(i, ins[0], ins[1])) {
            i_stop = i;
            break;
        }
        if (i + 1 < i1 && !step(i + 1, ins[1], ins[0])) {
            i_stop = i + 1;
            break;
        }
    }
    const bool aborted = i_stop < i1;
    if (owner) {
        if (aborted) {
            const float nan = __builtin_nanf("");
            for (int i = i_stop + 1; i < i1; ++i) {
                float* op = gout + ((size_t)orow * T + (T - 1 - i)) * 4 * H;
                op[u] = nan;
                op[H + u] = nan;
                op[2 * H + u] = nan;
                op[3 * H + u] = nan;
            }
        }
        dh0[(size_t)orow * H + u] = aborted ? __builtin_nanf("") : dh;
    }
}

const void* wide_kernel(int dir, int H) {
    const int S = (H + WU - 1) / WU;
    if (dir == 1)
        return S <= 16 ? reinterpret_cast<const void*>(&gru_bwd_wide_kernel<2>)
                       : reinterpret_cast<const void*>(&gru_bwd_wide_kernel<3>);
    const int kp = ((H + 15) / 16 + 7) / 8 * 8;
    switch (kp) {
        case 24: return reinterpret_cast<const void*>(&gru_fwd_wide_kernel<24>);
        case 32: return reinterpret_cast<const void*>(&gru_fwd_wide_kernel<32>);
        case 40: return reinterpret_cast<const void*>(&gru_fwd_wide_kernel<40>);
        default: return reinterpret_cast<const void*>(&gru_fwd_wide_kernel<48>);
    }
}

// Groups of four rows per launch: one workgroup per CU on 256 CUs, a
// multiple of 8 from 8 up so that each group shares an XCD.
int wide_groups_per_launch(int batch, int S) {
    int cap = 256 / S;
    if (cap >= 8) cap -= cap % 8;
    return std::min((batch + WR - 1) / WR, std::max(cap, 1));
}

}  // namespace

bool wide_takes(int H) { return H > 256 && H <= 768; }

size_t wide_exchange_words(int dir, int batch, int H) {
    const size_t S = (H + WU - 1) / WU;
    if (dir == 0) return (size_t)2 * batch * H;
    // two slots of one launch's words: the launches of a call share them,
    // their step tags differ
    return (size_t)2 * wide_groups_per_launch(batch, (int)S) * S * S * (WR * WU);
}

int wide_choose(int dir, int batch, int hidden, const DeviceInfo& dev, RecConfig* cfg) {
    if (!wide_takes(hidden)) return fail(RKA_ERR_UNSUPPORTED_SHAPE, "wide recurrence: 257 to 768 hidden units");
    const int S = (hidden + WU - 1) / WU;
    int per_cu = 0;
    RKA_RETURN_IF_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, wide_kernel(dir, hidden), NTH, 0));
    const long resident = (long)per_cu * dev.num_cus;
    const int groups = wide_groups_per_launch(batch, S);
    if ((long)groups * S > resident)
        return fail(RKA_ERR_TOO_LARGE_FOR_RESIDENT_LAUNCH, "wide recurrence: no resident grid at hidden_size " +
                                                               std::to_string(hidden));
    cfg->kind = REC_REGISTER;
    cfg->batch_per_launch = std::min(batch, groups * WR);
    cfg->launches = (batch + cfg->batch_per_launch - 1) / cfg->batch_per_launch;
    cfg->groups = groups;
    cfg->slices = S;
    cfg->units = WU;
    cfg->rows = WR;
    cfg->pair_waves = 0;
    cfg->chunk = WU;
    cfg->lds_bytes = 0;
    cfg->resident = resident;
    return 0;
}

int wide_launch(int dir, const RecConfig& c, const rec::Args& a, hipStream_t stream) {
    if (!wide_takes(a.H) || c.slices != (a.H + WU - 1) / WU || c.rows != WR)
        return fail(RKA_ERR_UNSUPPORTED_SHAPE, "wide recurrence: bad config");
    WideParams prm{a.B, a.T, a.H, c.groups, c.slices, a.t_begin, a.t_end, a.xcc_words, a.xcc_tag, a.tag_base,
                   a.spin_limit, a.abort_count, a.stall_block};
    const void* k = wide_kernel(dir, a.H);
    const dim3 grid((unsigned)(grid_groups(c, c.groups) * c.slices));
    if (dir == 0) {
        void* args[] = {(void*)&a.gx, (void*)&a.h0, (void*)&a.w_hh, (void*)&a.b_hh, (void*)&a.y, (void*)&a.hn,
                        (void*)&a.reserve, (void*)&a.exch, (void*)&a.abort_flag, (void*)&prm};
        RKA_RETURN_IF_HIP(hipLaunchKernel(k, grid, dim3(NTH), args, 0, stream));
    } else {
        void* args[] = {(void*)&a.dy, (void*)&a.dhn, (void*)&a.reserve, (void*)&a.h0, (void*)&a.y,
                        (void*)&a.w_hh, (void*)&a.gout, (void*)&a.dh0, (void*)&a.exch, (void*)&a.abort_flag,
                        (void*)&prm};
        RKA_RETURN_IF_HIP(hipLaunchKernel(k, grid, dim3(NTH), args, 0, stream));
    }
    return 0;
}

}  // namespace rka
