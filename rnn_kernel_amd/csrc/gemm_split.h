// fp32 products on the bf16 matrix cores, for the large ones: a float32 is the
// exact sum of three bf16 values (24 mantissa bits in three rounded pieces of 8,
// x = p0 + p1 + p2), so a product of two is nine bf16 products, each exact in
// float32.  The three smallest (p1 q2, p2 q1, p2 q2, together at most about 2^-24
// of the product) are left out, the other six go to v_mfma_f32_32x32x16_bf16,
// smallest first, into one float32 accumulator: six matrix instructions of 32
// clocks per 32x32x16 block where the fp32 ones (32x32x2) take eight of 64.
// Included by gemm_f32.hip, whose GemmArgs and tile orders it shares.
//
// Error against float64 (2-norm, MI355X, normal values; this / fp32 MFMA): m =
// 32768, n = 768, k = 256: 2.4e-7 / 2.9e-7; n = 256, k = 768: 4.2e-7 / 5.0e-7;
// k = 2304: 7.5e-7 / 8.6e-7: smaller at every size, since one instruction sums
// sixteen products before it rounds.  A second accumulator for the five small
// products brings 9e-8 at k = 256 but costs the third workgroup per CU (94 vs
// 83 us), and is not used.
//
// What bounds it: nothing alone.  The matrix cores are busy 0.40 to 0.54 of the
// cycles and the VALU issues on 0.11 to 0.16 of them; the wavefronts wait to issue
// for 0.35 to 0.46 of theirs and on counters (the loads, LDS) for 0.2 to 0.33, one
// barrier per 16-deep stage (24 MFMAs per wavefront, 72 KB of LDS traffic per
// workgroup).  The clock falls to 1.8-1.9 GHz meanwhile.  128x128 tiles
// of four wavefronts, 64x64 each; the operands are loaded as float32 two stages
// ahead in registers, split there and written to LDS as three planes (48 KB for
// two stages: three workgroups per CU).  Measured against the fp32
// tiles they replace (us): 32768 x 768, k = 256: 113 -> 81; 8192 x 2304, k = 768:
// 237 -> 165; 16384 x 1536, k = 512: 211 -> 141; the weight-gradient pair 768 x
// (256 + 256), k = 32768: 229 -> 162, k = 262144: 1725 -> 1245.
//
// Operands without aligned float4 rows (odd sizes; UA, any row length from 4) are
// loaded in the same float4 from 4-byte-aligned addresses.  Against the fp32
// register-staged tiles they replace (us): 32768 x 387, k = 129: 60 -> 40; 32768 x
// 129, k = 387: 58 -> 46; 19200 x 1533, k = 511: 308 -> 190; the pair 387 x (129 +
// 129), k = 32768: 155 -> 117; 993 x (331 + 331), k = 8192: 152 -> 86.
//
// Non-finite values: the pieces of an infinity are not finite sums, so a workgroup
// one of whose outputs comes out infinite or NaN computes its tile again in 64x64
// fp32 tiles (gemm_small.h) and replaces those outputs; finite results are never
// touched.  Where every output is NaN (after a diverged step, or an aborted
// recurrence) a product takes both forms' time: 32768 x 768, k = 256 256 us
// against 86; a training pass at batch 64, 512 steps, I = H = 256 1.26 ms against
// 1.15 (11.4 and 17.4 ms when each lane went over its outputs one by one).

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));

constexpr int kSplitTile = 128;                  // tile edge
constexpr int kPlane = kSplitTile * 8;           // dwords of a plane: 128 rows x 16 k of bf16
constexpr int kSplitStage = 2 * 3 * kPlane;      // dwords of a stage

// Operands are multiplied by 2^23 before they are split, products by 2^-46 in the
// end.  The smallest float32 is 2^-149, so that every piece is then at least
// 2^-126, and a product of pieces that could be lost is below 2^-172: nothing
// is lost that a float32 holds.  Without the scale the lower pieces of values
// below some 1e-33 were: error of a product with one operand of 1e-36 2.7e-5
// (2-norm, against 2.4e-7), of 1e-38 2.7e-3.  Operands from 2^105 or sums from 2^82
// overflow, and are computed again as other results that are not finite.  The
// multiplication costs 1 to 3 % of a product (pair at k = 32768: 157 -> 161 us).
constexpr float kSplitScale = 8388608.f;                  // 2^23
constexpr float kSplitUnscale = 1.f / kSplitScale / kSplitScale;

// v_mfma_f32_32x32x16_bf16 rounds its sums towards minus infinity (what the
// addends hold below the largest one's last bits is cut off): on average -2e-8 of
// an output's mean magnitude at k = 256, -1.5e-7 at k = 2304, in every row alike.
// What later sums over rows (the gradients of a stack's lower layers) adds that
// up, where roundings to nearest cancel.  So half of A's rows are split with the
// opposite sign and their sums negated in the end, which turns the direction of
// their rounding: the mean over all rows is then below 3e-10, as on the fp32 matrix
// cores.  Which rows is a hash of the row's own values (split_hash), not of its
// place, so that equal sequences of a batch give equal results.  In the split-K
// products, whose rows are the gate units, it is the odd rows; odd slices change sign
// too, so that the error cancels in the sum of the slices (k = 262144: 1.6e-6 ->
// 8.8e-7).  (Negating the sums every eight stages instead took 2 % of the pair.)

// The three pieces of a and b times s (a scale of either sign), packed in pairs
// (a low).
__device__ __forceinline__ void split3(float a, float b, float s, unsigned (&p)[3]) {
    a *= s;
    b *= s;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const bf16x2 v = {(__bf16)a, (__bf16)b};
        p[c] = __builtin_bit_cast(unsigned, v);
        if (c < 2) {
            a -= __uint_as_float(p[c] << 16);
            b -= __uint_as_float(p[c] & 0xffff0000u);
        }
    }
}

// The parity of the bits of a row's first sixteen values (of what the first stage
// loads for them; the four threads of the row hold four each).
__device__ __forceinline__ bool split_hash(const float4& v) {
    unsigned h = __float_as_uint(v.x) ^ __float_as_uint(v.y) ^ __float_as_uint(v.z) ^ __float_as_uint(v.w);
    h ^= __shfl_xor(h, 1, 4);
    h ^= __shfl_xor(h, 2, 4);
    return __popc(h) & 1;
}

// LDS planes of an operand's stage.  Row-major: [row][16 k] (32 bytes a row;
// thread x of a pass holds k 4 (x % 4) of row x / 4).  k-major: [k pair][row] of
// dwords (thread: rows 4 (t % 32) .. + 3 at k 2 (t / 32) and the next).  Bank
// conflicts counted per LDS instruction: 0 with both operands k-major, 1.2 with one,
// 2.6 cycles with both row-major.  s: the scales of the thread's two rows
// (row-major), or of its even and odd rows (k-major).
template <int KMAJOR>
__device__ __forceinline__ void split_store(unsigned* lds, int tid, const float (&s)[2], const float4 (&v)[2]) {
    if constexpr (KMAJOR == 0) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            unsigned p[3], q[3];
            split3(v[j].x, v[j].y, s[j], p);
            split3(v[j].z, v[j].w, s[j], q);
#pragma unroll
            for (int c = 0; c < 3; ++c)
                *reinterpret_cast<uintx2*>(lds + c * kPlane + (tid + NT * j) * 2) = uintx2{p[c], q[c]};
        }
    } else {
        unsigned p[4][3];
        split3(v[0].x, v[1].x, s[0], p[0]);
        split3(v[0].y, v[1].y, s[1], p[1]);
        split3(v[0].z, v[1].z, s[0], p[2]);
        split3(v[0].w, v[1].w, s[1], p[3]);
#pragma unroll
        for (int c = 0; c < 3; ++c)
            *reinterpret_cast<uintx4*>(lds + c * kPlane + (tid / 32) * kSplitTile + 4 * (tid % 32)) =
                uintx4{p[0][c], p[1][c], p[2][c], p[3][c]};
    }
}

// A wavefront's fragments, block x and piece c: lane 32 h + i holds k 8 h .. + 7
// of tile row row0 + 32 x + i (row-major) or row0 + 2 i + x (k-major).
template <int KMAJOR>
__device__ __forceinline__ void split_frag(const unsigned* lds, int row0, int i, int h, bf16x8 (&f)[2][3]) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if constexpr (KMAJOR == 0) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
                f[x][c] = *reinterpret_cast<const bf16x8*>(lds + c * kPlane + (row0 + 32 * x + i) * 8 + 4 * h);
        } else {
            uintx4 a, b;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uintx2 u =
                    *reinterpret_cast<const uintx2*>(lds + c * kPlane + (4 * h + q) * kSplitTile + row0 + 2 * i);
                a[q] = u[0];
                b[q] = u[1];
            }
            f[0][c] = __builtin_bit_cast(bf16x8, a);
            f[1][c] = __builtin_bit_cast(bf16x8, b);
        }
    }
}

// Four floats from an address that is a multiple of 4 bytes (global_load_dwordx4
// asks for no more).
struct __attribute__((packed, aligned(4))) Float4U {
    float x, y, z, w;
};
template <bool UA>
__device__ __forceinline__ float4 split_load4(const char* p) {
    if constexpr (UA) {
        const Float4U v = *reinterpret_cast<const Float4U*>(p);
        return make_float4(v.x, v.y, v.z, v.w);
    } else {
        return *reinterpret_cast<const float4*>(p);
    }
}
// v moved down by sh elements (sh <= 3; what moves in from past v is not used).
__device__ __forceinline__ float4 split_shift(const float4& v, int sh) {
    // (loaded first: loads under the selects would be merged into one of a
    // selected address, and v would live in scratch)
    const float x = v.x, y = v.y, z = v.z, w = v.w;
    return make_float4(sh == 0 ? x : sh == 1 ? y : sh == 2 ? z : w, sh == 0 ? y : sh == 1 ? z : w, sh == 0 ? z : w, w);
}

// The loads of one operand.  Rows past the operand read its last rows, k past
// the range its last k (split_tile zeroes those).  UA: rows that are not aligned
// float4, of any length from 4: a float4 that would cross the operand's last
// row (k-major) or the end of the range (row-major) starts early enough to end
// there, and its values are moved down by `rsh`, or kshift(), elements.
template <int KMAJOR, bool UA>
struct SplitLoader {
    const char* base;
    size_t stage_bytes;
    unsigned kunit, row[2];  // (unsigned: one uniform base and 32-bit lane offsets)
    int rsh;

    static __device__ __forceinline__ int k_of(int tid, int j) {
        return KMAJOR ? 2 * (tid / 32) + j : 4 * (tid % 4);
    }
    __device__ __forceinline__ SplitLoader(const GemmOperand& op, int rows, int r0, int kbeg, int, int tid) {
        const size_t ld = (size_t)op.ld;
        const int back = UA && KMAJOR ? min(r0, 3) : 0;  // (rows >= 4: only a later tile has fewer than 4 rows)
        base = reinterpret_cast<const char*>(op.ptr + (KMAJOR ? (size_t)kbeg * ld + (r0 - back) : (size_t)r0 * ld + kbeg));
        stage_bytes = (size_t)16 * (KMAJOR ? 4 * ld : 4);
        kunit = KMAJOR ? 4u * (unsigned)op.ld : 4u;
        const int r = min(4 * (tid % 32), rows - r0 - 4);
        rsh = UA && KMAJOR ? min(4 * (tid % 32) - r, 3) : 0;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            row[j] = KMAJOR ? 4u * (unsigned)(r + back)
                            : 4u * (unsigned)op.ld * (unsigned)min((tid + NT * j) / 4, rows - r0 - 1);
    }
    // stage kb, or the last one again past it
    __device__ __forceinline__ void load(int kb, int nkb, int klen, int tid, float4 (&v)[2]) const {
        const int st = min(kb, nkb - 1);
        const char* p = base + (size_t)st * stage_bytes;
        const int lim = klen - 16 * st - (KMAJOR ? 1 : 4);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int k = min(k_of(tid, j), lim);
            if constexpr (UA && !KMAJOR)  // (k may be negative)
                v[j] = split_load4<UA>(p - 16 + (row[j] + 4u * (unsigned)(k + 4)));
            else
                v[j] = split_load4<UA>(p + (row[j] + (unsigned)k * kunit));
        }
    }
    // the last stage of rem < 16 values: what its float4 started early by
    static __device__ __forceinline__ int kshift(int tid, int rem) {
        return UA && !KMAJOR ? min(max(k_of(tid, 0) - (rem - 4), 0), 3) : 0;
    }
};

// The k-major [h0 ; y[:, :-1]] operand (ShiftLoader in gemm_small.h): stages in
// order, k past the range read row 0 of shift_first.
template <bool UA>
struct SplitShiftLoader {
    using Plain = SplitLoader<1, UA>;
    const float* ptr;
    const float* first;
    size_t ld;
    int T, left, row, rsh, t, b, k;  // (t, b, k: of the first of the thread's two k)

    __device__ __forceinline__ SplitShiftLoader(const GemmOperand& op, int rows, int r0, int kbeg, int klen, int tid)
        : ptr(op.ptr), first(op.shift_first), ld((size_t)op.ld), T(op.shift_T), left(klen) {
        row = min(r0 + 4 * (tid % 32), rows - 4);
        rsh = UA ? min(r0 + 4 * (tid % 32) - row, 3) : 0;
        k = kbeg + Plain::k_of(tid, 0);
        b = k / T;
        t = k - b * T;
    }
    __device__ __forceinline__ void load(int, int, int, int tid, float4 (&v)[2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const bool in = Plain::k_of(tid, j) < left;
            const bool wrap = t + j >= T;  // j = 1: the next sequence's first step
            const bool start = !in || wrap || t + j == 0;
            const float* src = start ? first : ptr;
            const size_t line = !in ? 0 : start ? (size_t)(b + (wrap ? 1 : 0)) : (size_t)(k + j - 1);
            v[j] = split_load4<UA>(reinterpret_cast<const char*>(src + line * ld + row));
        }
        k += 16;
        t += 16;
        if (t >= T) {
            const int q = t / T;
            b += q;
            t -= q * T;
        }
        left -= 16;
    }
    static __device__ __forceinline__ int kshift(int, int) { return 0; }
};

// The tile (bx, by) again in fp32, for the outputs that are not finite.
template <int AK, int BKM, bool SPLIT, bool SHIFT, bool UA>
__device__ __forceinline__ void split_redo(const GemmArgs& p, int bx, int by, int bz, unsigned* smem) {
    using S = SmallTile<64, 64, 32, 32, 16>;
    static_assert(S::smem<AK, BKM>() <= 2 * kSplitStage, "fits the stages' memory");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the wavefront's outputs are stored
#pragma unroll 1
    for (int q = 0; q < 4; ++q) {
        __syncthreads();
        const int sx = 2 * bx + (q & 1), sy = 2 * by + (q >> 1);
        if (S::TM * sx < p.m && S::TN * sy < p.n)
            small_tile<AK, BKM, S, !UA, SPLIT, SHIFT, true>(p, sx, sy, bz, reinterpret_cast<float*>(smem));
    }
}

// One 128x128 tile (bx, by); SPLIT: the partial products of k slice bz, with the
// column sums of A in the first column of tiles (as small_tile).
template <int AK, int BKM, bool SPLIT, bool SHIFT, bool UA>
__device__ __forceinline__ void split_tile(const GemmArgs& p, int bx, int by, int bz, unsigned* smem) {
    static_assert(!SPLIT || (AK == 1 && BKM == 1), "split-K products take k-major operands");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int i = lane & 31, h = lane >> 5;
    const int m0 = bx * kSplitTile, n0 = by * kSplitTile;
    const int kbeg = SPLIT ? bz * p.kchunk : 0;
    const int klen = SPLIT ? max(0, min(p.k - kbeg, p.kchunk)) : p.k;
    const int nkb = (klen + 15) / 16;
    const bool colsum = SPLIT && p.want_colsum && by == 0;
    __shared__ int s_odd;  // an output is not finite
    if (tid == 0) s_odd = 0;
    float4 cs = make_float4(0.f, 0.f, 0.f, 0.f);

    using LA = SplitLoader<AK, UA>;
    using LB = std::conditional_t<SHIFT, SplitShiftLoader<UA>, SplitLoader<BKM, UA>>;
    const LA la(p.a, p.m, m0, kbeg, klen, tid);
    LB lb(p.b, p.n, n0, kbeg, klen, tid);
    float4 ra[2][2], rb[2][2];
    const float sign = SPLIT && (bz & 1) ? -1.f : 1.f;  // of the tile's even rows (k-major A)
    float scale_a[2] = {sign * kSplitScale, -sign * kSplitScale};
    const float scale_b[2] = {kSplitScale, kSplitScale};
    __shared__ __attribute__((aligned(16))) float s_unscale[AK ? 4 : kSplitTile];  // of each row of a row-major A
    floatx16 acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[x][y][r] = 0.f;
    // the last, shorter stage: zero past the range (UA, row-major: value by value)
    auto zero_past = [&](auto kmajor, int rem, int sh, float4 (&v)[2]) {
        constexpr int KM = decltype(kmajor)::value;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int k = SplitLoader<KM, UA>::k_of(tid, j);
            constexpr int s = UA && !KM ? 1 : 0;
            if constexpr (s == 1) v[j] = split_shift(v[j], sh);
            v[j] = make_float4(k < rem ? v[j].x : 0.f, k + s < rem ? v[j].y : 0.f, k + 2 * s < rem ? v[j].z : 0.f,
                               k + 3 * s < rem ? v[j].w : 0.f);
        }
    };
    // tiles whose last k-major float4 would cross the operand's last row
    const bool edge_a = UA && AK && m0 + kSplitTile > p.m, edge_b = UA && BKM && n0 + kSplitTile > p.n;
    auto stage = [&](int kb, auto st) {
        constexpr int ST = decltype(st)::value;
        unsigned* as = smem + ST * kSplitStage;
        unsigned* bs = as + 3 * kPlane;
        if (klen - 16 * kb < 16) {  // the last, shorter stage
            const int rem = klen - 16 * kb;
            zero_past(std::integral_constant<int, AK>{}, rem, LA::kshift(tid, rem), ra[ST]);
            zero_past(std::integral_constant<int, BKM>{}, rem, LB::kshift(tid, rem), rb[ST]);
        }
        if constexpr (UA && AK) {
            if (edge_a) {
#pragma unroll
                for (int j = 0; j < 2; ++j) ra[ST][j] = split_shift(ra[ST][j], la.rsh);
            }
        }
        if constexpr (UA && BKM) {
            if (edge_b) {
#pragma unroll
                for (int j = 0; j < 2; ++j) rb[ST][j] = split_shift(rb[ST][j], lb.rsh);
            }
        }
        if constexpr (SPLIT) {
            if (colsum) {
                cs.x += ra[ST][0].x + ra[ST][1].x;
                cs.y += ra[ST][0].y + ra[ST][1].y;
                cs.z += ra[ST][0].z + ra[ST][1].z;
                cs.w += ra[ST][0].w + ra[ST][1].w;
            }
        }
        split_store<AK>(as, tid, scale_a, ra[ST]);
        split_store<BKM>(bs, tid, scale_b, rb[ST]);
        la.load(kb + 2, nkb, klen, tid, ra[ST]);
        lb.load(kb + 2, nkb, klen, tid, rb[ST]);
        __syncthreads();
        bf16x8 fa[2][3], fb[2][3];
        split_frag<AK>(as, 64 * wm, i, h, fa);
        split_frag<BKM>(bs, 64 * wn, i, h, fb);
        // four independent blocks between two products of one
        auto product = [&](int pa, int pb) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[x][pa], fb[y][pb], acc[x][y], 0, 0, 0);
        };
        product(2, 0);
        product(0, 2);
        product(1, 1);
        product(1, 0);
        product(0, 1);
        product(0, 0);
    };
    if (nkb > 0) {
        la.load(0, nkb, klen, tid, ra[0]);
        lb.load(0, nkb, klen, tid, rb[0]);
        la.load(1, nkb, klen, tid, ra[1]);
        lb.load(1, nkb, klen, tid, rb[1]);
        if constexpr (!AK) {
            // (read behind the loop's barriers)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const bool neg = split_hash(ra[0][j]);
                scale_a[j] = neg ? -kSplitScale : kSplitScale;
                if (tid % 4 == 0) s_unscale[tid / 4 + 64 * j] = neg ? -kSplitUnscale : kSplitUnscale;
            }
        }
        int kb = 0;
        for (; kb + 1 < nkb; kb += 2) {
            stage(kb, std::integral_constant<int, 0>{});
            stage(kb + 1, std::integral_constant<int, 1>{});
        }
        if (kb < nkb) stage(kb, std::integral_constant<int, 0>{});
    }

    // acc[x][y][r] is C(row(x, r), col(y)): the row of register r in a block is 8
    // (r / 4) + 4 h + r % 4, its column i
    const bool direct = !SPLIT || p.c != nullptr;  // (SPLIT: one slice, rows rotated)
    auto row_of = [&](int x, int r) {
        const int lr = 8 * (r / 4) + 4 * h + r % 4;
        return m0 + 64 * wm + (AK ? 2 * lr + x : 32 * x + lr);
    };
    auto col_of = [&](int y) { return n0 + 64 * wn + (BKM ? 2 * i + y : 32 * y + i); };
    auto dst_of = [&](int m) -> float* {
        if constexpr (SPLIT) {
            if (!direct) return p.partial + ((size_t)(p.z_off + bz) * p.m + m) * p.n;
            return p.c + (size_t)(m >= p.rot ? m - p.rot : m - p.rot + p.m) * p.ldc;
        } else {
            return p.c + (size_t)m * p.ldc;
        }
    };
    float bias[2] = {0.f, 0.f};
    if (!SPLIT && p.bias) {
#pragma unroll
        for (int y = 0; y < 2; ++y) bias[y] = p.bias[min(col_of(y), p.n - 1)];
    }
    bool odd = false;  // an output that is not finite
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = row_of(x, r);
            const float u = AK ? (x ? -sign : sign) * kSplitUnscale  // (m odd: x is 1)
                               : s_unscale[64 * wm + 32 * x + 8 * (r / 4) + 4 * h + r % 4];
            const float v[2] = {fmaf(acc[x][0][r], u, bias[0]), fmaf(acc[x][1][r], u, bias[1])};
            odd = odd || !__builtin_isfinite(v[0]) || !__builtin_isfinite(v[1]);
            if (m >= p.m) continue;
            float* dst = dst_of(m);
            typedef float floatx2 __attribute__((ext_vector_type(2)));
            if (BKM && p.c_vec && col_of(1) < p.n) {
                const floatx2 vv = {v[0], v[1]};
                if (SPLIT)
                    *reinterpret_cast<floatx2*>(dst + col_of(0)) = vv;
                else
                    __builtin_nontemporal_store(vv, reinterpret_cast<floatx2*>(dst + col_of(0)));
            } else {
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    if (col_of(y) >= p.n) continue;
                    if (SPLIT)
                        dst[col_of(y)] = v[y];
                    else
                        __builtin_nontemporal_store(v[y], dst + col_of(y));
                }
            }
        }
    if (__any(odd) && lane == 0) s_odd = 1;
    if constexpr (SPLIT) {
        if (colsum) {
            // rows 4 (tid % 32) .. + 3 from the eight threads that share them
            __syncthreads();
            float* red = reinterpret_cast<float*>(smem);  // [8][128]
            *reinterpret_cast<float4*>(red + (tid / 32) * kSplitTile + 4 * (tid % 32)) = cs;
            __syncthreads();
            if (tid < kSplitTile && m0 + tid < p.m) {
                float s = 0.f;
#pragma unroll
                for (int q = 0; q < 8; ++q) s += red[q * kSplitTile + tid];
                const int m = m0 + tid;
                if (direct)
                    p.colsum[m >= p.rot ? m - p.rot : m - p.rot + p.m] = s;
                else
                    (p.partial + (size_t)p.ksplit_total * p.m * p.n)[(size_t)(p.z_off + bz) * p.m + m] = s;
            }
        }
    }
    __syncthreads();
    if (__builtin_expect(s_odd != 0, 0)) split_redo<AK, BKM, SPLIT, SHIFT, UA>(p, bx, by, bz, smem);
}

template <int BKM, bool UA>
__global__ __launch_bounds__(NT, 3) void gemm_split_kernel(GemmArgs p) {
    __shared__ __attribute__((aligned(16))) unsigned smem[2 * kSplitStage];
    for (size_t i = (size_t)blockIdx.x * NT + threadIdx.x; i < p.zero_words; i += (size_t)gridDim.x * NT) p.zero[i] = 0ull;
    int bx, by;
    direct_coords(p, blockIdx.x, bx, by);
    split_tile<0, BKM, false, false, UA>(p, bx, by, 0, smem);
}

template <int BKM, bool UA>
__global__ __launch_bounds__(NT, 3) void gemm_split_reduce_kernel(GemmArgs p, ReduceJob j0, ReduceJob j1) {
    __shared__ __attribute__((aligned(16))) unsigned smem[2 * kSplitStage];
    if ((int)blockIdx.x >= p.tiles) {
        reduce_range(j0, j1, (int)blockIdx.x - p.tiles, (int)gridDim.x - p.tiles);
        return;
    }
    int bx, by;
    direct_coords(p, blockIdx.x, bx, by);
    split_tile<0, BKM, false, false, UA>(p, bx, by, 0, smem);
}

// The weight-gradient pair (the first product with the row remap).
template <bool UA>
__global__ __launch_bounds__(NT, 3) void gemm_split_pair_kernel(GemmArgs p0, GemmArgs p1) {
    __shared__ __attribute__((aligned(16))) unsigned smem[2 * kSplitStage];
    const int blocks0 = p0.tiles * p0.ksplit;
    int bx, by, bz;
    if ((int)blockIdx.x < blocks0) {
        split_coords(p0, blockIdx.x, bx, by, bz);
        split_tile<1, 1, true, true, UA>(p0, bx, by, bz, smem);
    } else {
        split_coords(p1, blockIdx.x - blocks0, bx, by, bz);
        split_tile<1, 1, true, false, UA>(p1, bx, by, bz, smem);
    }
}
