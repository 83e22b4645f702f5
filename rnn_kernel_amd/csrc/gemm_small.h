// Register-staged form of the direct fp32 products (input projection, dx) in
// tiles from 32x32 to 128x64, for products that 128x128 tiles would spread
// unevenly over the CUs or leave most of them idle, and for operands that are
// not 16-byte aligned.  Included by gemm_f32.hip, whose GemmArgs, operand
// descriptions and tile orders it shares; direct_tile there chooses.
//
// What bounds a product of few tiles is latency, not the matrix cores: the
// 128x128 ring walks its k extent 16 at a time at 1.1-1.4 us per stage when few
// workgroups run (55 us at k = 768 for one row of x).  Here a workgroup's tile
// is up to 16 times smaller, so there are up to 16 times the workgroups, and
// the 32x32 form runs 64-deep stages of which its four wavefronts take a
// quarter each: 8 us.  Two stages are in flight in registers besides the one
// in LDS; the loads carry no branches, 64-bit address arithmetic or selects
// between objects, each of which cost more than the MFMAs.  Large products
// that divide evenly run within a few per cent of the ring (the figures stand
// at direct_tile).

// A TM x TN tile of four wavefronts, each computing a WT x WTN sub-tile of it;
// where there are fewer sub-tiles than wavefronts, WK of them share one and
// split each stage's k (their sums are added in LDS at the end, in a fixed
// order).
template <int TM_, int TN_, int WTM_, int WTN_, int BK_>
struct SmallTile {
    static constexpr int TM = TM_, TN = TN_, WTM = WTM_, WTN = WTN_, BK = BK_;
    static constexpr int WM = TM / WTM, WN = TN / WTN, WK = 4 / (WM * WN);
    static constexpr int MB = WTM / 16, NB = WTN / 16;  // 16x16 blocks of a sub-tile
    static constexpr int NG = BK / 16 / WK;             // 16-deep k groups per wavefront and stage
    static_assert(WM * WN * WK == 4 && NG >= 1, "four wavefronts");
    // LDS forms as in gemm_f32.hip: [row][k] for a row-major operand, [k][row]
    // for a k-major one; both padded by 4
    template <int KMAJOR, int R>
    static constexpr int ld() {
        return KMAJOR ? R + 4 : BK + 4;
    }
    template <int KMAJOR, int R>
    static constexpr int floats() {
        return KMAJOR ? BK * (R + 4) : R * (BK + 4);
    }
    template <int AK, int BKM>
    static constexpr int smem() {
        constexpr int stages = 2 * (floats<AK, TM>() + floats<BKM, TN>());
        constexpr int red = WK * TM * (TN + 4);
        return stages > red ? stages : red;
    }
};

// The loads of one operand's stages (R rows from r0, BK deep) into registers, NV
// float4 per thread.  VEC: float4 loads (both operands vec_ok), else one float
// per lane in consecutive addresses; a template parameter, because a branch
// around the loads makes the compiler wait for them behind it.  A lane's byte
// offset from the tile's first row is a row part and a k part, fixed before the
// loop; a stage adds its wave-uniform start.  Rows past the operand read its
// last row (their products are not stored); k past the extent is clamped (one
// minimum per load) and zeroed when the stage is written to LDS.
template <int KMAJOR, int R, int BK, bool VEC, int NV>
struct SmallLoader {
    static constexpr int NL = VEC ? NV : 4 * NV;
    const char* base;      // operand at (r0, kbeg), wave-uniform
    size_t stage_bytes;    // bytes from one stage to the next
    unsigned kunit;        // bytes per k
    unsigned row[NL], kk[NL];

    // x-th element (float4 or float) of the stage: its row and k
    static __device__ __forceinline__ int row_of(int x) {
        if constexpr (VEC) return KMAJOR ? 4 * (x % (R / 4)) : x / (BK / 4);
        return KMAJOR ? x % R : x / BK;
    }
    static __device__ __forceinline__ int k_of(int x) {
        if constexpr (VEC) return KMAJOR ? x / (R / 4) : 4 * (x % (BK / 4));
        return KMAJOR ? x / R : x % BK;
    }

    __device__ __forceinline__ SmallLoader(const GemmOperand& op, int rows, int r0, int kbeg, int klen, int tid) {
        (void)klen;
        const size_t ld = (size_t)op.ld;
        base = reinterpret_cast<const char*>(op.ptr + (KMAJOR ? (size_t)kbeg * ld + r0 : (size_t)r0 * ld + kbeg));
        kunit = KMAJOR ? 4u * (unsigned)op.ld : 4u;
        stage_bytes = (size_t)BK * (KMAJOR ? 4 * ld : 4);
        const int last = rows - r0 - (VEC && KMAJOR ? 4 : 1);  // last row (row group) of the tile
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int x = tid + NT * j;
            row[j] = (unsigned)min(row_of(x), last) * (KMAJOR ? 4u : 4u * (unsigned)op.ld);
            kk[j] = (unsigned)k_of(x) * kunit;
        }
    }
    // stage kb of the nkb that klen values make, or the last one again past it
    __device__ __forceinline__ void load(int kb, int nkb, int klen, float4 (&v)[NV]) const {
        const int st = min(kb, nkb - 1);
        const char* p = base + (size_t)st * stage_bytes;
        // (a stage's own k at most: klen rows of a wide operand are past 32 bits)
        const unsigned lim = (unsigned)min(klen - st * BK - (VEC && !KMAJOR ? 4 : 1), BK) * kunit;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            if constexpr (VEC) {
                v[j] = *reinterpret_cast<const float4*>(p + (row[j] + min(kk[j], lim)));
            } else {
                float e[4];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    e[c] = *reinterpret_cast<const float*>(p + (row[4 * j + c] + min(kk[4 * j + c], lim)));
                v[j] = make_float4(e[0], e[1], e[2], e[3]);
            }
        }
    }
};

// The same for the k-major [h0 ; y[:, :-1]] operand (GemmOperand::shift_T): k =
// b T + t reads row k - 1 of ptr, or row b of shift_first where t = 0.  Stages
// are loaded in order, so each element carries its t and b and one stage on is
// an addition (a division only where a sequence ends).
template <int R, int BK, bool VEC, int NV>
struct ShiftLoader {
    using Plain = SmallLoader<1, R, BK, VEC, NV>;
    static constexpr int NL = Plain::NL;
    const float* ptr;
    const float* first;
    size_t ld;
    int T, left;           // left: k values from this stage's start to the end of the range
    int row[NL], t[NL], b[NL], k[NL];

    __device__ __forceinline__ ShiftLoader(const GemmOperand& op, int rows, int r0, int kbeg, int klen, int tid)
        : ptr(op.ptr), first(op.shift_first), ld((size_t)op.ld), T(op.shift_T), left(klen) {
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int x = tid + NT * j;
            row[j] = min(r0 + Plain::row_of(x), rows - (VEC ? 4 : 1));
            k[j] = kbeg + Plain::k_of(x);
            b[j] = k[j] / T;
            t[j] = k[j] - b[j] * T;
        }
    }
    // the next stage; elements past the range read row 0 of shift_first
    __device__ __forceinline__ void load(int, int, int, float4 (&v)[NV]) {
        float e[NL][VEC ? 4 : 1];
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const bool in = Plain::k_of((int)threadIdx.x + NT * j) < left;
            const bool start = !in || t[j] == 0;
            const float* src = start ? first : ptr;
            const size_t line = !in ? 0 : start ? (size_t)b[j] : (size_t)(k[j] - 1);
            src += line * ld + row[j];
            if constexpr (VEC) {
                const float4 u = *reinterpret_cast<const float4*>(src);
                e[j][0] = u.x;
                e[j][1] = u.y;
                e[j][2] = u.z;
                e[j][3] = u.w;
            } else {
                e[j][0] = *src;
            }
            k[j] += BK;
            t[j] += BK;
            if (t[j] >= T) {
                const int q = t[j] / T;
                b[j] += q;
                t[j] -= q * T;
            }
        }
        left -= BK;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            if constexpr (VEC)
                v[j] = make_float4(e[j][0], e[j][1], e[j][2], e[j][3]);
            else
                v[j] = make_float4(e[4 * j][0], e[4 * j + 1][0], e[4 * j + 2][0], e[4 * j + 3][0]);
        }
    }
};

template <int KMAJOR, int R, int BK, bool VEC, int NV>
__device__ __forceinline__ void small_store(float* lds, int kend, int k0, int tid, const float4 (&v)[NV]) {
    using Loader = SmallLoader<KMAJOR, R, BK, VEC, NV>;
    constexpr int LD = KMAJOR ? R + 4 : BK + 4;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        if constexpr (VEC) {
            const int x = tid + NT * j;
            const int r = Loader::row_of(x), k = Loader::k_of(x);
            // component by component: a select of two float4 objects became a
            // select of their addresses, and the stage registers scratch memory
            const bool in = k0 + k < kend;
            *reinterpret_cast<float4*>(lds + (KMAJOR ? k * LD + r : r * LD + k)) =
                make_float4(in ? v[j].x : 0.f, in ? v[j].y : 0.f, in ? v[j].z : 0.f, in ? v[j].w : 0.f);
        } else {
            const float e[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int x = tid + NT * (4 * j + c);
                const int r = Loader::row_of(x), k = Loader::k_of(x);
                lds[KMAJOR ? k * LD + r : r * LD + k] = k0 + k < kend ? e[c] : 0.f;
            }
        }
    }
}

// Fragments of a wavefront's 16 NBL rows for the 16-deep group at k: block x,
// MFMA step j (k = 4 g + j).  [row][k]: block x's row i is tile row 16 x + i;
// [k][row]: tile row NBL i + x.
template <int KMAJOR, int LD, int NBL>
__device__ __forceinline__ void small_frag(const float* lds, int row0, int k, int i, int g, float (&f)[NBL][4]) {
    static_assert(NBL == 2 || NBL == 4, "32 or 64 rows");
    if constexpr (KMAJOR == 0) {
#pragma unroll
        for (int x = 0; x < NBL; ++x) {
            const float4 v = *reinterpret_cast<const float4*>(lds + (row0 + 16 * x + i) * LD + k + 4 * g);
            f[x][0] = v.x;
            f[x][1] = v.y;
            f[x][2] = v.z;
            f[x][3] = v.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float* src = lds + (k + 4 * g + j) * LD + row0 + NBL * i;
            if constexpr (NBL == 2) {
                const float2 v = *reinterpret_cast<const float2*>(src);
                f[0][j] = v.x;
                f[1][j] = v.y;
            } else {
                const float4 v = *reinterpret_cast<const float4*>(src);
                f[0][j] = v.x;
                f[1][j] = v.y;
                f[2][j] = v.z;
                f[3][j] = v.w;
            }
        }
    }
}

// A weight gradient sums thousands of time steps: the 64x64 form closes its
// float32 sums every kFoldStages stages (128 values) and adds those up apart, so
// that a slice may be as long as the launch wants it and no chain of additions is
// longer than in the ring's shortest slices.  Error against float64 (2-norm) at
// batch 16, 256 steps, I = H = 256 in eight slices: 4.1e-7 -> 2.1e-7 (the ring, 32
// slices: 2.1e-7); time of the backward's products 69 -> 71 us.  The 128x64
// form would lose a workgroup per CU to the second set of sums (235 -> 276 us at
// 75, 258, 3, 308); its slices are kept as short as the ring's (make_pair_plan).
constexpr int kFoldStages = 8;

// One tile (bx, by); SPLIT: the partial products of k slice bz, with the column
// sums of A (the bias gradients) in the first column of tiles.  REDO: only outputs
// that are not finite are replaced (gemm_split.h), and no column sums formed.
template <int AK, int BKM, typename S, bool VEC, bool SPLIT = false, bool BSHIFT = false, bool REDO = false>
__device__ __forceinline__ void small_tile(const GemmArgs& p, int bx, int by, int bz, float* smem) {
    static_assert(!SPLIT || (AK == 1 && BKM == 1 && S::WK == 1), "split-K products take k-major operands");
    constexpr int TM = S::TM, TN = S::TN, BK = S::BK, MB = S::MB, NB = S::NB;
    constexpr int NVA = TM * BK / (4 * NT), NVB = TN * BK / (4 * NT);
    constexpr int AF = S::template floats<AK, TM>(), BF = S::template floats<BKM, TN>();
    constexpr int LDA = S::template ld<AK, TM>(), LDB = S::template ld<BKM, TN>();
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % S::WK, wm = wave / S::WK % S::WM, wn = wave / (S::WK * S::WM);
    const int i = lane & 15, g = lane >> 4;
    const int m0 = bx * TM, n0 = by * TN;
    const int kbeg = SPLIT ? bz * p.kchunk : 0;
    const int klen = SPLIT ? max(0, min(p.k - kbeg, p.kchunk)) : p.k;
    const int nkb = (klen + BK - 1) / BK;
    const bool colsum = SPLIT && !REDO && p.want_colsum && by == 0;
    float cs = 0.f;
    // the columns a thread stores are the same in every row it stores
    static_assert(NT % (TN / 4) == 0, "a thread's columns");
    const int scol = 4 * (tid % (TN / 4)), sn = n0 + scol;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (!SPLIT && p.bias) {
#pragma unroll
        for (int q = 0; q < 4; ++q) bias[q] = p.bias[min(sn + q, p.n - 1)];
    }
    floatx4 acc[MB][NB];
#pragma unroll
    for (int x = 0; x < MB; ++x)
#pragma unroll
        for (int y = 0; y < NB; ++y) acc[x][y] = floatx4{0.f, 0.f, 0.f, 0.f};
    const SmallLoader<AK, TM, BK, VEC, NVA> la(p.a, p.m, m0, kbeg, klen, tid);
    using LoaderB =
        std::conditional_t<BSHIFT, ShiftLoader<TN, BK, VEC, NVB>, SmallLoader<BKM, TN, BK, VEC, NVB>>;
    LoaderB lb(p.b, p.n, n0, kbeg, klen, tid);
    float4 ra[2][NVA], rb[2][NVB];
    auto load = [&](int kb, int st) {
        la.load(kb, nkb, klen, ra[st]);
        lb.load(kb, nkb, klen, rb[st]);
    };
    // stage kb: registers to LDS, the loads of stage kb + 2 into the same
    // registers, one barrier (the other LDS buffer's readers are past it), MFMAs
    auto stage = [&](int kb, auto st) {
        constexpr int ST = decltype(st)::value;
        float* as = smem + ST * (AF + BF);
        float* bs = as + AF;
        small_store<AK, TM, BK, VEC>(as, klen, kb * BK, tid, ra[ST]);
        small_store<BKM, TN, BK, VEC>(bs, klen, kb * BK, tid, rb[ST]);
        load(kb + 2, ST);
        __syncthreads();
        if constexpr (SPLIT) {
            if (colsum && tid < TM) {
#pragma unroll
                for (int kk = 0; kk < BK; ++kk) cs += as[kk * LDA + tid];
            }
        }
#pragma unroll
        for (int q = 0; q < S::NG; ++q) {
            const int k = 16 * (S::NG * wk + q);
            float fa[MB][4], fb[NB][4];
            small_frag<AK, LDA>(as, S::WTM * wm, k, i, g, fa);
            small_frag<BKM, LDB>(bs, S::WTN * wn, k, i, g, fb);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int x = 0; x < MB; ++x)
#pragma unroll
                    for (int y = 0; y < NB; ++y)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[x][j], fb[y][j], acc[x][y], 0, 0, 0);
        }
    };
    if (nkb > 0) {
        // every stage loads unconditionally (past the last one: the clamped
        // places again), so that no branch stands between a load and its use
        // and the compiler waits for the older stage's loads only
        load(0, 0);
        load(1, 1);
        int kb = 0;
        auto run = [&](int end) {
            for (; kb + 1 < end; kb += 2) {
                stage(kb, std::integral_constant<int, 0>{});
                stage(kb + 1, std::integral_constant<int, 1>{});
            }
        };
        if constexpr (SPLIT && TM == 64) {
            floatx4 sum[MB][NB];
            float csum = 0.f;
#pragma unroll
            for (int x = 0; x < MB; ++x)
#pragma unroll
                for (int y = 0; y < NB; ++y) sum[x][y] = floatx4{0.f, 0.f, 0.f, 0.f};
            while (kb + kFoldStages < nkb) {
                run(kb + kFoldStages);
#pragma unroll
                for (int x = 0; x < MB; ++x)
#pragma unroll
                    for (int y = 0; y < NB; ++y) {
                        sum[x][y] += acc[x][y];
                        acc[x][y] = floatx4{0.f, 0.f, 0.f, 0.f};
                    }
                csum += cs;
                cs = 0.f;
            }
            run(nkb);
            if (kb < nkb) stage(kb, std::integral_constant<int, 0>{});
#pragma unroll
            for (int x = 0; x < MB; ++x)
#pragma unroll
                for (int y = 0; y < NB; ++y) acc[x][y] += sum[x][y];
            cs += csum;
        } else {
            run(nkb);
            if (kb < nkb) stage(kb, std::integral_constant<int, 0>{});
        }
    }
    // through LDS: the wavefronts that split k are added in order, and rows of C
    // are written whole
    __syncthreads();
    constexpr int LDC = TN + 4;
    float* red = smem + wk * TM * LDC;
#pragma unroll
    for (int x = 0; x < MB; ++x)
#pragma unroll
        for (int y = 0; y < NB; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = S::WTM * wm + (AK ? MB * (4 * g + r) + x : 16 * x + 4 * g + r);
                const int col = S::WTN * wn + (BKM ? NB * i + y : 16 * y + i);
                red[row * LDC + col] = acc[x][y][r];
            }
    __syncthreads();
#pragma unroll
    for (int row = tid / (TN / 4); row < TM; row += NT / (TN / 4)) {
        const int m = m0 + row;
        float4 v = *reinterpret_cast<const float4*>(smem + row * LDC + scol);
#pragma unroll
        for (int w = 1; w < S::WK; ++w) {
            const float4 u = *reinterpret_cast<const float4*>(smem + w * TM * LDC + row * LDC + scol);
            v.x += u.x;
            v.y += u.y;
            v.z += u.z;
            v.w += u.w;
        }
        const float c[4] = {v.x + bias[0], v.y + bias[1], v.z + bias[2], v.w + bias[3]};
        if (m >= p.m || sn >= p.n) continue;
        float* dst;
        if constexpr (SPLIT) {
            // one slice: the sums are the result, its rows rotated (out[o] = C[(o + rot) % m])
            dst = p.c ? p.c + (size_t)(m >= p.rot ? m - p.rot : m - p.rot + p.m) * p.ldc + sn
                      : p.partial + ((size_t)(p.z_off + bz) * p.m + m) * p.n + sn;
        } else {
            dst = p.c + (size_t)m * p.ldc + sn;
        }
        if constexpr (REDO) {
#pragma unroll
            for (int q = 0; q < 4; ++q)  // (stored by other lanes: read past the L1)
                if (sn + q < p.n &&
                    !__builtin_isfinite(__hip_atomic_load(dst + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
                    dst[q] = c[q];
        } else if (p.c_vec && sn + 3 < p.n) {
            *reinterpret_cast<float4*>(dst) = make_float4(c[0], c[1], c[2], c[3]);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (sn + q < p.n) dst[q] = c[q];
        }
    }
    if constexpr (SPLIT) {
        if (colsum && tid < TM && m0 + tid < p.m) {
            const int m = m0 + tid;
            if (p.c)
                p.colsum[m >= p.rot ? m - p.rot : m - p.rot + p.m] = cs;
            else
                (p.partial + (size_t)p.ksplit_total * p.m * p.n)[(size_t)(p.z_off + bz) * p.m + m] = cs;
        }
    }
}

template <int AK, int BKM, typename S, bool VEC>
__global__ __launch_bounds__(NT) void gemm_small_kernel(GemmArgs p) {
    __shared__ __attribute__((aligned(16))) float smem[S::template smem<AK, BKM>()];
    for (size_t i = (size_t)blockIdx.x * NT + threadIdx.x; i < p.zero_words; i += (size_t)gridDim.x * NT) p.zero[i] = 0ull;
    int bx, by;
    direct_coords(p, blockIdx.x, bx, by);
    small_tile<AK, BKM, S, VEC>(p, bx, by, 0, smem);
}

// The same with the reductions of one or two split-K products in the
// workgroups after the tiles (gemm_direct_reduce_kernel).
template <int AK, int BKM, typename S, bool VEC>
__global__ __launch_bounds__(NT) void gemm_small_reduce_kernel(GemmArgs p, ReduceJob j0, ReduceJob j1) {
    __shared__ __attribute__((aligned(16))) float smem[S::template smem<AK, BKM>()];
    if ((int)blockIdx.x >= p.tiles) {
        reduce_range(j0, j1, (int)blockIdx.x - p.tiles, (int)gridDim.x - p.tiles);
        return;
    }
    int bx, by;
    direct_coords(p, blockIdx.x, bx, by);
    small_tile<AK, BKM, S, VEC>(p, bx, by, 0, smem);
}

// The two split-K weight-gradient products in one launch (gemm_f32_pair_kernel).
template <typename S, bool VEC>
__global__ __launch_bounds__(NT, S::TM == 64 ? 4 : 2) void gemm_small_pair_kernel(GemmArgs p0, GemmArgs p1) {
    __shared__ __attribute__((aligned(16))) float smem[S::template smem<1, 1>()];
    const int blocks0 = p0.tiles * p0.ksplit;
    int bx, by, bz;
    if ((int)blockIdx.x < blocks0) {
        split_coords(p0, blockIdx.x, bx, by, bz);
        small_tile<1, 1, S, VEC, true, true>(p0, bx, by, bz, smem);
    } else {
        split_coords(p1, blockIdx.x - blocks0, bx, by, bz);
        small_tile<1, 1, S, VEC, true, false>(p1, bx, by, bz, smem);
    }
}
