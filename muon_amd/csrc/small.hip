// The whole Muon step of a small matrix in one workgroup: momentum, norm, normalise, the Newton-Schulz
// iteration and the parameter step, with the iterate and its Gram matrix in LDS throughout.
//
// A matrix whose short side is at most 128 and whose iterate fits the 160 KB of LDS of a CU beside two
// Gram matrices needs nothing from other CUs between two products, so the 17 launches of the general
// path (4 us each on the GPU, 3.3 us each on the host, whatever the size) become one.  One CU is what a matrix
// gets, and what bounds it there is the vector ALU and LDS: of the 39 us of a 64 x 576 matrix the loads take 8, the
// normalise pass 2, each of the five iterations 5 (X X^T 1.9, the update 2.7) and the parameter step 2.5.
// muon_update of a 64 x 64 x 3 x 3 filter: 106 us in separate launches; 62 us with 8 waves, the index of
// every element from a division of its own, scaled divisions, all four 32 x 32 tiles of X X^T and 8-byte accesses
// to tiles; 48 us with 16 waves and without those.
//
// Every rounding and every order of summation is the general path's (elementwise.hip, ns_gemm.hip): the
// sum of squares goes by blocks of 8192 elements and 256 threads, the products accumulate k-step after
// k-step, so a matrix gets the same bits on either path.
#include "common.h"

namespace muon_amd {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4s __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int SMALL_THREADS = 1024, SMALL_WAVES = SMALL_THREADS / 64;
constexpr int SUM_BLOCK = 8192;                     // elements per partial sum (EW_BLOCK_ELEMS) ...
constexpr int SUM_THREADS = 256, SUM_ITERS = 8;     // ... and how its threads share them (4 in a row each)
constexpr int SMALL_LDS_MAX = 163840;
constexpr int SMALL_MAX_BLOCKS = 16;                // partial sums of the largest matrix that fits

// Rows are padded by 16 bytes: 16-byte reads of one chunk of 8 consecutive rows hit all banks.
__host__ __device__ constexpr int small_pitch(int cols) { return cols * 2 + 16; }
static size_t small_lds_bytes(int mp, int np) {
    return static_cast<size_t>(mp) * small_pitch(np) + 2 * static_cast<size_t>(mp) * small_pitch(mp) +
           SMALL_MAX_BLOCKS * 4 * sizeof(float);
}

template <typename T>
struct SmallIo;
template <>
struct SmallIo<float> {
    static constexpr uintptr_t kAlign = 16;
    static __device__ __forceinline__ f32x4s ld4(const float* p) { return *(const __attribute__((address_space(1))) f32x4s*)(p); }
    static __device__ __forceinline__ void st4(float* p, f32x4s v) { *(__attribute__((address_space(1))) f32x4s*)(p) = v; }
    static __device__ __forceinline__ float ld(const float* p) { return *p; }
    static __device__ __forceinline__ void st(float* p, float v) { *p = v; }
    static __device__ __forceinline__ float rnd(float v) { return v; }
};
template <>
struct SmallIo<uint16_t> {
    static constexpr uintptr_t kAlign = 8;
    static __device__ __forceinline__ f32x4s ld4(const uint16_t* p) {
        const u32x2 r = *(const __attribute__((address_space(1))) u32x2*)(p);
        return f32x4s{bf_lo(r.x), bf_hi(r.x), bf_lo(r.y), bf_hi(r.y)};
    }
    static __device__ __forceinline__ void st4(uint16_t* p, f32x4s v) {
        *(__attribute__((address_space(1))) u32x2*)(p) = u32x2{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])};
    }
    static __device__ __forceinline__ float ld(const uint16_t* p) { return bf2f(*p); }
    static __device__ __forceinline__ void st(uint16_t* p, float v) { *p = f2bf(v); }
    static __device__ __forceinline__ float rnd(float v) { return round_bf(v); }
};

__device__ __forceinline__ bool small_aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// 16 bytes of an LDS row as an MFMA operand: lane l holds k = 8 (l / 32) .. + 7 of row l % 32.
__device__ __forceinline__ bf16x8 row_frag(const char* base, int pitch, int row0, int ks, int lane) {
    return *reinterpret_cast<const bf16x8*>(base + (row0 + (lane & 31)) * pitch + ks * 32 + (lane >> 5) * 16);
}
// The same from a k-major operand (rows = k): two transposing reads of 4 rows x 16 columns per 16 lanes.
__device__ __forceinline__ bf16x8 col_frag(const char* base, int pitch, int col0, int ks, int lane) {
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    const char* const p = base + (ks * 16 + (lane >> 5) * 8 + ((lane & 15) >> 2)) * pitch +
                          (col0 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4) * 2;
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * pitch)));
    return __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y});
}
__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    return z;
}
// A 32 x 32 tile of packed bf16 pairs as the MFMAs leave it (lane = row l % 32, pair 2q + i = columns
// 8q + 4 (l / 32) + 2i) to LDS rows and back.  The halves of two neighbouring chunks of 8 columns are exchanged between
// lanes l and l + 32, so that a lane moves 8 columns in a row: 16-byte accesses hit all banks, the 8-byte
// ones of the layout itself meet rows 16 apart in the same bank.
__device__ __forceinline__ void tile_store(char* base, int pitch, int row0, int col0, int lane, const uint32_t (&po)[8]) {
    char* const p = base + (row0 + (lane & 31)) * pitch + (col0 + (lane >> 5) * 8) * 2;
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
        const auto x = __builtin_amdgcn_permlane32_swap(po[2 * q], po[2 * q + 2], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(po[2 * q + 1], po[2 * q + 3], false, false);
        *reinterpret_cast<u32x4*>(p + q * 16) = u32x4{x[0], y[0], x[1], y[1]};
    }
}
__device__ __forceinline__ void tile_load(uint32_t (&po)[8], const char* base, int pitch, int row0, int col0, int lane) {
    const char* const p = base + (row0 + (lane & 31)) * pitch + (col0 + (lane >> 5) * 8) * 2;
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(p + q * 16);
        const auto x = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
        po[2 * q] = x[0];
        po[2 * q + 1] = y[0];
        po[2 * q + 2] = x[1];
        po[2 * q + 3] = y[1];
    }
}
// The same tile as the columns of its mirror image.
__device__ __forceinline__ void tile_store_mirrored(char* base, int pitch, int row0, int col0, int lane, const uint32_t (&po)[8]) {
    char* const p = base + (col0 + (lane >> 5) * 4) * pitch + (row0 + (lane & 31)) * 2;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        char* const c = p + (8 * (k >> 1) + 2 * (k & 1)) * pitch;
        *reinterpret_cast<uint16_t*>(c) = static_cast<uint16_t>(po[k]);
        *reinterpret_cast<uint16_t*>(c + pitch) = static_cast<uint16_t>(po[k] >> 16);
    }
}
// o = alpha * acc + beta * D as the epilogue of the GEMM kernel rounds it; po holds D on entry and o on return.
template <bool ROUND>
__device__ __forceinline__ void tile_add(uint32_t (&po)[8], const f32x16& acc, float alpha, float beta) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t dk = po[k];
        if constexpr (ROUND) {
            // every term rounded to bf16, their sum rounded again, by the instructions of the GEMM epilogue (a dot
            // product with (1, 1) in place of unpacking and adding gives +0 for -0 + -0)
            const uint32_t t1 = pack2bf(alpha * acc[2 * k], alpha * acc[2 * k + 1]);
            const uint32_t t2 = pack2bf(beta * bf_lo(dk), beta * bf_hi(dk));
            po[k] = pack2bf(bf_lo(t1) + bf_lo(t2), bf_hi(t1) + bf_hi(t2));
        } else {
            po[k] = pack2bf(fmaf(alpha, acc[2 * k], beta * bf_lo(dk)), fmaf(alpha, acc[2 * k + 1], beta * bf_hi(dk)));
        }
    }
}

// Row and column of an element index that grows by a fixed stride: two divisions, then additions.
struct Walk {
    int r, c, dr, dc, cols;
    __device__ __forceinline__ Walk(int e, int stride, int cols_) : cols(cols_) {
        r = e / cols;
        c = e - r * cols;
        dr = stride / cols;
        dc = stride - dr * cols;
    }
    __device__ __forceinline__ void next() {
        r += dr;
        c += dc;
        if (c >= cols) {
            c -= cols;
            ++r;
        }
    }
};

// One tile of X X^T.  The reads of the next U k-steps are in flight under the MFMAs of the current ones; the
// rows of a diagonal tile are read once for both operands.  `nks` is a multiple of 4.
template <bool DIAG>
__device__ __forceinline__ void gram_tile(f32x16& acc, const char* X, int px, int i0, int j0, int nks, int lane) {
    constexpr int U = 4;
    bf16x8 fp[2][U], fq[2][U];
    const auto fetch = [&](int buf, int ks) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            fp[buf][u] = row_frag(X, px, i0, ks + u, lane);
            if constexpr (!DIAG) fq[buf][u] = row_frag(X, px, j0, ks + u, lane);
        }
    };
    const auto multiply = [&](int buf) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(DIAG ? fp[buf][u] : fq[buf][u], fp[buf][u], acc, 0, 0, 0);
    };
    fetch(0, 0);
    int ks = 0;
    for (; ks + 3 * U <= nks; ks += 2 * U) {
        fetch(1, ks + U);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0);
        fetch(0, ks + 2 * U);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1);
    }
    if (ks + 2 * U <= nks) {
        fetch(1, ks + U);
        multiply(0);
        multiply(1);
    } else {
        multiply(0);
    }
}

// X from gradient and momentum (muon.py:9-10, 277-279), and the partial sums of squares: block b of 8192
// elements by threads 256 (b % 4) .. + 255.
template <typename T>
__device__ __forceinline__ void small_load(const MuonMatDesc& d, char* X, int pitch, bool wide, float w, float beta,
                                           int nesterov, int mutate_grad, float* sums, int tid) {
    typedef SmallIo<T> S;
    const int numel = d.rows * d.cols, cols = d.cols;
    T* const g = static_cast<T*>(d.grad);
    T* const mom = static_cast<T*>(d.momentum);
    const bool has_m = mom != nullptr, write_g = has_m && nesterov && mutate_grad;
    const bool aligned = small_aligned(g, S::kAlign) && small_aligned(mom, S::kAlign);
    const bool in_row = (cols & 3) == 0;
    const int t = tid & (SUM_THREADS - 1);
    for (int b = tid / SUM_THREADS; b * SUM_BLOCK < numel; b += SMALL_THREADS / SUM_THREADS) {
        float ss = 0.f;
        Walk at(b * SUM_BLOCK + t * 4, SUM_THREADS * 4, cols);
#pragma unroll 1
        for (int first = b * SUM_BLOCK + t * 4; first < (b + 1) * SUM_BLOCK; first += SUM_BLOCK / 2) {
            f32x4s gv[SUM_ITERS / 2], mv[SUM_ITERS / 2];
#pragma unroll
            for (int it = 0; it < SUM_ITERS / 2; ++it) {
                const int e = first + it * SUM_THREADS * 4;
                gv[it] = mv[it] = f32x4s{0.f, 0.f, 0.f, 0.f};
                if (aligned && e + 4 <= numel) {
                    gv[it] = S::ld4(g + e);
                    if (has_m) mv[it] = S::ld4(mom + e);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (e + k < numel) {
                            gv[it][k] = S::ld(g + e + k);
                            if (has_m) mv[it][k] = S::ld(mom + e + k);
                        }
                }
            }
#pragma unroll
            for (int it = 0; it < SUM_ITERS / 2; ++it, at.next()) {
                const int e = first + it * SUM_THREADS * 4;
                if (e >= numel) continue;
                f32x4s gg = gv[it], mm = mv[it];
                const bool whole = e + 4 <= numel;
                uint32_t ub[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float u = gg[k];
                    if (has_m) {
                        mm[k] = S::rnd(lerp_torch(mm[k], gg[k], w));            // momentum.lerp_(grad, 1 - beta)
                        u = mm[k];
                        if (nesterov) u = gg[k] = S::rnd(lerp_torch(gg[k], mm[k], beta));   // grad.lerp_(momentum, beta)
                    }
                    ub[k] = f2bf(u);
                    if (whole || e + k < numel) {
                        const float uf = bf2f(static_cast<uint16_t>(ub[k]));
                        ss = fmaf(uf, uf, ss);
                    }
                }
                if (in_row) {          // (then every group of four is whole, and lies in one row)
                    if (wide) {
                        *reinterpret_cast<u32x2*>(X + at.r * pitch + at.c * 2) = u32x2{ub[0] | (ub[1] << 16), ub[2] | (ub[3] << 16)};
                    } else {
                        char* const p = X + at.c * pitch + at.r * 2;
#pragma unroll
                        for (int k = 0; k < 4; ++k) *reinterpret_cast<uint16_t*>(p + k * pitch) = static_cast<uint16_t>(ub[k]);
                    }
                } else {
                    int r = at.r, c = at.c;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        if (whole || e + k < numel)
                            *reinterpret_cast<uint16_t*>(wide ? X + r * pitch + c * 2 : X + c * pitch + r * 2) = static_cast<uint16_t>(ub[k]);
                        if (++c == cols) {
                            c = 0;
                            ++r;
                        }
                    }
                }
                if (aligned && whole) {
                    if (has_m) S::st4(mom + e, mm);
                    if (write_g) S::st4(g + e, gg);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (e + k < numel) {
                            if (has_m) S::st(mom + e + k, mm[k]);
                            if (write_g) S::st(g + e + k, gg[k]);
                        }
                }
            }
        }
        ss = wave_sum(ss);
        if ((tid & 63) == 0) sums[b * 4 + (t >> 6)] = ss;
    }
}

// The parameter step (muon.py:14, 98-99) from the result in LDS, 4 elements in a row per access.
template <typename T>
__device__ __forceinline__ void small_apply(const MuonMatDesc& d, const char* X, int pitch, bool wide, float neg_lr,
                                            float wd_factor, int tid) {
    typedef SmallIo<T> S;
    const int numel = d.rows * d.cols, cols = d.cols;
    T* const p = static_cast<T*>(d.param);
    uint16_t* const out = d.out;
    const bool aligned = small_aligned(p, S::kAlign) && small_aligned(out, 8);
    const bool in_row = (cols & 3) == 0;
    constexpr int UN = 2;
    Walk at(tid * 4, SMALL_THREADS * 4, cols);
    for (int e0 = tid * 4; e0 < numel; e0 += SMALL_THREADS * 4 * UN) {
        f32x4s pv[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int e = e0 + u * SMALL_THREADS * 4;
            pv[u] = f32x4s{0.f, 0.f, 0.f, 0.f};
            if (!p) continue;
            if (aligned && e + 4 <= numel) {
                pv[u] = S::ld4(p + e);
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (e + k < numel) pv[u][k] = S::ld(p + e + k);
            }
        }
#pragma unroll
        for (int u = 0; u < UN; ++u, at.next()) {
            const int e = e0 + u * SMALL_THREADS * 4;
            if (e >= numel) continue;
            float us[4];
            if (in_row && wide) {
                const u32x2 o = *reinterpret_cast<const u32x2*>(X + at.r * pitch + at.c * 2);
#pragma unroll
                for (int k = 0; k < 4; ++k) us[k] = (k & 1) ? bf_hi(o[k / 2]) : bf_lo(o[k / 2]);
            } else {
                int r = at.r, c = at.c;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    us[k] = 0.f;
                    if (e + k < numel)
                        us[k] = bf2f(*reinterpret_cast<const uint16_t*>(wide ? X + r * pitch + c * 2 : X + c * pitch + r * 2));
                    if (++c == cols) {
                        c = 0;
                        ++r;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                us[k] = round_bf(us[k] * d.scale);
                pv[u][k] = S::rnd(fmaf(neg_lr, us[k], S::rnd(pv[u][k] * wd_factor)));
            }
            if (aligned && e + 4 <= numel) {
                if (p) S::st4(p + e, pv[u]);
                if (out) *(__attribute__((address_space(1))) u32x2*)(out + e) = u32x2{pack2bf(us[0], us[1]), pack2bf(us[2], us[3])};
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (e + k < numel) {
                        if (p) S::st(p + e + k, pv[u][k]);
                        if (out) out[e + k] = f2bf(us[k]);
                    }
            }
        }
    }
}

// One matrix by one workgroup.  MP: its short side rounded up to 32, 64 or 128; the long side is rounded up to
// 64 (a k-block of the general path).  The products are shared out by 32 x 32 tiles of the Gram matrix and
// by blocks of 32 columns of X; X' overwrites X, whose columns depend on nothing but themselves and B.
template <int MP, bool ROUND>
__device__ __forceinline__ void small_matrix(char* lds, const MuonMatDesc& d, int steps, float ca, float cb, float cc, float w, float beta,
                                             int nesterov, int mutate_grad, float eps, float neg_lr, float wd_factor) {
    constexpr int MT = MP / 32, TILES = MT * MT, TPW = (TILES + SMALL_WAVES - 1) / SMALL_WAVES;
    constexpr int SYM_TILES = MT * (MT + 1) / 2, SPW = (SYM_TILES + SMALL_WAVES - 1) / SMALL_WAVES;
    constexpr bool KEEP_B = MP <= 64;                // (of the 128 registers a thread can have at 16 waves)
    constexpr int PA = small_pitch(MP);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int lane = tid & 63;
    const bool wide = d.rows <= d.cols;
    const int m = wide ? d.rows : d.cols, n = wide ? d.cols : d.rows;
    const int np = (n + 63) & ~63, px = small_pitch(np);
    float* const sums = reinterpret_cast<float*>(lds);
    char* const A = lds + SMALL_MAX_BLOCKS * 4 * sizeof(float);
    char* const B = A + MP * PA;                     // c A, then the polynomial
    char* const X = B + MP * PA;

    if (m < MP || n < np) {
        for (int o = tid * 16; o < MP * px; o += SMALL_THREADS * 16) *reinterpret_cast<u32x4*>(X + o) = u32x4{0u, 0u, 0u, 0u};
        __syncthreads();
    }
    if (d.src_dtype == MUON_AMD_SRC_BF16) small_load<uint16_t>(d, X, px, wide, w, beta, nesterov, mutate_grad, sums, tid);
    else small_load<float>(d, X, px, wide, w, beta, nesterov, mutate_grad, sums, tid);
    __syncthreads();
    float den;                                       // muon.py:282, as norm_finalize_kernel forms it
    {
        const int nblk = (d.rows * d.cols + SUM_BLOCK - 1) / SUM_BLOCK;
        const float* const q = sums + lane * 4;
        const float nrm = sqrtf(wave_sum(lane < nblk ? (q[0] + q[1]) + (q[2] + q[3]) : 0.f));
        den = ROUND ? round_bf(round_bf(nrm) + eps) : nrm + eps;
    }
    {
        const UniformDivisor by(den);
        const int chunks = np / 8;                   // of 8 columns
        Walk at(tid, SMALL_THREADS, chunks);
        for (; at.r < m; at.next()) {
            u32x4* const p = reinterpret_cast<u32x4*>(X + at.r * px + at.c * 16);
            const u32x4 v = *p;
            u32x4 o;                                 // (columns beyond n hold zero and stay zero)
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = pack2bf(by.divide(bf_lo(v[k])), by.divide(bf_hi(v[k])));
            if (!by.ok || UniformDivisor::tiny(v)) { // (an element is at most the norm: no quotient overflows)
#pragma unroll
                for (int k = 0; k < 4; ++k) o[k] = pack2bf(bf_lo(v[k]) / den, bf_hi(v[k]) / den);
            }
            if (at.c * 8 + 8 > n) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    o[k] &= (at.c * 8 + 2 * k < n ? 0xffffu : 0u) | (at.c * 8 + 2 * k + 1 < n ? 0xffff0000u : 0u);
            }
            *p = o;
        }
    }
    __syncthreads();

    for (int step = 0; step < steps; ++step) {
        asm volatile("" : "+v"(lane));               // LDS addresses are formed where they are used, not kept in registers
        // A = X X^T and, where the reference rounds it, c A: the tiles on and above the diagonal (X X^T is
        // symmetric bit for bit), each by one wave.  The reads of the next four k-steps are in flight under
        // the MFMAs of the current four; the rows of a diagonal tile are read once for both operands.
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
            const int t = wave + s * SMALL_WAVES;
            if (t >= SYM_TILES) continue;
            int ti = 0, tj = t;                      // diagonal tiles first, then the first off-diagonal, ...
            for (int len = MT; tj >= len; --len) tj -= len, ++ti;
            const int i0 = tj * 32, j0 = (tj + ti) * 32;
            const bool diag = ti == 0;
            f32x16 acc = zero16();
            if (diag) gram_tile<true>(acc, X, px, i0, j0, np / 16, lane);
            else gram_tile<false>(acc, X, px, i0, j0, np / 16, lane);
            uint32_t po[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) po[k] = pack2bf(acc[2 * k], acc[2 * k + 1]);
            tile_store(A, PA, i0, j0, lane, po);
            if (!diag) tile_store_mirrored(A, PA, i0, j0, lane, po);
            if constexpr (ROUND) {
#pragma unroll
                for (int k = 0; k < 8; ++k) po[k] = pack2bf(cc * bf_lo(po[k]), cc * bf_hi(po[k]));
                tile_store(B, PA, i0, j0, lane, po);
                if (!diag) tile_store_mirrored(B, PA, i0, j0, lane, po);
            }
        }
        __syncthreads();
        // B = b A + (c A) A
        uint32_t pb[TPW][8];
#pragma unroll
        for (int s = 0; s < TPW; ++s) {
            const int t = wave + s * SMALL_WAVES;
            if (t >= TILES) continue;
            const int i0 = t / MT * 32, j0 = t % MT * 32;
            f32x16 acc = zero16();
#pragma unroll
            for (int ks = 0; ks < MP / 16; ++ks)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(row_frag(A, PA, j0, ks, lane), row_frag(ROUND ? B : A, PA, i0, ks, lane), acc, 0, 0, 0);
            tile_load(pb[s], A, PA, i0, j0, lane);
            tile_add<ROUND>(pb[s], acc, ROUND ? 1.f : cc, cb);
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < TPW; ++s) {
            const int t = wave + s * SMALL_WAVES;
            if (t >= TILES) continue;
            tile_store(B, PA, t / MT * 32, t % MT * 32, lane, pb[s]);
        }
        __syncthreads();
        // X = a X + B X, a block of 32 columns at a time; the rows of B stay in registers where they fit
        bf16x8 bq[KEEP_B ? MT : 1][KEEP_B ? MP / 16 : 1];
        if constexpr (KEEP_B) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int ks = 0; ks < MP / 16; ++ks) bq[i][ks] = row_frag(B, PA, i * 32, ks, lane);
        }
        for (int j0 = wave * 32; j0 < np; j0 += SMALL_WAVES * 32) {
            bf16x8 q[MP / 16];
#pragma unroll
            for (int ks = 0; ks < MP / 16; ++ks) q[ks] = col_frag(X, px, j0, ks, lane);
#pragma unroll KEEP_B ? MT : 1
            for (int i = 0; i < MT; ++i) {
                f32x16 acc = zero16();
                uint32_t po[8];
                tile_load(po, X, px, i * 32, j0, lane);
#pragma unroll
                for (int ks = 0; ks < MP / 16; ++ks) {
                    const bf16x8 b = KEEP_B ? bq[KEEP_B ? i : 0][KEEP_B ? ks : 0] : row_frag(B, PA, i * 32, ks, lane);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(q[ks], b, acc, 0, 0, 0);
                }
                // (with one rounding the alpha of the general path is a run-time 1: beta * D is rounded before
                // the sum there, and must not be contracted into it here)
                float alpha = 1.f;
                if constexpr (!ROUND) asm volatile("" : "+s"(alpha));
                tile_add<ROUND>(po, acc, alpha, ca);
                tile_store(X, px, i * 32, j0, lane, po);
            }
        }
        __syncthreads();
    }
    if (d.src_dtype == MUON_AMD_SRC_BF16) small_apply<uint16_t>(d, X, px, wide, neg_lr, wd_factor, tid);
    else small_apply<float>(d, X, px, wide, neg_lr, wd_factor, tid);
}

// One workgroup per matrix, all of class MP at most, or (MP = 0) each in its own class: a launch per class takes at least
// what its longest matrix takes, one after the other, and the largest class for all of them pads the others.  32 x 2400,
// 16 of 64 x 64 and 4 of 128 x 300: 67 us, 136 in a launch per class, 100 on the general path; 2000 of 20 x 30 and one of
// 128 x 300: 100 us, 213 in class 128, 247 on the general path.  A class of its own is 1 to 6 % faster over many
// matrices than this kernel (1000 of 128 x 128: 149 against 159 us), so both are here.
template <int MP, bool ROUND>
__global__ __launch_bounds__(SMALL_THREADS) void ns_small_kernel(
    const MuonMatDesc* __restrict__ descs, int steps, float ca, float cb, float cc, float w, float beta, int nesterov,
    int mutate_grad, float eps, float neg_lr, float wd_factor, const float* __restrict__ sc) {
    extern __shared__ __align__(16) char lds[];
    if (sc) {   // {1 - beta, beta, lr, wd_factor} read at run time instead of the arguments
        w = sc[0];
        beta = sc[1];
        neg_lr = -sc[2];
        wd_factor = sc[3];
    }
    const MuonMatDesc d = descs[blockIdx.x];
    if constexpr (MP != 0) {
        small_matrix<MP, ROUND>(lds, d, steps, ca, cb, cc, w, beta, nesterov, mutate_grad, eps, neg_lr, wd_factor);
    } else {
        const int m = d.rows < d.cols ? d.rows : d.cols;
        if (m <= 32) small_matrix<32, ROUND>(lds, d, steps, ca, cb, cc, w, beta, nesterov, mutate_grad, eps, neg_lr, wd_factor);
        else if (m <= 64) small_matrix<64, ROUND>(lds, d, steps, ca, cb, cc, w, beta, nesterov, mutate_grad, eps, neg_lr, wd_factor);
        else small_matrix<128, ROUND>(lds, d, steps, ca, cb, cc, w, beta, nesterov, mutate_grad, eps, neg_lr, wd_factor);
    }
}

template <int MP, bool ROUND>
static int raise_small_limit() {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(ns_small_kernel<MP, ROUND>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            SMALL_LDS_MAX) != hipSuccess) {
        (void)hipGetLastError();
        set_error("small: cannot raise dynamic LDS to %d bytes", SMALL_LDS_MAX);
        return MUON_AMD_ELAUNCH;
    }
    return MUON_AMD_OK;
}

int raise_small_limits() {
    int rc = raise_small_limit<0, true>();
    if (rc == MUON_AMD_OK) rc = raise_small_limit<0, false>();
    if (rc == MUON_AMD_OK) rc = raise_small_limit<32, true>();
    if (rc == MUON_AMD_OK) rc = raise_small_limit<32, false>();
    if (rc == MUON_AMD_OK) rc = raise_small_limit<64, true>();
    if (rc == MUON_AMD_OK) rc = raise_small_limit<64, false>();
    if (rc == MUON_AMD_OK) rc = raise_small_limit<128, true>();
    if (rc == MUON_AMD_OK) rc = raise_small_limit<128, false>();
    return rc;
}

}  // namespace muon_amd

using namespace muon_amd;

extern "C" {

int muon_amd_small_class(int rows, int cols) {
    if (rows <= 0 || cols <= 0) return 0;
    const int m = rows < cols ? rows : cols;
    const int64_t n = rows < cols ? cols : rows;
    const int mp = m <= 32 ? 32 : m <= 64 ? 64 : m <= 128 ? 128 : 0;
    if (!mp || n > 65536 || (static_cast<int64_t>(rows) * cols + SUM_BLOCK - 1) / SUM_BLOCK > SMALL_MAX_BLOCKS) return 0;
    return small_lds_bytes(mp, static_cast<int>((n + 63) & ~63)) <= SMALL_LDS_MAX ? mp : 0;
}

int muon_amd_validate_small(const MuonMatDesc* descs, int nmat, int small_class, int max_long_side) {
    MUON_REQUIRE(descs && nmat > 0, "validate_small: nmat=%d", nmat);
    for (int i = 0; i < nmat; ++i) {
        const MuonMatDesc& d = descs[i];
        const int own = muon_amd_small_class(d.rows, d.cols);
        MUON_REQUIRE(own && (own <= small_class || small_class == 0) && (d.rows > d.cols ? d.rows : d.cols) <= max_long_side,
                     "mat %d: %d x %d does not fit class %d with a long side of %d", i, d.rows, d.cols, small_class, max_long_side);
        MUON_REQUIRE(d.grad && (d.param || d.out), "mat %d: null source or neither param nor out given", i);
        MUON_REQUIRE(d.src_dtype == MUON_AMD_SRC_F32 || d.src_dtype == MUON_AMD_SRC_BF16, "mat %d: src_dtype=%d", i, d.src_dtype);
    }
    return MUON_AMD_OK;
}

int muon_amd_small_step(const MuonMatDesc* descs_dev, int nmat, int small_class, int max_long_side, int steps,
                        const float* coeffs, int flags, float one_minus_beta, float beta, int nesterov, int mutate_grad,
                        float eps, float lr, float wd_factor, const float* scalars_dev, void* stream) {
    MUON_REQUIRE(descs_dev && coeffs, "small_step: null table");
    MUON_REQUIRE(nmat > 0 && steps >= 0, "small_step: nmat=%d steps=%d", nmat, steps);
    MUON_REQUIRE(small_class == 0 || small_class == 32 || small_class == 64 || small_class == 128, "small_step: class %d", small_class);
    MUON_REQUIRE(max_long_side > 0 && max_long_side <= 65536, "small_step: long side %d", max_long_side);
    // (classes mixed: as much as any matrix can need; a CU holds one workgroup of 16 waves in any case)
    const size_t bytes = small_class ? small_lds_bytes(small_class, (max_long_side + 63) & ~63) : SMALL_LDS_MAX;
    MUON_REQUIRE(bytes <= SMALL_LDS_MAX, "small_step: a long side of %d does not fit", max_long_side);
    const int rc = muon_amd_init();
    if (rc != MUON_AMD_OK) return rc;
    const auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(nmat), dim3(SMALL_THREADS), bytes, static_cast<hipStream_t>(stream), descs_dev, steps,
                           coeffs[0], coeffs[1], coeffs[2], one_minus_beta, beta, nesterov, mutate_grad, eps, -lr, wd_factor,
                           scalars_dev);
    };
    const bool round = (flags & MUON_AMD_ROUND_REFERENCE) != 0;
    if (small_class == 0) round ? go(ns_small_kernel<0, true>) : go(ns_small_kernel<0, false>);
    else if (small_class == 32) round ? go(ns_small_kernel<32, true>) : go(ns_small_kernel<32, false>);
    else if (small_class == 64) round ? go(ns_small_kernel<64, true>) : go(ns_small_kernel<64, false>);
    else round ? go(ns_small_kernel<128, true>) : go(ns_small_kernel<128, false>);
    return check_launch("small_step");
}

}  // extern "C"
