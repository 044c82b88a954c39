// Regularised normal equations (Z^T Z + lambda I) alpha = Z^T y: fp64 Cholesky factorisation
// A = U^T U of the symmetric positive definite matrix, in place in the upper triangle, and the
// two triangular solves.  The reference calls torch.linalg.solve (LU) at this point
// (qml_lightning/models/kernel.py:226-234).
//
// Row-major A with row stride ld, 128-column blocks grouped in panels of 512 rows.  Per block k:
//   1. the block's 128 rows (columns k..F) take the product of the panel's rows above them
//      (fp64 MFMA tile product, depth up to 384);
//   2. one workgroup factors the 128x128 diagonal block in registers and also produces the
//      inverse of the factor (both orientations, kept for the solves);
//   3. U12 = U11^-T A12 as a product with that inverse on the same MFMA tiles.
// After a panel, the trailing matrix takes A22 -= U12^T U12 (512 rows deep) on the tiles on or
// above the diagonal.  The depth of 512 is what makes the trailing update MFMA-bound: at a
// depth of 128 the read-modify-write of the trailing matrix dominates.
// For whole tiles (F a multiple of 128) a panel and the trailing update of the panel before it are ONE
// launch (panel_kernel below); any other F takes a launch per step with the tile kernel of gram.hip. A caller
// that copies the matrix anyway pads it to whole tiles (qmll_copy_upper_padded_f64): 704 features 633 -> 348 us.
// Only elements on or above the diagonal are read; below the diagonal only the lower halves of
// the 128x128 diagonal tiles are overwritten.  Flops: F^3/3.  Large matrices take the updates by all rows
// but the last few thousand from the int8 matrix cores (slab_end below).
#include <algorithm>
#include <type_traits>
#include <utility>

#include "qmll_common.h"
#include "gram_tiles.h"

// gram.hip: tiles on/above the diagonal of C[n,n] (row stride ldc) += sign * Z^T Z, Z = M rows
// of n columns with row stride ldz
int qmll_internal_syrk_upper(const double* Z, int M, int n, long long ldz, double* C, long long ldc, double sign,
                             hipStream_t stream);
// gram_modular.hip: a slab of `rows` rows of the factor and the n columns from its first diagonal entry on (A): scales, the
// residues of rows that are final, the update of what is behind i0 by the slab's first k rows
size_t qmll_internal_slab_bytes(int rows, int n);
int qmll_internal_slab_begin(const double* A, long long ld, int rows, int n, void* workspace, const char* who, hipStream_t stream);
int qmll_internal_slab_rows(const double* A, long long ld, int rows, int n, int k0, int m, int f0, void* workspace, const char* who,
                            hipStream_t stream);
int qmll_internal_slab_update(double* A, long long ld, int rows, int n, int k, int i0, int band, void* workspace, const char* who,
                              hipStream_t stream);

// gram.hip: C[ra,n] = or += sign * Za^T Zb, Za = M x ra (row stride lda), Zb = M x n (row stride ldb)
int qmll_internal_gemm_tn(const double* Za, long long lda, int ra, const double* Zb, long long ldb, int n, int M,
                          double* C, long long ldc, double sign, int overwrite, hipStream_t stream);

namespace {

constexpr int NB = 128;       // block edge
constexpr int OB = 512;       // panel depth of the trailing update
constexpr int PT = 512;           // threads of a factorisation workgroup (and of the tile product's eight wavefronts)
constexpr int SB = 16;            // sub-block edge of the diagonal-block factorisation (one fp64 MFMA tile)
constexpr int NSB = NB / SB;      // sub-blocks per edge
constexpr int NSUB = NSB * (NSB + 1) / 2;     // sub-blocks on or above (or on or below) the diagonal
constexpr int MWAVES = PT / 64 - 2;           // wavefronts that hold sub-blocks; wavefront 0 factors the diagonal ones
constexpr int NSLOT = (2 * NSUB + MWAVES - 1) / MWAVES;
constexpr int SSTRIDE = NB + 16;  // doubles per row of a 16-row strip in LDS (rows 32 banks apart, see gram.hip)
constexpr int DSTRIDE = SB + 1;

typedef double double4_t __attribute__((ext_vector_type(4)));

// LDS of the diagonal-block factorisation, 41 KB
struct PotrfShared {
    double ustrip[SB][SSTRIDE];   // block row K of U
    double wstrip[SB][SSTRIDE];   // block row K of W = L^-1
    double dblk[SB][DSTRIDE];     // the diagonal sub-block about to be factored
    double vblk[SB][DSTRIDE];     // the inverse of its factor
    int failed;
};

__device__ __forceinline__ double value_of_lane(double v, int lane) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Sub-block t of the list the wavefronts 1, 2, 3, 5, 6, 7 are dealt their register slots from (the w-th of them holds
// t = 6 s + w - 1 in slot s): first the 36 sub-blocks of S on or above the diagonal, row by row, then the
// 36 of W on or below it.  kind 0: S, 1: W.
struct SubId {
    int kind, i, j;
};
constexpr SubId sub_id(int t) {
    SubId b{t >= NSUB ? 1 : 0, 0, 0};
    int u = b.kind ? t - NSUB : t;
    if (!b.kind) {
        while (u >= NSB - b.i) { u -= NSB - b.i; ++b.i; }
        b.j = b.i + u;
    } else {
        while (u >= b.i + 1) { u -= b.i + 1; ++b.i; }
        b.j = u;
    }
    return b;
}

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>); the second form stops at the first false
template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}
template <class F, int... Is>
__device__ __forceinline__ bool static_all_impl(F& f, std::integer_sequence<int, Is...>) {
    return (f(std::integral_constant<int, Is>{}) && ...);
}
template <int N, class F>
__device__ __forceinline__ bool static_all(F&& f) {
    return static_all_impl(f, std::make_integer_sequence<int, N>{});
}

// Factor the nb x nb block at (k0,k0) (nb <= 128; the rest is padded with the identity) and invert the factor.
// Blocked right-looking Cholesky on 16 x 16 sub-blocks, S = U^T U, with the same block operations applied to
// the identity: W = L^-1 = U^-T.  The sub-blocks live in registers in the accumulator layout of
// v_mfma_f64_16x16x4_f64 (register r of a lane: row lane/16 + 4r, column lane%16), which is also the layout
// of both operands (row = the summed index), so a sub-block feeds the matrix pipe as it stands.  Six wavefronts
// hold the 72 sub-blocks, twelve each; which ones is fixed at compile time (one instance of the code
// per wavefront), so a finished sub-block's registers are free again and no index is computed at run time.
// Wavefront 4 has none: it shares its SIMD with wavefront 0, whose fp64 arithmetic waits for matrix instructions there (dealt to
// seven wavefronts a block in a launch of its own takes 35.6 us, to six 33.5; 2048 features 1.335 and 1.305 ms).
// Wavefront 0 holds none and does the serial part.  Step K of eight:
//   1. the owner of S(K,K) puts it into LDS; wavefront 0 factors it, a lane per column: sixteen pivots, each
//      a reciprocal square root and the pivot row handed round with v_readlane, no barrier and no LDS inside;
//      the same row operations on the identity give V = U_KK^-1;
//   2. block row K: U(K,J) = V^T S(K,J), W(K,J) = V^T W(K,J), four MFMAs each, to LDS and to memory;
//   3. S(I,J) -= U(K,I)^T U(K,J) and W(I,J) -= U(K,I)^T W(K,J) for the rows I > K: S(K+1,K+1) at once, the others
//      beside step 1 of K + 1, which waits for that one only (a 128 x 128 block in a launch of its own took 45.5 us with all of them before it, 40.4 so).
// 24 barriers instead of the 128 of an elimination pivot by pivot, and the multiply-adds on the matrix pipe.
// Output: upper triangle of the block <- U11; inv[m*128+i] = U11^-1[m,i] = W[i,m]; invT[i*128+m] the same.
// info: 0, or 1 + the index of the first pivot that is not positive (later launches then exit).

// Stores and loads past the caches of this XCD, whose L2 the others do not see: no fence, which would write a whole L2 back or
// drop it, is needed beside them.
__device__ __forceinline__ void store_past_caches(double* p, double v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_past_caches(unsigned* p, unsigned v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double load_past_caches(const double* p) {
    return __longlong_as_double((long long)__hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT));
}

// inv[m, 16 K + i] = W[16 K + i, m] for the columns m of block row K, from the strip in LDS: thread = (m, half a
// row of sixteen), 64 contiguous bytes each.  Wavefronts 4..7: 0 is the one that is waited for.
__device__ __forceinline__ void store_inverse_columns(int K, double* inv, const PotrfShared& ps) {
    const int m = ((int)threadIdx.x - PT / 2) >> 1, half = (int)threadIdx.x & 1;
    if (m >= 0 && m < (K + 1) * SB) {
#pragma unroll
        for (int q = 0; q < SB / 2; ++q) inv[m * NB + K * SB + half * (SB / 2) + q] = ps.wstrip[half * (SB / 2) + q][m];
    }
}

// wavefront 0: the diagonal sub-blocks, one after the other
__device__ __forceinline__ bool potrf_factor_wave(double* blk, long long ld, int k0, int nb, double* inv, int* info,
                                                  PotrfShared& ps) {
    const int lane = (int)threadIdx.x & 63, l16 = lane & 15;
    for (int K = 0; K < NSB; ++K) {
        __syncthreads();                                               // S(K,K) is in LDS
        // lanes 0..15: column l16 of the sub-block; the others: row l16 of V, which takes the same row operations
        double v[SB];
#pragma unroll
        for (int i = 0; i < SB; ++i) v[i] = lane < SB ? ps.dblk[i][l16] : i == l16 ? 1.0 : 0.0;
        int bad = -1;                                                  // the first pivot that is not positive
#pragma unroll
        for (int j = 0; j < SB; ++j) {
            double piv = value_of_lane(v[j], j);                       // the same value in every lane
            if (!(piv > 0.0)) {
                bad = bad < 0 ? j : bad;
                piv = 1.0;
            }
            // 1/sqrt by the hardware estimate and two Newton steps
            double y = __builtin_amdgcn_rsq(piv);
            const double h = 0.5 * piv;
            y = fma(y, fma(-h * y, y, 0.5), y);
            y = fma(y, fma(-h * y, y, 0.5), y);
            const double u = v[j] * y;                                 // U[j, l16], W[j, l16]
            v[j] = u;
#pragma unroll
            for (int i0 = j + 1; i0 < SB; i0 += 4) {                   // four multipliers at a time, or each multiply-add
                // waits for its own (a block 33.5 us, 32.1 so; 2048 features 1.305 and 1.284 ms)
                double m[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) m[q] = i0 + q < SB ? value_of_lane(u, i0 + q) : 0.0;     // U[j, i] = L[i, j]
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (i0 + q < SB) v[i0 + q] = fma(-m[q], u, v[i0 + q]);
                // pins the updates to this step (no instruction is emitted): left alone the compiler carries multipliers in scalar
                // registers that it does not have
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (i0 + q < SB) asm volatile("" : "+v"(v[i0 + q]));
            }
        }
        if (bad >= 0 && lane == 0) {
            *info = k0 + K * SB + bad + 1;
            ps.failed = 1;
        }
        if (lane >= SB) {                                              // (the three copies write the same values)
#pragma unroll
            for (int i = 0; i < SB; ++i) ps.vblk[l16][i] = v[i];       // V[c, i] = W[i, c]
        }
        __syncthreads();                                               // V is in LDS
        if (ps.failed) return false;
#pragma unroll
        for (int i = 0; i < SB; ++i) {
            const int row = K * SB + i, col = K * SB + l16;
            if (lane < SB && i <= l16 && col < nb) blk[(size_t)row * ld + col] = v[i];
        }
        __syncthreads();                                               // block row K is in LDS
    }
    return true;
}

// wavefront 4, which shares its SIMD with wavefront 0: no matrix instructions.  It writes the columns of the inverse, and block row K of U
// right of the diagonal and the diagonal sub-block of the inverse past the caches, for the workgroups that follow this factorisation step
// by step (follow_block): *steps is the number of block rows that are there.  (Nobody does where steps is null: the wavefronts that work
// them out then store both; 704 features in launches of their own 659 us with the detour, 630 so.)  All of a step's stores are this wavefront's, so that waiting
// for them is all the order they need.
__device__ __forceinline__ bool potrf_store_wave(double* blk, long long ld, int nb, double* inv, double* invT, unsigned* steps,
                                                 PotrfShared& ps) {
    const int lane = (int)threadIdx.x & 63;
    auto done = [&](unsigned count) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (lane == 0) store_past_caches(steps, count);
    };
    for (int K = 0; K < NSB; ++K) {
        __syncthreads();                                               // S(K,K) is in LDS
        if (K > 0) {
            if (steps) {
                const int row0 = (K - 1) * SB;
#pragma unroll 4
                for (int r = 0; r < SB; ++r)
                    for (int col = K * SB + lane; col < nb; col += QMLL_WAVE)
                        if (row0 + r < nb) store_past_caches(&blk[(size_t)(row0 + r) * ld + col], ps.ustrip[r][col]);
                done((unsigned)K);
            }
            store_inverse_columns(K - 1, inv, ps);
        }
        __syncthreads();                                               // V is in LDS
        if (ps.failed) return false;
        if (steps) {
#pragma unroll
            for (int e = lane; e < SB * SB; e += QMLL_WAVE)            // W(K,K) = V^T
                store_past_caches(&invT[(K * SB + e / SB) * NB + K * SB + e % SB], ps.vblk[e % SB][e / SB]);
            if (K == NSB - 1) done(NSB);
        }
        __syncthreads();                                               // block row K is in LDS
    }
    store_inverse_columns(NSB - 1, inv, ps);
    return true;
}

// the WV-th (1..6) of the wavefronts 1, 2, 3, 5, 6, 7: its share of the sub-blocks
template <int WV>
__device__ __forceinline__ bool potrf_mfma_wave(double* blk, long long ld, int nb, double* inv, double* invT,
                                                bool handed_out, PotrfShared& ps) {
    const int lane = (int)threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4;
    const int ldi = (int)ld;
    // per-lane parts of every address; what is added per sub-block is a constant
    double* const blk_lane = blk + (size_t)lk * ld + l16;
    double* const invT_lane = invT + lk * NB + l16;
    double* const us_lane = &ps.ustrip[lk][l16];
    double* const ws_lane = &ps.wstrip[lk][l16];
    double4_t sub[NSLOT];
    static_for<NSLOT>([&](auto s_) {
        constexpr int s = decltype(s_)::value, t = s * MWAVES + WV - 1;
        if constexpr (t < 2 * NSUB) {
            constexpr SubId b = sub_id(t);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = b.i * SB + lk + 4 * r, col = b.j * SB + l16;
                if constexpr (b.kind == 0) {
                    const int lo = row < col ? row : col, hi = row < col ? col : row;
                    // (32-bit offsets: 128 rows of at most 2^23 doubles)
                    sub[s][r] = hi < nb ? blk[(unsigned)(lo * ldi + hi)] : (row == col ? 1.0 : 0.0);
                } else {
                    sub[s][r] = row == col ? 1.0 : 0.0;
                }
            }
        }
    });
    // the diagonal sub-block K goes to wavefront 0
    auto hand_diagonal = [&](auto K_) {
        constexpr int K = decltype(K_)::value;
        static_for<NSLOT>([&](auto s_) {
            constexpr int s = decltype(s_)::value, t = s * MWAVES + WV - 1;
            if constexpr (t < 2 * NSUB) {
                constexpr SubId b = sub_id(t);
                if constexpr (b.kind == 0 && b.i == K && b.j == K) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) ps.dblk[lk + 4 * r][l16] = sub[s][r];
                }
            }
        });
    };
    // the update by block row K of the next diagonal sub-block (only) or of all others
    auto update = [&](auto K_, auto diagonal_) {
        constexpr int K = decltype(K_)::value;
        static_for<NSLOT>([&](auto s_) {
            constexpr int s = decltype(s_)::value, t = s * MWAVES + WV - 1;
            if constexpr (t < 2 * NSUB) {
                constexpr SubId b = sub_id(t);
                constexpr bool next = b.kind == 0 && b.i == K + 1 && b.j == K + 1;
                if constexpr (b.i > K && (b.kind == 0 || b.j <= K) && next == decltype(diagonal_)::value) {
                    const double* right = b.kind == 0 ? us_lane : ws_lane;
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk) {
                        const double fa = -us_lane[4 * kk * SSTRIDE + b.i * SB];
                        const double fb = right[4 * kk * SSTRIDE + b.j * SB];
                        sub[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa, fb, sub[s], 0, 0, 0);
                    }
                }
            }
        });
    };
    hand_diagonal(std::integral_constant<int, 0>{});
    return static_all<NSB>([&](auto K_) -> bool {
        constexpr int K = decltype(K_)::value;
        __syncthreads();                                               // S(K,K) is in LDS
        if constexpr (K > 0) {                                         // beside wavefront 0: what it does not wait for
            update(std::integral_constant<int, K - 1>{}, std::false_type{});
            store_inverse_columns(K - 1, inv, ps);
        }
        __syncthreads();                                               // wavefront 0 has factored it: V is in LDS
        if (ps.failed) return false;
        double va[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) va[kk] = ps.vblk[4 * kk + lk][l16];
        static_for<NSLOT>([&](auto s_) {
            constexpr int s = decltype(s_)::value, t = s * MWAVES + WV - 1;
            if constexpr (t < 2 * NSUB) {
                constexpr SubId b = sub_id(t);
                if constexpr (b.i == K && (b.kind == 1 || b.j > K)) {
                    double4_t res = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk)
                        res = __builtin_amdgcn_mfma_f64_16x16x4f64(va[kk], sub[s][kk], res, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if constexpr (b.kind == 0) {
                            us_lane[4 * r * SSTRIDE + b.j * SB] = res[r];
                            if (!handed_out && b.j * SB + l16 < nb && K * SB + lk + 4 * r < nb)
                                blk_lane[(size_t)(K * SB + 4 * r) * ld + b.j * SB] = res[r];
                        } else {
                            ws_lane[4 * r * SSTRIDE + b.j * SB] = res[r];
                            if (b.j < K || !handed_out) invT_lane[(K * SB + 4 * r) * NB + b.j * SB] = res[r];
                        }
                    }
                }
            }
        });
        __syncthreads();                                               // block row K is in LDS
        if constexpr (K + 1 < NSB) {
            update(K_, std::true_type{});
            hand_diagonal(std::integral_constant<int, K + 1>{});
        } else {
            store_inverse_columns(K, inv, ps);
        }
        return true;
    });
}

// Called by all PT threads of the workgroup.  False when a pivot is not positive (info is then set).
// HANDED_OUT: step by step, with the number of steps in *steps.
template <bool HANDED_OUT>
__device__ __forceinline__ bool potrf_block(double* A, long long ld, int k0, int nb, double* inv, double* invT,
                                            int* info, unsigned* steps, PotrfShared& ps) {
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    double* blk = A + (size_t)k0 * ld + k0;
    // the sub-blocks of inv / invT that stay zero (the others are written when their block row is final)
    for (int e = tid; e < (NSUB - NSB) * SB * SB; e += PT) {
        int b = e / (SB * SB), I = 0;
        const int r = (e / SB) % SB, c = e % SB;
        while (b >= NSB - 1 - I) { b -= NSB - 1 - I; ++I; }
        const int J = I + 1 + b;                                  // I < J
        invT[(I * SB + r) * NB + J * SB + c] = 0.0;
        inv[(J * SB + r) * NB + I * SB + c] = 0.0;
    }
    if (tid == 0) ps.failed = 0;
    bool ok;
    switch (wave) {
        case 0: ok = potrf_factor_wave(blk, ld, k0, nb, inv, info, ps); break;
        case 1: ok = potrf_mfma_wave<1>(blk, ld, nb, inv, invT, HANDED_OUT, ps); break;
        case 2: ok = potrf_mfma_wave<2>(blk, ld, nb, inv, invT, HANDED_OUT, ps); break;
        case 3: ok = potrf_mfma_wave<3>(blk, ld, nb, inv, invT, HANDED_OUT, ps); break;
        case 4: ok = potrf_store_wave(blk, ld, nb, inv, invT, HANDED_OUT ? steps : nullptr, ps); break;
        case 5: ok = potrf_mfma_wave<4>(blk, ld, nb, inv, invT, HANDED_OUT, ps); break;
        case 6: ok = potrf_mfma_wave<5>(blk, ld, nb, inv, invT, HANDED_OUT, ps); break;
        default: ok = potrf_mfma_wave<6>(blk, ld, nb, inv, invT, HANDED_OUT, ps); break;
    }
    if (!ok) return false;                                        // every wavefront saw the same flag
    __syncthreads();
    return true;
}

__global__ __launch_bounds__(PT, 4) void potrf_block_kernel(double* A, long long ld, int k0, int nb, double* inv,
                                                         double* invT, int* info) {
    __shared__ PotrfShared ps;
    if (*info != 0) return;
    potrf_block<false>(A, ld, k0, nb, inv, invT, info, nullptr, ps);
}

// ---- one launch per panel -------------------------------------------------------------------
//
// Steps 1-3 above are eleven dependent launches per panel, each of at most F/128 workgroups and a few
// tens of microseconds, and the trailing update that follows has to wait for them.  For whole 128-column
// tiles a panel is one launch instead, and that launch also carries the trailing update of the panel
// before it.
//
// The chain.  Workgroup b < 4 owns block column b of the panel.  It first gives its tiles the update of the previous panel (rows
// R0 .. P0 of the factor, already final: the part of that panel's trailing update that falls into this panel's rows), then, for each
// block l < b, follows the factorisation of block l on its CU step by step (follow_block): the strip (l, b) and the update of
// its own diagonal tile are done a step after the factorisation is.  Then it factors its diagonal tile and publishes the inverse.
//     for l < b:  wait for "tile (l, b) has its updates";  follow block l;  publish "strip (l, b)"
//     factor block b, handing out its block rows as they are done;  publish "block b factored"
// The updates of the panel's tiles beside its diagonal, tile (b, w) -= strip(l, b)^T strip(l, w), stand between one factorisation and the next
// but one, so that four workgroups each take a quarter of such a tile.  These owners and quarters wait for each other: they are the first
// workgroups behind the head tiles (sixteen, of a CU each), so that all of them are resident before any other of the launch.
// us per solve before this chain (strip and updates behind the whole block's inverse, a workgroup to a column of tiles) and with it: 512
// features 260 / 186, 2048 1281 / 951, 4096 2800 / 2048, 8192 6900 / 5560, 16384 22030 / 19950, 24576 51460 / 48520.  A block of the chain takes 44 us,
// 68 before, 30 of them its factorisation.  With 151 to 166 registers a workgroup has a CU to itself; held to the 128 of two the
// followers spilled (51 us a block), and nothing else gained from the second.
//
// Column owners.  One or two workgroups own a column of tiles (or half of it) of the panel's rows right of the panel:
//     first the update of the previous panel, as above;  then for l = 0 .. 3:
//     wait for "block l factored";  tile(l, w) = U11_l^-T tile(l, w)                      row strip
//     for the block rows b > l:  wait for "strip (l, b) done";  tile(b, w) -= strip(l, b)^T tile(l, w)
// They wait for lower workgroup ids only.  Every wait is bounded; one that runs out sets info to -1 and the workgroup leaves, and as every
// wait looks at info now and then the others leave behind it.  (The look is kept off the way that the chain takes, and setting the flags that the
// workgroup still owes is not worth it: either took 16384 features 0.3 to 0.6 % longer.  Waiting polls with
// relaxed loads: with an acquire at each poll the waiting owners kept emptying the L2 of those at work, a panel of 120 columns 326 us, 280 so.)
//
// Head tiles.  Once the trailing matrix is small a launch lasts as long as its slowest owner, and four of an
// owner's fourteen tile products are that first update.  The host then puts workgroups for those tiles in
// front of the owners (one per tile, waiting for nobody); each counts itself into its column's counter
// when done, and an owner starts by waiting for its column's count.
//
// Trailing tiles.  The workgroups after the owners (their count rounded up to a multiple of eight, so
// that the XCD of a tile is what gram_tiles.h deals) take the previous panel's update of the tiles
// on or above the diagonal below this panel, 512 deep, and wait for nobody.  While the panel's chain of
// dependent steps (four factorisations, each waiting for the strip before it) runs on a few CUs, the rest
// of the chip is busy with these.
constexpr int PKB = 16;                 // rows staged per step
constexpr int PSTRIDE = NB + 16;        // doubles per staged row (see gram.hip)
constexpr int P_TPR = PT / PKB;         // threads per staged row
constexpr int P_CPT = NB / P_TPR;       // doubles per thread and row
constexpr int P_UN = P_CPT / 2;         // 16-byte units per thread
constexpr unsigned FLAG_DONE = 1u, FLAG_FAILED = 0x80000000u;   // (a counter never gets near the second)
constexpr int PBLK = OB / NB;                        // blocks per panel
// "block l factored": [l]; "strip (l, b) done": [PBLK + l PBLK + b]; block rows of block l that are there: [STEPS + l]; quarters of updates
// that tile (b, w) of the panel's own columns has had: [QUARTERS + b PBLK + w]
constexpr int STEPS = PBLK + PBLK * PBLK, QUARTERS = STEPS + PBLK, FLAGS_PER_PANEL = QUARTERS + PBLK * PBLK;
constexpr int CUS = 256;
constexpr int SPLIT_HEADS_BELOW = 48;       // trailing tiles per edge
constexpr unsigned SPIN_LIMIT = 1u << 21;   // polls of about a microsecond each before a wait gives up

typedef double double2_t __attribute__((ext_vector_type(2)));

struct TileShared {
    double a[2][PKB][PSTRIDE], b[2][PKB][PSTRIDE];
};

constexpr int TRIANGULAR = 1;
// The 128 x COLS tile at C (row stride ldc) = or += sign * Za^T Zb, Za `depth` rows (a multiple of 32) of 128
// columns, Zb of COLS; the tile product of gram.hip for whole tiles (same staging, same MFMA order).  C may be Zb
// (depth 128, overwrite): everything is read before anything is written.  Ends with a barrier.
// TRIANGULAR: Za[m][i] = 0 for m > i (the inverse of a diagonal block), whose 16 x 16 sub-blocks below the diagonal are left out:
// 36 of 64 remain.
template <int COLS, int MODE = 0>
__device__ __forceinline__ void tile_product(const double* Za, long long lda, const double* Zb, long long ldb,
                                             int depth, double* C, long long ldc, double sign, bool overwrite,
                                             TileShared& sm) {
    static_assert(COLS == NB || COLS == NB / 2, "whole tiles or their halves");
    constexpr int P = COLS == NB ? 4 : 2;                          // sub-blocks of a wavefront one below the other (two beside each other)
    constexpr int B_CPT = COLS / P_TPR, B_UN = B_CPT / 2;
    constexpr int AHEAD = COLS == NB ? 1 : 2;                      // steps on the way
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);     // (uniform: a matrix instruction takes no lane mask)
    const int wj = (COLS == NB ? wave & 3 : wave & 1) * 32;
    // first row of sub-block p: in half a tile a wavefront has rows from both ends, which makes their work on a triangle equal
    auto wi = [&](int p) { return COLS == NB ? (wave / 4) * 64 + p * 16 : (p == 0 ? wave / 2 : NSB - 1 - wave / 2) * 16; };
    const int l16 = lane & 15, lk = lane >> 4;
    double4_t acc[P][2];
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[p][q] = (double4_t){0.0, 0.0, 0.0, 0.0};
    const int lr = tid / P_TPR, lc = (tid % P_TPR) * P_CPT, lcb = (tid % P_TPR) * B_CPT;
    double2_t ra[AHEAD][P_UN], rb[AHEAD][B_UN];
    auto load_panels = [&](int m0, double2_t (&ta)[P_UN], double2_t (&tb)[B_UN]) {
        const double2_t* pa = reinterpret_cast<const double2_t*>(Za + (size_t)(m0 + lr) * lda + lc);
        const double2_t* pb = reinterpret_cast<const double2_t*>(Zb + (size_t)(m0 + lr) * ldb + lcb);
#pragma unroll
        for (int q = 0; q < P_UN; ++q) ta[q] = pa[q];
#pragma unroll
        for (int q = 0; q < B_UN; ++q) tb[q] = pb[q];
    };
    const int nsteps = depth / PKB;
    auto one_step = [&](int step, int cur, double2_t (&ta)[P_UN], double2_t (&tb)[B_UN]) {
        double2_t* da = reinterpret_cast<double2_t*>(&sm.a[cur][lr][lc]);
        double2_t* db = reinterpret_cast<double2_t*>(&sm.b[cur][lr][lcb]);
#pragma unroll
        for (int q = 0; q < P_UN; ++q) da[q] = ta[q];
#pragma unroll
        for (int q = 0; q < B_UN; ++q) db[q] = tb[q];
        __syncthreads();
        if (step + AHEAD < nsteps) load_panels((step + AHEAD) * PKB, ta, tb);   // in flight during the MFMAs
        if constexpr (MODE == 0) {
#pragma unroll
            for (int kk = 0; kk < PKB; kk += 4) {
                double fa[P], fb[2];
#pragma unroll
                for (int p = 0; p < P; ++p) fa[p] = sm.a[cur][kk + lk][wi(p) + l16];
#pragma unroll
                for (int q = 0; q < 2; ++q) fb[q] = sm.b[cur][kk + lk][wj + q * 16 + l16];
#pragma unroll
                for (int p = 0; p < P; ++p)
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                        acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[p], fb[q], acc[p][q], 0, 0, 0);
            }
        } else {
            double fb[2][4];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int k = 0; k < 4; ++k) fb[q][k] = sm.b[cur][4 * k + lk][wj + q * 16 + l16];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                if (step * PKB > wi(p)) continue;                                // rows of zeros
                double fa[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) fa[k] = sm.a[cur][4 * k + lk][wi(p) + l16];
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int k = 0; k < 4; ++k) acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[k], fb[q][k], acc[p][q], 0, 0, 0);
            }
        }
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) load_panels(u * PKB, ra[u], rb[u]);
#pragma unroll 1
    for (int step = 0; step < nsteps; step += AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) one_step(step + u, AHEAD == 1 ? step & 1 : u, ra[u], rb[u]);
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                double* c = C + (size_t)(wi(p) + lk + 4 * r) * ldc + wj + q * 16 + l16;
                const double v = sign * acc[p][q][r];
                // (the sum is left to the memory side: no wait for the old value; every element of C takes its
                // additions in one order, so the result does not depend on any)
                if (overwrite) *c = v;
                else unsafeAtomicAdd(c, v);
            }
    __syncthreads();
}

// every store of the workgroup so far becomes visible to the device, then the flag is set / counted up
// (one wavefront writes the L2 back, when the stores of all of them have reached it: not 0, which the factorisation that may come next waits
// for)
__device__ __forceinline__ void publish(unsigned* flag, unsigned value) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == PT / 2) __hip_atomic_store(flag, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish_one_more(unsigned* counter) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until the word is at least `target` and returns it; a wait that runs out sets info to -1 and
// returns FLAG_FAILED.  So does one that finds, every 64 polls, that info is set: what it waits for may never come then.
__device__ __forceinline__ unsigned await(unsigned* flag, unsigned target, unsigned spin_limit, int* info,
                                          unsigned& seen) {
    if (threadIdx.x == 0) {
        unsigned v = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (unsigned n = 0; v < target && n < spin_limit; ++n) {
            __builtin_amdgcn_s_sleep(32);
            v = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((n & 63) == 63 && __hip_atomic_load(info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
        }
        if (v < target) {
            atomicCAS(info, 0, -1);
            v = FLAG_FAILED;
        }
        seen = v;
    }
    __syncthreads();
    const unsigned v = seen;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");    // every wavefront reads what was published
    __syncthreads();                                       // `seen` may be written again
    return v;
}

// A quarter of the tile at C -= Za^T Zb, Za and Zb 128 rows of 128 columns: all loads on the way at once, since the chain of a panel waits for
// it.  Ends with a barrier.
__device__ __forceinline__ void quarter_product(const double* Za, const double* Zb, long long ld, double* C, int quarter, TileShared& sm) {
    constexpr int Q = NB / 2, STAGES = NB / PKB;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i0 = Q * (quarter >> 1), j0 = Q * (quarter & 1), wi = (wave >> 1) * SB, wj = (wave & 1) * 2 * SB;
    const int lr = tid / 32, lc = (tid % 32) * 2;
    double2_t ra[STAGES], rb[STAGES];
#pragma unroll
    for (int k = 0; k < STAGES; ++k) {
        ra[k] = *reinterpret_cast<const double2_t*>(Za + (size_t)(PKB * k + lr) * ld + i0 + lc);
        rb[k] = *reinterpret_cast<const double2_t*>(Zb + (size_t)(PKB * k + lr) * ld + j0 + lc);
    }
    double4_t acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll
    for (int k = 0; k < STAGES; ++k) {
        *reinterpret_cast<double2_t*>(&sm.a[k & 1][lr][lc]) = ra[k];
        *reinterpret_cast<double2_t*>(&sm.b[k & 1][lr][lc]) = rb[k];
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < PKB; kk += 4) {
            const double fa = sm.a[k & 1][kk + lk][wi + l16];
#pragma unroll
            for (int q = 0; q < 2; ++q)
                acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa, sm.b[k & 1][kk + lk][wj + q * SB + l16], acc[q], 0, 0, 0);
        }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            unsafeAtomicAdd(C + (size_t)(i0 + wi + lk + 4 * r) * ld + j0 + wj + q * SB + l16, -acc[q][r]);
    __syncthreads();
}

struct FollowShared {
    double us[SB][SSTRIDE];       // block row K of U, right of the diagonal
    double ts[SB][SSTRIDE];       // block row K of the strip
    double v[SB][DSTRIDE];        // the inverse of the diagonal sub-block
};

// The strip T <- U11^-T T of the tile at (k0, j0) and the update of the diagonal tile at (j0, j0), D -= T^T T (on and above its
// diagonal), step by step beside the factorisation of the block at (k0, k0) on another CU: with block row K of U and the inverse V
// of its diagonal sub-block, T(K) <- V^T (T(K) - S(K)), S(I) += U(K,I)^T T(K) for I > K, D += T(K)^T T(K).  A wavefront has 16 columns of
// T and S in the accumulator layout, which is that of both operands, and every eighth sub-block of D.  (S by itself: subtracted from T as
// it comes, every product would round T; solutions of 256 to 2048 features were off by a tenth more.)
// Waiting for the whole block instead, then the strip, then the update, put two products of 8 us each and two trips through memory behind
// each factorisation of the chain.
// Ends with everything of this workgroup's in memory.  False: the factorisation failed, or the wait ran out (info is then -1).
__device__ __forceinline__ bool follow_block(double* A, long long ld, int k0, int j0, const double* invT, unsigned* steps,
                                             unsigned spin_limit, int* info, unsigned& seen, FollowShared& fs) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));      // (or the addresses of all steps are worked out ahead of the caller's loop, and spilled)
    const int lane = tid & 63, l16 = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int DSLOT = (NSUB + PT / 64 - 1) / (PT / 64);
    const double* U = A + (size_t)k0 * ld + k0;
    double* at = A + (size_t)(k0 + lk) * ld + j0 + SB * wave + l16;     // walks down the tile, four rows at a time (and is kept from being
    auto down = [&](double*& q) {                                       // worked out ahead of the loops, in registers that are not there)
        q += 4 * ld;
        asm volatile("" : "+v"(q));
    };
    double4_t S[NSB], D[DSLOT];
    int di[DSLOT], dj[DSLOT];
#pragma unroll
    for (int I = 0; I < NSB; ++I) S[I] = (double4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < DSLOT; ++s) {
        D[s] = (double4_t){0.0, 0.0, 0.0, 0.0};
        int t = 8 * s + wave, i = 0;
        while (i < NSB && t >= NSB - i) t -= NSB - i++;
        di[s] = i;                                                     // NSB: there is none
        dj[s] = i + t;
    }
    const int ur = tid / 32, uc = tid % 32;
    double nv = 0.0, nu[NB / 32] = {0.0, 0.0, 0.0, 0.0};               // this thread's part of a step on its way from memory
    auto fetch = [&](auto K_) {
        constexpr int K = decltype(K_)::value;
        if (tid < SB * SB) nv = load_past_caches(&invT[(K * SB + tid / SB) * NB + K * SB + tid % SB]);
#pragma unroll
        for (int q = (K + 1) * SB / 32; q < NB / 32; ++q)
            if (uc + 32 * q >= (K + 1) * SB) nu[q] = load_past_caches(&U[(size_t)(K * SB + ur) * ld + uc + 32 * q]);
    };
    unsigned there = 0u;                                               // block rows that were there when last looked
    return static_all<NSB>([&](auto K_) -> bool {
        constexpr int K = decltype(K_)::value;
        double4_t rest;                                                // T(K)
        {
            double* q = at;
#pragma unroll
            for (int r = 0; r < 4; ++r, down(q)) rest[r] = *q;
        }
        if (there < K + 1u) {
            if (tid == 0) {
                unsigned v = __hip_atomic_load(steps, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                for (unsigned n = 0; v < K + 1u && n < spin_limit; ++n) {
                    __builtin_amdgcn_s_sleep(4);
                    v = __hip_atomic_load(steps, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (__builtin_expect((n & 4095) == 4095, 0) && __hip_atomic_load(info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
                        n = spin_limit - 1;
                }
                if (__builtin_expect(v < K + 1u, 0)) {
                    atomicCAS(info, 0, -1);
                    v = FLAG_FAILED;
                }
                seen = v;
            }
            __syncthreads();
            there = __builtin_amdgcn_readfirstlane(seen);
            if (there & FLAG_FAILED) return false;
            fetch(K_);
        }
        if (tid < SB * SB) fs.v[tid % SB][tid / SB] = nv;
#pragma unroll
        for (int q = (K + 1) * SB / 32; q < NB / 32; ++q) fs.us[ur][uc + 32 * q] = nu[q];      // (columns left of the diagonal are not read)
        __syncthreads();
        if constexpr (K + 1 < NSB) {
            if (there > K + 1u) fetch(std::integral_constant<int, K + 1>{});       // beside this step's products
        }
        rest -= S[K];
        double4_t res = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) res = __builtin_amdgcn_mfma_f64_16x16x4f64(fs.v[4 * kk + lk][l16], rest[kk], res, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r, down(at)) {
            fs.ts[lk + 4 * r][SB * wave + l16] = res[r];
            *at = res[r];
        }
#pragma unroll
        for (int I = K + 1; I < NSB; ++I) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
                S[I] = __builtin_amdgcn_mfma_f64_16x16x4f64(fs.us[4 * kk + lk][SB * I + l16], res[kk], S[I], 0, 0, 0);
            if (I % 2 == 0) __builtin_amdgcn_sched_barrier(0);         // (or all operands are read first)
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < DSLOT; ++s)
            if (di[s] < NSB) {
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
                    D[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(fs.ts[4 * kk + lk][SB * di[s] + l16], fs.ts[4 * kk + lk][SB * dj[s] + l16],
                                                                D[s], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        if constexpr (K == NSB - 1) {
#pragma unroll
            for (int s = 0; s < DSLOT; ++s)
                if (di[s] < NSB) {
                    double* c = A + (size_t)(j0 + SB * di[s] + lk) * ld + j0 + SB * dj[s] + l16;
#pragma unroll
                    for (int r = 0; r < 4; ++r, down(c)) unsafeAtomicAdd(c, -D[s][r]);
                }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
        return true;
    });
}

// Panel rows [P0, P0 + 128 nblk); [R0, P0) are the rows of the panel before it, whose update the trailing
// matrix has not had yet (R0 = P0: nothing outstanding).  Workgroup ids: [0, nhead_pad) the tiles of this
// panel's rows that take that update ("head": column w has min(w, nblk - 1) + 1 of them, columns in order),
// then nown_pad ids for the column owners, then the tiles of the trailing matrix below this panel, nt per edge
// (0: none).  flags: FLAGS_PER_PANEL words, then one counter per column (head tiles done), all zero.
__global__ __launch_bounds__(PT, 2) void panel_kernel(double* A, long long ld, int F, int R0, int P0, int nblk,
                                                      int nhead_pad, int sharers, int nown_pad, int nt, TileMap tm,
                                                      double* invs, int* info, unsigned* flags, unsigned spin_limit) {
    // the tile product, the factorisation and the following of one never run at the same time: one piece of LDS for all (74 KB)
    __shared__ __attribute__((aligned(16))) union {
        TileShared tile;
        PotrfShared potrf;
        FollowShared follow;
    } lds;
    TileShared& sm = lds.tile;
    PotrfShared& ps = lds.potrf;
    __shared__ unsigned seen;
    if (*info != 0) return;
    unsigned* heads_done = flags + FLAGS_PER_PANEL;
    int bid = (int)blockIdx.x;
    if (bid < nhead_pad) {                                   // a head tile: waits for nobody
        int w, b;
        const int tri = nblk * (nblk + 1) / 2;               // the columns of the panel itself form a triangle
        if (bid < tri) {
            w = 0;
            while (bid >= (w + 1) * (w + 2) / 2) ++w;
            b = bid - w * (w + 1) / 2;
        } else {
            w = nblk + (bid - tri) / nblk;
            b = (bid - tri) % nblk;
        }
        const int k0 = P0 + b * NB, j0 = P0 + w * NB;
        if (j0 >= F) return;
        tile_product<NB>(A + (size_t)R0 * ld + k0, ld, A + (size_t)R0 * ld + j0, ld, P0 - R0, A + (size_t)k0 * ld + j0, ld,
                     -1.0, false, sm);
        publish_one_more(heads_done + w);
        return;
    }
    bid -= nhead_pad;
    if (bid >= nown_pad) {                                   // a tile of the trailing matrix
        int ti, tj;
        tile_of_block<true>((unsigned)(bid - nown_pad), nt, nt, tm, ti, tj);
        if (ti < 0 || ti > tj) return;
        const int Q = P0 + nblk * NB;
        const int i0 = Q + ti * NB, c0 = Q + tj * NB;
        tile_product<NB>(A + (size_t)R0 * ld + i0, ld, A + (size_t)R0 * ld + c0, ld, P0 - R0, A + (size_t)i0 * ld + c0, ld,
                     -1.0, false, sm);
        return;
    }
    // Quarters of the panel's tiles right of its diagonal ones, whose updates stand between a factorisation of the chain and the next but one:
    // four workgroups for tile (b, w), 1 <= b < w < nblk.  They come ahead of the other owners, so that they are running while owners wait for them.
    const int nquarter = 2 * (nblk - 1) * (nblk - 2);
    if (bid >= nblk && bid < nblk + nquarter) {
        __builtin_amdgcn_s_setprio(3);                       // (a CU may have other workgroups)
        int b = 1, w = 2, t = (bid - nblk) >> 2;
        while (t >= w - 1) t -= w++ - 1;
        b += t;
        double* into = A + (size_t)(P0 + b * NB) * ld + P0 + w * NB;
        for (int l = 0; l < b; ++l) {
            const double* strips = A + (size_t)(P0 + l * NB) * ld + P0;
            if (await(flags + PBLK + l * PBLK + b, FLAG_DONE, spin_limit, info, seen) != FLAG_DONE) return;
            if (await(flags + PBLK + l * PBLK + w, FLAG_DONE, spin_limit, info, seen) != FLAG_DONE) return;
            quarter_product(strips + b * NB, strips + w * NB, ld, into, (bid - nblk) & 3, sm);
            publish_one_more(flags + QUARTERS + b * PBLK + w);
        }
        return;
    }
    // a column owner: owner o < nblk has column o of the panel, the one with its diagonal tile in it; one or two each (`sharers`) have a
    // column of tiles right of the panel
    const int ncol = (F - P0) / NB;
    const int right = bid - nblk - nquarter;                 // of the panel
    const int w = bid < nblk ? bid : nblk + right / sharers;
    if (w >= ncol) return;
    const int j0 = P0 + w * NB + (bid < nblk ? 0 : right % sharers * (NB / 2));
    const int jend = P0 + w * NB + (bid < nblk || right % sharers == sharers - 1 ? NB : NB / 2);
    const int mine = bid < nblk ? bid : nblk - 1;            // last block row with a tile on or above the diagonal
    if (P0 > R0 && nhead_pad > 0) {
        if (await(heads_done + w, (unsigned)(mine + 1), spin_limit, info, seen) == FLAG_FAILED) return;
    } else if (P0 > R0) {                                    // no workgroups for the head tiles: the owner's own work
        for (int b = 0; b <= mine; ++b) {
            const double* above = A + (size_t)R0 * ld;
            double* into = A + (size_t)(P0 + b * NB) * ld + j0;
            if (jend - j0 == NB) tile_product<NB>(above + P0 + b * NB, ld, above + j0, ld, P0 - R0, into, ld, -1.0, false, sm);
            else tile_product<NB / 2>(above + P0 + b * NB, ld, above + j0, ld, P0 - R0, into, ld, -1.0, false, sm);
        }
    }
    if (bid < nblk) {                                        // the panel's own columns, which the chain is waiting for
        __builtin_amdgcn_s_setprio(3);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
#pragma unroll 1
        for (int l = 0; l < bid; ++l) {
            const int k0 = P0 + l * NB;
            if (l > 0) {                                      // the tile has had its updates by the strips above
                if (await(flags + QUARTERS + l * PBLK + bid, 4u * l, spin_limit, info, seen) == FLAG_FAILED) return;
            }
            unsigned* strip_done = flags + PBLK + l * PBLK + bid;
            if (!follow_block(A, ld, k0, j0, invs + ((size_t)(k0 / NB) * 2 + 1) * NB * NB, flags + STEPS + l, spin_limit, info, seen,
                              lds.follow)) {
                if (threadIdx.x == 0) store_past_caches(strip_done, FLAG_FAILED);
                return;
            }
            publish(strip_done, FLAG_DONE);
        }
        double* inv = invs + (size_t)(j0 / NB) * 2 * NB * NB;     // the own diagonal tile: every update is in
        const bool ok = potrf_block<true>(A, ld, j0, NB, inv, inv + NB * NB, info, flags + STEPS + bid, ps);
        // where a pivot is not positive every workgroup right of this column leaves at one of these flags; where a wait has run out, at info
        if (!ok && threadIdx.x == 0) store_past_caches(flags + STEPS + bid, FLAG_FAILED);
        publish(flags + bid, ok ? FLAG_DONE : FLAG_FAILED);
        return;
    }
    for (int l = 0; l < nblk; ++l) {
        const int k0 = P0 + l * NB;
        const double* inv = invs + (size_t)(k0 / NB) * 2 * NB * NB;
        if (await(flags + l, FLAG_DONE, spin_limit, info, seen) != FLAG_DONE) return;
        for (int j = j0; j < jend; j += NB / 2) {
            double* tile = A + (size_t)k0 * ld + j;
            tile_product<NB / 2, TRIANGULAR>(inv, NB, tile, ld, NB, tile, ld, 1.0, true, sm);
        }
        for (int b = l + 1; b < nblk; ++b) {
            if (await(flags + PBLK + l * PBLK + b, FLAG_DONE, spin_limit, info, seen) != FLAG_DONE) return;
            const double* strip = A + (size_t)k0 * ld + P0 + b * NB;
            if (jend - j0 == NB) tile_product<NB>(strip, ld, A + (size_t)k0 * ld + j0, ld, NB, A + (size_t)(P0 + b * NB) * ld + j0, ld, -1.0, false, sm);
            else tile_product<NB / 2>(strip, ld, A + (size_t)k0 * ld + j0, ld, NB, A + (size_t)(P0 + b * NB) * ld + j0, ld, -1.0, false, sm);
        }
    }
}

__global__ __launch_bounds__(256) void zero_words_kernel(unsigned* p, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// ---- triangular solves with one right-hand side -----------------------------------------
//
// One launch per direction, one workgroup per 128-row block.  Forward, U^T z = b: workgroup k keeps
// acc = b_k - sum_{i<k} U(i,k)^T z_i, taking the tiles U(i,k) in the order of i, then z_k = U11_k^-T acc through
// the stored inverse.  Backward, U x = z: the same from the last block to the first with the tiles U(k,j),
// j > k.  The values handed from workgroup to workgroup are their own flags: z (and the exchange copy of x)
// start out as a NaN with a payload no computation produces, a producer stores its 128 results with
// device-scope atomic stores, and a consumer polls the very values it needs with device-scope atomic loads
// (the tile they multiply is final and already on its way from memory): no fence, no separate flag, one trip
// through memory per step of the chain.  Every workgroup waits only for workgroups with lower ids (the backward
// launch numbers the blocks from the end), so whoever is waited for is running or done; the waits are bounded
// all the same, and one that runs out hands on a NaN, which ends up in the solution instead of a wrong number.
// Every sum is four, put together at its end: as fast (a step is its trip through memory), and its rounding errors add up over a quarter as many
// terms.
constexpr int ST = 512;            // threads of a solve workgroup
constexpr int SQ = ST / NB;        // row quarters: thread (c = tid % 128, q = tid / 128) has rows 32 q .. 32 q + 31
constexpr int SR = NB / SQ;
typedef double columns_t __attribute__((ext_vector_type(2), aligned(8)));     // of any row: the matrix may be a view
constexpr unsigned long long NOT_YET = 0x7FF8C0DEC0DE0001ULL;

__device__ __forceinline__ unsigned long long peek(const double* p) {
    return __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void hand_on(double* p, double v) {
    unsigned long long bits = (unsigned long long)__double_as_longlong(v);
    if (bits == NOT_YET) bits ^= 2ULL;                                // (never: keeps a consumer from waiting for ever)
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// out[c] = sum_m M[m,c] vec[m] with the thread's 32 rows of M in registers; the four partial sums through LDS
__device__ __forceinline__ double block_product(const double (&iv)[SR], const double* vec, double (*part)[NB], int c,
                                                int q) {
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < SR; ++m) s[m & 3] = fma(iv[m], vec[SR * q + m], s[m & 3]);
    part[q][c] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    return (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
}

__global__ __launch_bounds__(ST) void fwd_solve_kernel(const double* U, long long ld, int F, const double* invs,
                                                       const double* b, double* z, unsigned spin_limit) {
    __shared__ double part[SQ][NB], vec[NB];
    const int k = (int)blockIdx.x, k0 = k * NB;
    const int tid = threadIdx.x, lane = tid & 63, c = tid & (NB - 1), q = tid / NB;
    const double* inv = invs + (size_t)k * 2 * NB * NB;
    double iv[SR];
#pragma unroll
    for (int m = 0; m < SR; ++m) iv[m] = inv[(SR * q + m) * NB + c];
    const bool colok = k0 + c < F;
    double acc[4] = {(q == 0 && colok) ? b[k0 + c] : 0.0, 0.0, 0.0, 0.0};
    for (int i = 0; i < k; ++i) {
        const double* tile = U + (size_t)(i * NB + SR * q) * ld + k0 + c;
        double u[SR];
#pragma unroll
        for (int r = 0; r < SR; ++r) u[r] = colok ? tile[(size_t)r * ld] : 0.0;
        // lane r: row r of this wavefront's quarter of z_i
        const double* mine = z + i * NB + SR * q + (lane & (SR - 1));
        unsigned long long bits = peek(mine);
        for (unsigned n = 0; __builtin_amdgcn_ballot_w64(bits == NOT_YET) != 0ULL && n < spin_limit; ++n) {
            __builtin_amdgcn_s_sleep(4);
            bits = peek(mine);
        }
        const double zr = bits == NOT_YET ? __builtin_nan("") : __longlong_as_double((long long)bits);
#pragma unroll
        for (int r = 0; r < SR; ++r) acc[r & 3] = fma(-u[r], value_of_lane(zr, r), acc[r & 3]);
    }
    part[q][c] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    __syncthreads();
    if (tid < NB) vec[tid] = (part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]);
    __syncthreads();
    const double zk = block_product(iv, vec, part, c, q);
    if (tid < NB) hand_on(z + k0 + tid, zk);
}

__global__ __launch_bounds__(ST) void bwd_solve_kernel(const double* U, long long ld, int F, int nblk,
                                                       const double* invs, const double* z, double* xs, double* x,
                                                       unsigned spin_limit) {
    __shared__ double part[SQ][NB], vec[NB];
    const int k = nblk - 1 - (int)blockIdx.x, k0 = k * NB;
    const int tid = threadIdx.x, lane = tid & 63, c = tid & (NB - 1), q = tid / NB;
    const int csub = tid & 15, rowgrp = tid >> 4;          // sixteen lanes of four pairs of columns along a row; rows rowgrp + 32 a
    const double* invT = invs + (size_t)k * 2 * NB * NB + NB * NB;
    double iv[SR];
#pragma unroll
    for (int m = 0; m < SR; ++m) iv[m] = invT[(SR * q + m) * NB + c];
    double acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        acc[a][0] = csub == 0 ? z[k0 + rowgrp + 32 * a] : 0.0;
        acc[a][1] = acc[a][2] = acc[a][3] = 0.0;
    }
    for (int j = nblk - 1; j > k; --j) {
        // columns 32 e + 2 csub and the next: a load takes 256 bytes of a row, where eight neighbouring columns a lane took 32 loads of a
        // word in each of many lines: the launch 16.4 -> 10.5 us at 512 features, 63 -> 38 at 2048, 725 -> 419 at 16384.  One row a load, with
        // all its columns in a wavefront, needs sums over 64 lanes at the end: 26, 100 and 796 us
        const int col0 = j * NB + 2 * csub;
        columns_t u[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const double* row = U + (size_t)(k0 + rowgrp + 32 * a) * ld + col0;     // k < nblk - 1: a whole block of rows
            if (j * NB + NB <= F) {
#pragma unroll
                for (int e = 0; e < 4; ++e) u[a][e] = *reinterpret_cast<const columns_t*>(row + 32 * e);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    u[a][e][0] = col0 + 32 * e < F ? row[32 * e] : 0.0;
                    u[a][e][1] = col0 + 32 * e + 1 < F ? row[32 * e + 1] : 0.0;
                }
            }
        }
        // every wavefront polls the block's 128 values, two a lane, and hands each lane its eight (a lane that polled all it
        // needs itself took eight loads a poll, and the launch 1.18 ms at 16384 features where this took 0.72)
        const double* theirs = xs + j * NB + 2 * lane;
        unsigned long long b0 = peek(theirs), b1 = peek(theirs + 1);
        for (unsigned n = 0; __builtin_amdgcn_ballot_w64(b0 == NOT_YET || b1 == NOT_YET) != 0ULL && n < spin_limit; ++n) {
            __builtin_amdgcn_s_sleep(4);
            b0 = peek(theirs);
            b1 = peek(theirs + 1);
        }
        const double x0 = b0 == NOT_YET ? __builtin_nan("") : __longlong_as_double((long long)b0);
        const double x1 = b1 == NOT_YET ? __builtin_nan("") : __longlong_as_double((long long)b1);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const double xv = __shfl(e & 1 ? x1 : x0, csub + 16 * (e >> 1), 64);
#pragma unroll
            for (int a = 0; a < 4; ++a) acc[a][e & 3] = fma(-u[a][e >> 1][e & 1], xv, acc[a][e & 3]);
        }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        double sum = (acc[a][0] + acc[a][1]) + (acc[a][2] + acc[a][3]);
#pragma unroll
        for (int m = 8; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 16);
        if (csub == 0) vec[rowgrp + 32 * a] = sum;
    }
    __syncthreads();
    const double xk = block_product(iv, vec, part, c, q);
    if (tid < NB) {
        hand_on(xs + k0 + tid, xk);                         // whole blocks: the columns past F are zero
        if (k0 + tid < F) x[k0 + tid] = xk;
    }
}

__global__ __launch_bounds__(256) void fill_words64_kernel(unsigned long long* p, int n, unsigned long long v) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = v;
}

// the 128 x 128 tiles on or above the diagonal of A into U (the lower ones are never read); grid (column, row of tiles)
__global__ __launch_bounds__(256) void copy_upper_kernel(const double* __restrict__ A, long long lda, double* __restrict__ U,
                                                         long long ldu, int F, int Fp) {
    if (blockIdx.x < blockIdx.y) return;
    const int c = blockIdx.x * NB + (threadIdx.x & 63) * 2, r0 = blockIdx.y * NB + (threadIdx.x >> 6);
    const bool pairs = c + 1 < F && (lda | ldu) % 2 == 0 && ((uintptr_t)A | (uintptr_t)U) % 16 == 0;
#pragma unroll 8
    for (int r = r0; r < min(Fp, (int)(blockIdx.y + 1) * NB); r += 4) {
        const double* from = A + (size_t)r * lda + c;
        double* to = U + (size_t)r * ldu + c;
        if (pairs && r < F) *reinterpret_cast<double2_t*>(to) = *reinterpret_cast<const double2_t*>(from);
        else {
#pragma unroll
            for (int k = 0; k < 2; ++k)
                if (c + k < Fp) to[k] = r < F && c + k < F ? from[k] : r == c + k ? 1.0 : 0.0;
        }
    }
}

}  // namespace

// device workspace: the inverses of the diagonal blocks (both orientations), z of the forward solve and the
// exchange copy of x of the backward solve (whole blocks each), and the flags of the panel launches (per panel:
// FLAGS_PER_PANEL + one counter per block column)
namespace {
// Slabs: while more than 4096 rows are left, the rows of the factor above them act on the rest through exact int8 products
// (gram_modular.hip), before each panel of 512 rows on the panel's own rows only and at a slab's end on everything below it, so that
// the matrix is read and written once per slab and not once per panel.  In the last 4096 rows the panel launches of fp64 products
// are as fast, which are short there and wait for their chain of factorisations.  Up to 12288 rows a slab (15 bytes an entry
// for the residues, 3 GB at 16384 features); below 7168 features there is nothing to gain.  ms without slabs and with, taken when a
// block of the chain took 65 us (44 now, on both sides):
// 24576 features 90.3 / 54.4, 16384 31.6 / 23.0, 12288 16.2 / 13.8, 10240 11.3 / 10.3, 8192 7.6 / 7.3, 7168 6.1 / 6.0; a rest of 6144
// rows 23.4 at 16384 and 10.6 at 10240, of 3072 rows 23.1 and 10.3.
constexpr int SLAB = 12288, SLAB_REST = 4096, SLAB_LEAST = 3072;
// end of the slab of rows that starts at s0
int slab_end(int s0, int F) {
    const int below = (F - s0 - SLAB_REST) / OB * OB;          // rows that may go into slabs
    return below >= SLAB_LEAST ? s0 + std::min(SLAB, below) : F;
}

struct Workspace {
    double* invs;
    double* z;
    double* xs;
    unsigned* panel_flags;
    size_t nblk, npanel, bytes;
};
Workspace workspace_layout(void* base, int F) {
    Workspace w;
    w.nblk = ((size_t)F + NB - 1) / NB;
    w.npanel = ((size_t)F + OB - 1) / OB;
    w.invs = reinterpret_cast<double*>(base);
    w.z = w.invs + w.nblk * 2 * NB * NB;
    w.xs = w.z + w.nblk * NB;
    w.panel_flags = reinterpret_cast<unsigned*>(w.xs + w.nblk * NB);
    w.bytes = (w.nblk * 2 * NB * NB + 2 * w.nblk * NB) * sizeof(double) +
              w.npanel * (FLAGS_PER_PANEL + w.nblk) * sizeof(unsigned) + 256;
    return w;
}
}  // namespace

extern "C" size_t qmll_cholesky_workspace_bytes(int F) {
    if (F <= 0) return 0;
    return workspace_layout(nullptr, F).bytes;
}

extern "C" size_t qmll_cholesky_slabs_bytes(int F) {
    if (F <= 0 || F % NB != 0) return 0;
    size_t most = 0;
    for (int s0 = 0, s1 = slab_end(0, F); s1 < F; s0 = s1, s1 = slab_end(s0, F))
        most = std::max(most, qmll_internal_slab_bytes(s1 - s0, F - s0));
    return most;
}

namespace {

// rows [k0, k0+nb) of the panel that starts at P0: update from the panel's rows above, factor the
// diagonal block, solve the row strip to its right
int factor_block(double* A, int F, long long ld, int P0, int k0, double* invs, int* info, hipStream_t stream) {
    const int nb = F - k0 < NB ? F - k0 : NB;
    double* inv = invs + (size_t)(k0 / NB) * 2 * NB * NB;
    if (k0 > P0) {
        const double* above = A + (size_t)P0 * ld + k0;
        const int rc = qmll_internal_gemm_tn(above, ld, nb, above, ld, F - k0, k0 - P0, A + (size_t)k0 * ld + k0, ld,
                                             -1.0, 0, stream);
        if (rc != QMLL_OK) return rc;
    }
    hipLaunchKernelGGL(potrf_block_kernel, dim3(1), dim3(PT), 0, stream, A, ld, k0, nb, inv, inv + NB * NB, info);
    QMLL_CHECK_LAUNCH("qmll_cholesky_f64");
    const int n = F - k0 - nb;
    if (n > 0) {
        double* A12 = A + (size_t)k0 * ld + k0 + NB;
        return qmll_internal_gemm_tn(inv, NB, NB, A12, ld, n, NB, A12, ld, 1.0, 1, stream);
    }
    return QMLL_OK;
}

}  // namespace

extern "C" int qmll_copy_upper_f64(const double* A, long long lda, int F, double* U, long long ldu, qmll_stream_t stream) {
    return qmll_copy_upper_padded_f64(A, lda, F, U, ldu, F, stream);
}

extern "C" int qmll_copy_upper_padded_f64(const double* A, long long lda, int F, double* U, long long ldu, int Fp, qmll_stream_t stream) {
    QMLL_REQUIRE(F > 0 && Fp >= F && lda >= F && ldu >= Fp, QMLL_ERR_INVALID, "qmll_copy_upper_f64: bad size F=%d of %d lda=%lld ldu=%lld", F, Fp,
                 lda, ldu);
    QMLL_REQUIRE(A && U, QMLL_ERR_INVALID, "qmll_copy_upper_f64: null pointer");
    const unsigned n = ((unsigned)Fp + NB - 1) / NB;
    QMLL_REQUIRE(n <= 65535, QMLL_ERR_INVALID, "qmll_copy_upper_f64: F=%d too large", F);
    hipLaunchKernelGGL(copy_upper_kernel, dim3(n, n), dim3(256), 0, (hipStream_t)stream, A, lda, U, ldu, F, Fp);
    QMLL_CHECK_LAUNCH("qmll_copy_upper_f64");
    return QMLL_OK;
}

extern "C" int qmll_cholesky_f64(double* A, int F, long long ld, void* workspace, int* info, qmll_stream_t stream) {
    return qmll_cholesky_slabs_f64(A, F, ld, workspace, nullptr, info, stream);
}

extern "C" int qmll_cholesky_slabs_f64(double* A, int F, long long ld, void* workspace, void* slabs, int* info, qmll_stream_t stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    QMLL_REQUIRE(F > 0 && ld >= F, QMLL_ERR_INVALID, "qmll_cholesky_f64: bad size F=%d ld=%lld", F, ld);
    QMLL_REQUIRE(ld < (1LL << 23), QMLL_ERR_INVALID, "qmll_cholesky_f64: row stride %lld too large", ld);
    QMLL_REQUIRE(A && workspace && info, QMLL_ERR_INVALID, "qmll_cholesky_f64: null pointer");
    QMLL_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 16 == 0, QMLL_ERR_INVALID,
                 "qmll_cholesky_f64: the workspace must be 16-byte aligned");
    QMLL_REQUIRE(reinterpret_cast<uintptr_t>(slabs) % 16 == 0, QMLL_ERR_INVALID,
                 "qmll_cholesky_f64: the slabs' workspace must be 16-byte aligned");
    const Workspace ws = workspace_layout(workspace, F);
    double* invs = ws.invs;
    // whole tiles and 16-byte loads: one launch per panel, which also carries the trailing update of the panel
    // before it; otherwise a launch per step
    const bool whole_tiles = F % NB == 0 && ld % 2 == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0;
    if (whole_tiles) {
        unsigned* flags = ws.panel_flags;
        const int per_panel = FLAGS_PER_PANEL + (int)ws.nblk;
        const int nflags = (F + OB - 1) / OB * per_panel;
        hipLaunchKernelGGL(zero_words_kernel, dim3((nflags + 255) / 256), dim3(256), 0, stream, flags, nflags);
        QMLL_CHECK_LAUNCH("qmll_cholesky_f64");
        const char* who = "qmll_cholesky_f64";
        int S0 = 0, S1 = slabs ? slab_end(0, F) : F;          // rows of this slab; the last one has S1 = F
        for (int P0 = 0; P0 < F; P0 += OB) {
            const int pend = P0 + OB < F ? P0 + OB : F;       // this panel: rows [P0, pend)
            double* slab = A + (size_t)S0 * ld + S0;
            if (P0 > S0 && S1 < F) {                          // the panel before this one is final
                int rc = qmll_internal_slab_rows(slab, ld, S1 - S0, F - S0, P0 - OB - S0, OB, P0 - S0, slabs, who, stream);
                if (rc != QMLL_OK) return rc;
                // what this panel, or with a slab's last panel everything below, takes from the slab's rows
                rc = qmll_internal_slab_update(slab, ld, S1 - S0, F - S0, P0 - S0, P0 - S0, P0 < S1 ? OB / 256 : 0, slabs, who, stream);
                if (rc != QMLL_OK) return rc;
            }
            if (P0 == S1) {
                S0 = S1;
                S1 = slab_end(S0, F);
                slab = A + (size_t)S0 * ld + S0;
            }
            if (P0 == S0 && S1 < F) {
                const int rc = qmll_internal_slab_begin(slab, ld, S1 - S0, F - S0, slabs, who, stream);
                if (rc != QMLL_OK) return rc;
            }
            // the panel before it, whose update this launch carries: in the last slab only
            const int R0 = S1 == F && P0 > S0 ? P0 - OB : P0;
            const int nblk = (pend - P0) / NB;
            const int ncol = (F - P0) / NB;                   // columns of tiles from the panel's first to the last
            const int nt = P0 > R0 ? (F - pend) / NB : 0;
            // The head tiles (this panel's rows of the update of the panel before) go to workgroups of their own
            // once the trailing matrix is small, where a launch lasts as long as its slowest owner, which has four head
            // tiles and ten strip / update products in a row (16384 features 22.9 ms without, 21.8 so; 8192 8.15 and 7.09;
            // 4096 3.89 and 2.88; a line at 24 tiles an edge instead of 48 5.30 against 4.86 at 6144).
            // While the trailing tiles keep the chip busy for longer than that, the owners take their head tiles
            // themselves and no slot waits for another.
            const bool split_heads = P0 > R0 && nt <= SPLIT_HEADS_BELOW;
            // Two workgroups to a column of tiles right of the panel while all of them have a CU, since the launch lasts as long as a column's
            // four strips and six updates (640 features 372 -> 315 us, 4096 2.54 -> 2.19 ms); with more they would come one after the other.
            const int nchain = nblk + 2 * (nblk - 1) * (nblk - 2);            // the panel's own columns and their quarter tiles
            const int sharers = nchain + 2 * (ncol - nblk) <= CUS ? 2 : 1;
            const int nown_pad = (nchain + sharers * (ncol - nblk) + NXCD - 1) / NXCD * NXCD;
            const int nhead = split_heads ? nblk * (nblk + 1) / 2 + (ncol - nblk) * nblk : 0;
            const int nhead_pad = (nhead + NXCD - 1) / NXCD * NXCD;
            long long per_xcd = 0;
            TileMap tm = gram_tile_map(nt > 0 ? nt : 1, nt > 0 ? nt : 1, true, per_xcd);
            const long long grid = (long long)nhead_pad + nown_pad + (nt > 0 ? per_xcd * NXCD : 0);
            QMLL_REQUIRE(grid < 2147483647LL, QMLL_ERR_INVALID, "qmll_cholesky_f64: too many tiles");
            hipLaunchKernelGGL(panel_kernel, dim3((unsigned)grid), dim3(PT), 0, stream, A, ld, F, R0, P0, nblk, nhead_pad,
                               sharers, nown_pad, nt, tm, invs, info, flags + (size_t)(P0 / OB) * per_panel, SPIN_LIMIT);
            QMLL_CHECK_LAUNCH("qmll_cholesky_f64");
        }
        return QMLL_OK;
    }
    for (int P0 = 0; P0 < F; P0 += OB) {
        const int pend = P0 + OB < F ? P0 + OB : F;           // this panel: rows [P0, pend)
        for (int k0 = P0; k0 < pend; k0 += NB) {
            const int rc = factor_block(A, F, ld, P0, k0, invs, info, stream);
            if (rc != QMLL_OK) return rc;
        }
        if (pend >= F) break;
        const int rc = qmll_internal_syrk_upper(A + (size_t)P0 * ld + pend, pend - P0, F - pend, ld,
                                                A + (size_t)pend * ld + pend, ld, -1.0, stream);
        if (rc != QMLL_OK) return rc;
    }
    return QMLL_OK;
}

extern "C" int qmll_cholesky_solve_f64(const double* U, int F, long long ld, void* workspace, double* b,
                                       qmll_stream_t stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    QMLL_REQUIRE(F > 0 && ld >= F, QMLL_ERR_INVALID, "qmll_cholesky_solve_f64: bad size F=%d ld=%lld", F, ld);
    QMLL_REQUIRE(U && workspace && b, QMLL_ERR_INVALID, "qmll_cholesky_solve_f64: null pointer");
    const Workspace ws = workspace_layout(workspace, F);
    const int nblk = (int)ws.nblk;
    // z and the exchange copy of x are contiguous: "not yet" everywhere
    hipLaunchKernelGGL(fill_words64_kernel, dim3((2 * nblk * NB + 255) / 256), dim3(256), 0, stream,
                       reinterpret_cast<unsigned long long*>(ws.z), 2 * nblk * NB, NOT_YET);
    QMLL_CHECK_LAUNCH("qmll_cholesky_solve_f64");
    // U^T z = b, then U x = z with x into b
    hipLaunchKernelGGL(fwd_solve_kernel, dim3(nblk), dim3(ST), 0, stream, U, ld, F, ws.invs, b, ws.z, SPIN_LIMIT);
    QMLL_CHECK_LAUNCH("qmll_cholesky_solve_f64");
    hipLaunchKernelGGL(bwd_solve_kernel, dim3(nblk), dim3(ST), 0, stream, U, ld, F, nblk, ws.invs, ws.z, ws.xs, b,
                       SPIN_LIMIT);
    QMLL_CHECK_LAUNCH("qmll_cholesky_solve_f64");
    return QMLL_OK;
}
