// Z^T Z of fp64 rows on the int8 matrix cores: the same sums as gram.hip, from exact integer products.
//
// The fp64 matrix instruction does 32 flops per clock and SIMD, the int8 one 2048.  A column a of Z is scaled
// by a power of two so that its 2-norm lies in (2^(gamma-1), 2^gamma] and rounded to integers a'.  By
// Cauchy-Schwarz no entry of A'^T A' exceeds 2^(2 gamma) in magnitude, so it is known exactly from its residues
// for N pairwise coprime moduli p <= 256 whose product is above twice that bound (gamma = 54, N = 14:
// 2^108 against 2^110.2).  A residue of A'^T A' is an ordinary int8 product of the residues of A' with int32 sums.
// This is the modular form of a split product of Ozaki, Uchino and Imamura ("Ozaki Scheme II", 2025), derived
// here for the symmetric case; against slices of 7 or 8 bits (28 products for the same accuracy) it
// needs half the matrix work.
//
// The only roundings are a -> a' (at most 2^-54 of the column's norm per entry) and the result's to fp64.  The
// error of C_ij is therefore of the order 2^-54 |a_i| |a_j| whatever the number of rows, where a sum of M fp64
// products has errors growing with sqrt(M) of the largest partial sum.  Measured against extended precision on training rows of
// both models (1300 to 9600 rows of 768 to 4096 features): 4.9e-17 to 6.3e-17 of the 2-norm and at most 2.3e-16 of
// |a_i| |a_j|, the fp64 kernel 1.7e-15 to 4.6e-15 and 2.3e-14; on normal random rows 5.7e-16 against 9.4e-16 for 1000 rows and
// 9.2e-16 against 3.9e-15 for 20000.  Entry by entry, relative to s = sum_k |a_ki a_kj|, it depends on how far s is below
// |a_i| |a_j|.  In training rows it is not far (at least 0.03 of it, 0.7 to 0.99 for most entries: every feature sums over all
// atoms, so a row is large or small in all columns alike): rms 4.6e-17 to 8.7e-17 of s, fp64 1.4e-15 to 3.7e-15.  It is far where
// columns have their large entries in different rows: 800 rows of 256 columns with independent log-normal magnitudes (sigma 1, 2, 3, 5)
// 1.6e-16, 2.7e-15, 1.8e-13 and 1.3e-10 of s against 1.3e-16 to 7.2e-16.  So the caller chooses; training does, because its
// rows are of the first kind and because the factorisation that takes the matrix errs by F 2^-53 |a_i| |a_j| itself.
// Columns whose norm is no ordinary number
// (NaN, infinity, squares that over- or underflow) switch the whole call to the fp64 kernel, on the device.
//
// 32000 rows of 16384 features: 47 ms, 183 TFLOP/s of the fp64 sums it stands for, against 130 ms and 66 TFLOP/s of the fp64 kernel
// (which is 0.84 of what that unit does).  43 ms are modular_gemm, bound by the card's power: the int8 unit runs at
// 1.4 to 1.5 GHz under it; residues 2.2 ms and norms 0.7 ms are memory traffic (4.2 GB read twice, 7.3 GB written),
// reconstruction 1 ms.
//
//   column_norms      2-norms of the columns (and Z^T y from the same read), parts per 512 rows
//   column_scales     parts added in order, exponents, Z^T y, the switch
//   residues          one byte per entry and modulus, in the order in which the matrix instruction reads them
//   modular_gemm      per modulus and 256 x 256 tile on or above the diagonal: int8 product, residue, one byte out
//   reconstruct       Chinese remainder theorem in exact fp64 limbs, C += result
#include <algorithm>

#include "qmll_common.h"
#include "gram_modular.h"

namespace {

typedef int int4_t __attribute__((ext_vector_type(4)));
typedef int int2_t __attribute__((ext_vector_type(2)));

template <int N>
struct ModTable {
    int p[N];
    float inv[N];        // 1/p
    double dp[N], dinv[N];
    int y[N];            // (P/p)^-1 mod p, symmetric residue
    double m0[N], m1[N], m2[N];     // P/p in limbs of LIMB bits, the lowest first
    double P0, P1, P2;
};

// exact sums: a limb, a residue of 7 bits and up to 8 N terms stay below 2^53 (N = 14: 36 + 7 + 7, the top limb 31 + 14; 15: 38 + 7 + 7, 35 + 14)
template <int N>
constexpr int LIMB = N == 14 ? 36 : 38;
template <int N>
constexpr int GAMMA = modular_gamma(N);

template <int N>
constexpr ModTable<N> make_table() {
    ModTable<N> t{};
    const int p[15] = {256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197};
    unsigned __int128 P = 1;
    for (int i = 0; i < N; ++i) P *= (unsigned)p[i];
    const unsigned __int128 mask = (((unsigned __int128)1) << LIMB<N>) - 1;
    for (int i = 0; i < N; ++i) {
        const unsigned __int128 m = P / (unsigned)p[i];
        const int r = (int)(m % (unsigned)p[i]);
        int y = 1;
        while ((r * y) % p[i] != 1) ++y;
        t.p[i] = p[i];
        t.inv[i] = 1.0f / (float)p[i];
        t.dp[i] = (double)p[i];
        t.dinv[i] = 1.0 / (double)p[i];
        t.y[i] = y > p[i] / 2 ? y - p[i] : y;
        t.m0[i] = (double)(unsigned long long)(m & mask);
        t.m1[i] = (double)(unsigned long long)((m >> LIMB<N>) & mask);
        t.m2[i] = (double)(unsigned long long)(m >> (2 * LIMB<N>));
    }
    t.P0 = (double)(unsigned long long)(P & mask);
    t.P1 = (double)(unsigned long long)((P >> LIMB<N>) & mask);
    t.P2 = (double)(unsigned long long)(P >> (2 * LIMB<N>));
    return t;
}
template <int N>
constexpr ModTable<N> TAB = make_table<N>();
__constant__ const ModTable<14> DTAB14 = make_table<14>();
__constant__ const ModTable<15> DTAB15 = make_table<15>();
template <int N>
__device__ __forceinline__ const ModTable<N>& device_table() {
    if constexpr (N == 14) return DTAB14;
    else return DTAB15;
}

constexpr double SHIFTER = 6755399441055744.0;     // 1.5 * 2^52: adding it rounds to an integer in the low mantissa bits

// ---- norms -----------------------------------------------------------------------------------------
// sums of squares (and of products with y) over NORM_ROWS rows per column; thread = column, eight rows in flight
__global__ __launch_bounds__(256) void column_norms_kernel(const double* __restrict__ Z, long long ldz,
                                                           const double* __restrict__ y, int M, int F, double* __restrict__ parts,
                                                           double* __restrict__ yparts, int* __restrict__ flag) {
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *flag = 0;
    const int f = blockIdx.x * 256 + threadIdx.x;
    if (f >= F) return;
    const int m0 = blockIdx.y * NORM_ROWS, m1 = min(M, m0 + NORM_ROWS);
    double s = 0.0, t = 0.0;
    bool any = false;              // an entry that is not 0, whether or not its square is
    int m = m0;
    for (; m + 8 <= m1; m += 8) {
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = Z[(size_t)(m + q) * ldz + f];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            s = fma(v[q], v[q], s);
            any |= v[q] != 0.0;
            if (y) t = fma(v[q], y[m + q], t);
        }
    }
    for (; m < m1; ++m) {
        const double v = Z[(size_t)m * ldz + f];
        s = fma(v, v, s);
        any |= v != 0.0;
        if (y) t = fma(v, y[m], t);
    }
    parts[(size_t)blockIdx.y * F + f] = any && s == 0.0 ? 1e-300 : s;
    if (y) yparts[(size_t)blockIdx.y * F + f] = t;
}

__global__ __launch_bounds__(256) void column_scales_kernel(const double* __restrict__ parts, const double* __restrict__ yparts,
                                                            int nparts, int F, int Fp, double* __restrict__ scale,
                                                            int* __restrict__ expo, double* __restrict__ ZTy,
                                                            int* __restrict__ flag) {
    const int f = blockIdx.x * 256 + threadIdx.x;
    if (f >= Fp) return;
    double s = 0.0, t = 0.0;
    if (f < F) {
        for (int c = 0; c < nparts; ++c) s += parts[(size_t)c * F + f];
        if (yparts) {
            for (int c = 0; c < nparts; ++c) t += yparts[(size_t)c * F + f];
            ZTy[f] += t;
        }
    }
    int e = 0;
    if (s != 0.0) {
        // NaN, close to overflow, or so small that squares may have vanished from the sum
        if (!(s > 1e-200 && s < 1e280)) atomicOr(flag, 1);
        else {
            int x;
            (void)frexp(s * 1.0000001, &x);        // the factor is far above the sum's own rounding
            e = (x + 1) >> 1;                      // |a| < 2^e
        }
    }
    expo[f] = e;
    scale[f] = ldexp(1.0, GAMMA<GRAM_MODULI> - e);
}

// ---- residues --------------------------------------------------------------------------------------
// One wavefront takes 16 features x 64 rows: lane = (16 rows, feature), 16 loads of 128-byte row pieces, and
// writes one 1 KB operand per modulus.  Plane layout: [modulus][k / 64][feature / 16][lane][16 rows].
template <int N, bool FIX>
__device__ __forceinline__ void residue_bytes(const double (&v)[16], signed char* __restrict__ dst, size_t plane) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        int4_t out;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            unsigned b[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const double a = v[4 * g + q];
                if (i == 0) {                              // modulus 256: the low byte itself
                    b[q] = (unsigned)__double2loint(a + SHIFTER);
                    if (FIX) b[q] = (unsigned)(int)(long long)a;
                } else {
                    const double k = fma(a, TAB<N>.dinv[i], SHIFTER) - SHIFTER;
                    const double r = fma(-TAB<N>.dp[i], k, a);
                    int ri = __double2loint(r + SHIFTER);
                    if (FIX) {                             // the quotient of a large entry may be off by one
                        if (ri > 127) ri -= TAB<N>.p[i];
                        if (ri < -127) ri += TAB<N>.p[i];
                    }
                    b[q] = (unsigned)ri;
                }
            }
            const unsigned lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400);
            const unsigned hi = __builtin_amdgcn_perm(b[3], b[2], 0x04000c0c);
            out[g] = (int)(lo | hi);
        }
        *reinterpret_cast<int4_t*>(dst + (size_t)i * plane) = out;
    }
}

// Features f0 .. F of M rows, which are rows 64 kb0 .. of the planes.  sums (or null): the columns' squares, in units of 4^gamma.
template <int N>
__global__ __launch_bounds__(256) void residues_kernel(const double* __restrict__ Z, long long ldz, int M, int F, int Fp, int f0,
                                                       int kb0, const double* __restrict__ scale, const int* __restrict__ flag,
                                                       signed char* __restrict__ planes, size_t plane, double* __restrict__ sums) {
    if (*flag) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // workgroup: 64 rows x 64 features
    const int kb = blockIdx.y, fb = f0 / 16 + blockIdx.x * 4 + wave;
    const int f = fb * 16 + (lane & 15);
    const int k0 = kb * 64 + (lane >> 4) * 16;
    double v[16];
    const bool fin = f < F;
    if (fin && k0 + 16 <= M) {
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = Z[(size_t)(k0 + q) * ldz + f];
    } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = (fin && k0 + q < M) ? Z[(size_t)(k0 + q) * ldz + f] : 0.0;
    }
    const double s = scale[f];
    double big = 0.0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        v[q] = rint(v[q] * s);
        big = fmax(big, fabs(v[q]));
    }
    if (sums) {
        double q = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const double u = v[k] * (1.0 / (double)(1ll << GAMMA<N>));
            q = fma(u, u, q);
        }
        q += __shfl_xor(q, 16, 64);
        q += __shfl_xor(q, 32, 64);
        if (lane < 16 && fin) unsafeAtomicAdd(&sums[f], q);
    }
    signed char* dst = planes + ((size_t)(kb0 + kb) * (Fp / 16) + fb) * 1024 + lane * 16;
    // below 2^50 a / p is known to better than 1e-3 and its rounding leaves |residue| <= 127 (p = 255 is the tightest)
    if (__any(big > 1125899906842624.0))
        residue_bytes<N, true>(v, dst, plane);
    else
        residue_bytes<N, false>(v, dst, plane);
}

// tile number t of a launch: of the upper triangle behind the first `off` tile rows and columns of nt x nt, or of its first
// `band` tile rows
__device__ __forceinline__ void find_tile(int t, int off, int band, int nt, int& ti, int& tj) {
    if (band > 0) modular_band_tile(t, band, ti, tj);
    else modular_tile(t, nt - off, ti, tj);
    ti += off;
    tj += off;
}
constexpr double SUM_LIMIT = 1.1;     // of a column's squares in units of 4^gamma: half the product of the moduli is 1.72 4^gamma

// ---- products --------------------------------------------------------------------------------------
// One 16-byte piece per lane from global memory to LDS, 1 KB per wavefront, PIECE KB behind both addresses.  Written as
// assembly because the compiler, which cannot tell the stages of the LDS buffer apart, would otherwise wait for every load
// in flight before each LDS read; the waits are written out.
template <int PIECE>
__device__ __forceinline__ void stage_1k(const signed char* base, unsigned voff, unsigned lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3"
                 :
                 : "s"(lds), "v"(voff), "s"(base), "n"(PIECE * 1024)
                 : "memory");
}

// c += a.b of 16 x 64 by 64 x 16.  Assembly, because with 256 accumulator registers in use the compiler's allocator gives
// the result other registers than the addend and copies the sums about in the loop
__device__ __forceinline__ void multiply_add(int4_t& c, const int4_t& a, const int4_t& b) {
    asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

constexpr int STAGE = 32768;          // 64 rows of two 256-feature panels
constexpr int NSTAGE = 5;             // 160 KB, all of a CU's LDS

// Four wavefronts of 128 x 128 each (256 accumulator registers, one wavefront per SIMD), 64 rows per stage.  Per stage a
// wavefront reads 16 KB of operands for 64 matrix instructions of 16 clocks: the LDS is busy for half of the time and a
// quarter more with the stages written.  The next stage's operands are read between the first 32 instructions, and the eight
// loads of the stage five ahead go out one by one between the same: all at once they cost 4 ms of 47.  A loop of nothing but
// the instruction does 4.2 POP/s on random bytes (16 x 16 x 64; the 32 x 32 x 32 form 3.5: larger sums toggle per operation),
// this kernel 2.8; without its global loads it would take 35 ms of 43, on constant operands.
template <int N>
__global__ __launch_bounds__(256, 1) void modular_gemm_kernel(const signed char* __restrict__ planes, size_t plane, int Fp, int nk,
                                                              int pieces, int off, int band, int nt, int t0, int ntile,
                                                              const int* __restrict__ flag, signed char* __restrict__ out) {
    if (*flag) return;
    const unsigned b = blockIdx.x;
    // 32 consecutive items (one panel set of 4 x 8 tiles) per XCD: workgroup ids go round the XCDs
    const unsigned k = b / 8;
    const unsigned item = ((k / 32) * 8 + b % 8) * 32 + k % 32;
    const unsigned total = (unsigned)ntile * N * pieces;
    if (item >= total) return;
    const int tile = item % ntile, rest = item / ntile;
    const int mod = rest % N, piece = rest / N;
    int ti, tj;
    find_tile(t0 + tile, off, band, nt, ti, tj);
    // nk is even, and so is every row range; one past the end is empty
    const int per = (nk / 2 + pieces - 1) / pieces * 2;
    const int kb0 = min(piece * per, nk), n = min(nk - kb0, per);
    const int last = max(n - 1, 0), kbs = n > 0 ? kb0 : 0;

    extern __shared__ __attribute__((aligned(1024))) signed char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wi = wave >> 1, wj = wave & 1;
    const unsigned lbase = (unsigned)(uintptr_t)(__attribute__((address_space(3))) signed char*)lds;

    const size_t kstep = (size_t)Fp * 64;
    const signed char* pa = planes + (size_t)mod * plane + (size_t)kbs * kstep + (size_t)ti * 16384 + wave * 4096;
    const signed char* pb = planes + (size_t)mod * plane + (size_t)kbs * kstep + (size_t)tj * 16384 + wave * 4096;
    const unsigned voff = lane * 16;

    int4_t acc[8][8];
#pragma unroll
    for (int p = 0; p < 8; ++p)
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[p][q] = (int4_t)(0);

    int into = 0, from = 0;                              // places in LDS: of the next stage to load, of the next to read
    // piece j of stage s: 0..3 of the left panel, 4..7 of the right one
    auto issue = [&](int s, int j) {
        const int c = min(s, last);                      // past the end: the last stage once more, never multiplied
        const unsigned l = __builtin_amdgcn_readfirstlane(lbase + into + wave * 4096);
        const signed char* ga = pa + (size_t)c * kstep;
        const signed char* gb = pb + (size_t)c * kstep;
        switch (j) {
            case 0: stage_1k<0>(ga, voff, l); break;
            case 1: stage_1k<1>(ga, voff, l); break;
            case 2: stage_1k<2>(ga, voff, l); break;
            case 3: stage_1k<3>(ga, voff, l); break;
            case 4: stage_1k<0>(gb, voff, l + 16384); break;
            case 5: stage_1k<1>(gb, voff, l + 16384); break;
            case 6: stage_1k<2>(gb, voff, l + 16384); break;
            default: stage_1k<3>(gb, voff, l + 16384); into = into == (NSTAGE - 1) * STAGE ? 0 : into + STAGE;
        }
    };
    int4_t fa[2][8], fb[2][8];
    auto fetch = [&](int u, int4_t (&a)[8], int4_t (&bb)[8]) {
        const signed char* st = lds + from + lane * 16;
        if (u < 8) bb[u] = *reinterpret_cast<const int4_t*>(st + 16384 + (wj * 8 + u) * 1024);
        else a[u - 8] = *reinterpret_cast<const int4_t*>(st + (wi * 8 + u - 8) * 1024);
        if (u == 15) from = from == (NSTAGE - 1) * STAGE ? 0 : from + STAGE;
    };
    // stage i from registers, the operands of stage i + 1 read from LDS and stage i + 5 on its way behind the
    // first matrix instructions
    auto step = [&](int i, int h) {
        // stage i + 1 is here once only the loads of the three stages behind it are outstanding; behind the barrier it
        // is here for every wavefront, and every wavefront has its operands of stage i, whose place i + 5 takes
        asm volatile("s_waitcnt vmcnt(24) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 64; ++t) {
            multiply_add(acc[t >> 3][t & 7], fa[h][t >> 3], fb[h][t & 7]);
            if (t % 2 == 0 && t < 32) fetch(t / 2, fa[h ^ 1], fb[h ^ 1]);
            if (t % 4 == 1 && t < 32) issue(i + NSTAGE, t / 4);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int s = 0; s < NSTAGE; ++s) {
#pragma unroll
        for (int j = 0; j < 8; ++j) issue(s, j);
    }
    asm volatile("s_waitcnt vmcnt(32)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int u = 0; u < 16; ++u) fetch(u, fa[0], fb[0]);
    for (int i = 0; i < n; i += 2) {
        step(i, 0);
        step(i + 1, 1);
    }
    // no load may still write LDS when the workgroup ends; and the last products are on their way to the accumulators,
    // which nothing may read before: the compiler, which does not know what multiply_add is, keeps to the order of these
    asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int t = 0; t < 64; ++t) asm volatile("" : "+a"(acc[t >> 3][t & 7]));

    // residue of the sum times (P/p)^-1, one byte per entry in the order of the accumulator registers
    const int p = device_table<N>().p[mod], y = device_table<N>().y[mod];
    const float inv = device_table<N>().inv[mod];
    signed char* o = out + (((size_t)piece * N + mod) * ntile + tile) * 65536 + (size_t)wave * 16384 + lane * 16;
#pragma unroll
    for (int pp = 0; pp < 8; ++pp)
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
            int4_t w;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                unsigned bb[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = acc[pp][qq * 4 + g][e];
                    // |c| <= 2^30: the quotient is below 2^23 and off by less than two
                    const int r = c - __mul24((int)rintf((float)c * inv), p);
                    const int u = __mul24(r, y);
                    bb[e] = (unsigned)(u - __mul24((int)rintf((float)u * inv), p));
                }
                const unsigned lo = __builtin_amdgcn_perm(bb[1], bb[0], 0x0c0c0400);
                const unsigned hi = __builtin_amdgcn_perm(bb[3], bb[2], 0x04000c0c);
                w[g] = (int)(lo | hi);
            }
            *reinterpret_cast<int4_t*>(o + (pp * 2 + qq) * 1024) = w;
        }
}

// More than 64 KB of dynamic LDS have to be allowed, and what is allowed belongs to the device that is current: asked for before the
// launches of each call, which costs the host less than a launch, instead of remembered for the process
template <int N>
hipError_t allow_stages() {
    return hipFuncSetAttribute((const void*)modular_gemm_kernel<N>, hipFuncAttributeMaxDynamicSharedMemorySize, NSTAGE * STAGE);
}

// ---- reconstruction --------------------------------------------------------------------------------
// thread = half the entries of one lane's accumulator: V = sum_i t_i (P / p_i) - P rint(sum_i t_i / p_i), every limb sum an
// integer below 2^53 and so exact in fp64; C += (overwrite: =) V 2^-(2 gamma - e_i - e_j)
// Eight entries, so that the residues of all moduli and what is added to are on their way together; with
// sixteen the registers held one modulus at a time and every one was waited for.  All of a factorisation of 16384 columns 1657 -> 1209 us,
// two products of as many 1926 -> 1818 (4.4 TB/s)
constexpr int REC_PER_TILE = 32;       // workgroups of a 256 x 256 tile: four wavefronts with 32 lanes' entries each
template <int N>
__global__ __launch_bounds__(256) void reconstruct_kernel(const signed char* __restrict__ res, int pieces, int off, int band, int nt,
                                                          int t0, int ntile,
                                                          int F, const int* __restrict__ expo, const double* __restrict__ sums,
                                                          const int* __restrict__ flag,
                                                          double sign, int overwrite, double* __restrict__ C, long long ldc) {
    if (*flag) return;
    const int tile = blockIdx.x / REC_PER_TILE, sub = blockIdx.x % REC_PER_TILE;
    int ti, tj;
    find_tile(t0 + tile, off, band, nt, ti, tj);
    const int part = sub * 4 + (threadIdx.x >> 6), unit = part >> 1;        // a 16 x 64 block of the tile, half of its lanes
    const int lane = (part & 1) * 32 + ((threadIdx.x & 63) >> 1), first = (threadIdx.x & 1) * 8;       // the accumulator's lane, its entries
    const int wave = unit >> 4, pp = (unit >> 1) & 7, qq = unit & 1;
    const int i0 = ti * 256 + (wave >> 1) * 128 + pp * 16 + (lane >> 4) * 4;
    const int j0 = tj * 256 + (wave & 1) * 128 + qq * 64 + (lane & 15) + first * 4;
    if (i0 >= F || j0 >= F) return;
    if ((ti * 2 + (wave >> 1)) > (tj * 2 + (wave & 1))) return;     // a 128 x 128 tile below the diagonal
    const signed char* src = res + (size_t)tile * 65536 + (size_t)unit * 1024 + lane * 16 + first;
    constexpr int E = 8;
    double s0[E], s1[E], s2[E], old[E];
    float z[E];
    int2_t w[N];
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = *reinterpret_cast<const int2_t*>(src + (size_t)i * ntile * 65536);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = i0 + (e & 3), j = j0 + (e >> 2) * 16;
        old[e] = !overwrite && i < F && j < F ? C[(size_t)i * ldc + j] : 0.0;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        s0[e] = s1[e] = s2[e] = 0.0;
        z[e] = 0.0f;
    }
    for (int c = 0;;) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int t = (int)(signed char)(w[i][e >> 2] >> (8 * (e & 3)));
                const double d = (double)t;
                s0[e] = fma(d, TAB<N>.m0[i], s0[e]);
                s1[e] = fma(d, TAB<N>.m1[i], s1[e]);
                s2[e] = fma(d, TAB<N>.m2[i], s2[e]);
                z[e] = fmaf((float)t, TAB<N>.inv[i], z[e]);
            }
        }
        if (++c == pieces) break;
#pragma unroll
        for (int i = 0; i < N; ++i) w[i] = *reinterpret_cast<const int2_t*>(src + ((size_t)c * N + i) * ntile * 65536);
    }
    constexpr double B = (double)(1ll << LIMB<N>), IB = 1.0 / B;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = i0 + (e & 3), j = j0 + (e >> 2) * 16;
        if (i >= F || j >= F) continue;
        const double k = (double)rintf(z[e]);
        double a0 = fma(-k, TAB<N>.P0, s0[e]), a1 = fma(-k, TAB<N>.P1, s1[e]), a2 = fma(-k, TAB<N>.P2, s2[e]);
        const double c0 = floor(a0 * IB);
        a0 = fma(-c0, B, a0);
        a1 += c0;
        const double c1 = floor(a1 * IB);
        a1 = fma(-c1, B, a1);
        a2 += c1;
        const double v = fma(fma(a2, B, a1), B, a0);
        double* c = C + (size_t)i * ldc + j;
        if (sums && !(sums[i] <= SUM_LIMIT && sums[j] <= SUM_LIMIT)) *c = __builtin_nan("");
        else *c = old[e] + ldexp(sign * v, expo[i] + expo[j] - 2 * GAMMA<N>);
    }
}

}  // namespace

// gram.hip: the fp64 kernel over tiles on or above the diagonal, on the device only if *only_if is not 0
int qmll_internal_gram_if(const double* Z, long long ldz, int M, int F, double* C, long long ldc, double sign, int overwrite,
                          const int* only_if, const char* who, hipStream_t stream);

// C[F,F] (row stride ldc, tiles on or above the diagonal) += (overwrite: =) sign Z^T Z, Z = M rows of F columns with row stride ldz;
// ZTy += Z^T y
static int modular_syrk(const double* Z, long long ldz, const double* y, int M, int F, double* C, long long ldc, double sign,
                               int overwrite, double* ZTy, void* workspace, const char* who, hipStream_t stream) {
    const ModularPlan pl = modular_plan(M, F);
    char* ws = (char*)workspace;
    int* flag = (int*)ws;
    int* expo = (int*)(ws + pl.expo);
    double* scale = (double*)(ws + pl.scale);
    double* parts = (double*)(ws + pl.parts);
    double* yparts = y ? parts + (size_t)pl.max_parts * F : nullptr;
    signed char* planes = (signed char*)(ws + pl.planes);
    signed char* results = (signed char*)(ws + pl.results);
    const hipError_t lds = allow_stages<GRAM_MODULI>();
    QMLL_REQUIRE(lds == hipSuccess, QMLL_ERR_LAUNCH, "%s: %s", who, hipGetErrorString(lds));
    for (int m0 = 0; m0 < M; m0 += pl.rows) {
        const int m = M - m0 < pl.rows ? M - m0 : pl.rows;
        const double* z = Z + (size_t)m0 * ldz;
        const int nparts = (m + NORM_ROWS - 1) / NORM_ROWS, nk = (m + 127) / 128 * 2;
        const size_t plane = (size_t)nk * 64 * pl.Fp;
        hipLaunchKernelGGL(column_norms_kernel, dim3((F + 255) / 256, nparts), dim3(256), 0, stream, z, ldz, y ? y + m0 : nullptr, m,
                           F, parts, yparts, flag);
        QMLL_CHECK_LAUNCH(who);
        hipLaunchKernelGGL(column_scales_kernel, dim3(pl.Fp / 256), dim3(256), 0, stream, parts, yparts, nparts, F, pl.Fp, scale,
                           expo, ZTy, flag);
        QMLL_CHECK_LAUNCH(who);
        hipLaunchKernelGGL(residues_kernel<GRAM_MODULI>, dim3(pl.Fp / 64, nk), dim3(256), 0, stream, z, ldz, m, F, pl.Fp, 0, 0, scale, flag,
                           planes, plane, (double*)nullptr);
        QMLL_CHECK_LAUNCH(who);
        for (int t0 = 0; t0 < pl.tiles; t0 += pl.range) {
            const int nr = pl.tiles - t0 < pl.range ? pl.tiles - t0 : pl.range;
            const unsigned items = (unsigned)nr * GRAM_MODULI * pl.pieces;
            hipLaunchKernelGGL(modular_gemm_kernel<GRAM_MODULI>, dim3((items + 255) / 256 * 256), dim3(256), NSTAGE * STAGE, stream, planes, plane,
                               pl.Fp, nk, pl.pieces, 0, 0, pl.nt, t0, nr, flag, results);
            QMLL_CHECK_LAUNCH(who);
            hipLaunchKernelGGL(reconstruct_kernel<GRAM_MODULI>, dim3((unsigned)nr * REC_PER_TILE), dim3(256), 0, stream, results, pl.pieces, 0, 0, pl.nt, t0, nr,
                               F, expo, (const double*)nullptr, flag, sign, overwrite && m0 == 0, C, ldc);
            QMLL_CHECK_LAUNCH(who);
        }
        const int rc = qmll_internal_gram_if(z, ldz, m, F, C, ldc, sign, overwrite && m0 == 0, flag, who, stream);
        if (rc != QMLL_OK) return rc;
    }
    return QMLL_OK;
}

// ---- for the Cholesky factorisation ------------------------------------------------------------------
// Residues of the factor's rows, made once as the rows are finished and kept for a slab of them: the update of a later panel of the
// slab is one product over all rows above it, and so is the update of everything below the slab.  15 moduli and 58 bits: with the 14
// and 54 of the Gram product the factor's error |U^T U - A|_ij / sqrt(a_ii a_jj), in the mean square, was three times that of fp64
// sums (1.15e-17 against 3.4e-18 at 16384 features, well conditioned; 2.9e-17 against 6.9e-18 with half the rank), and the
// solution's 2.5 times; with these it is 2.4e-18 and 2.3e-18, the solution's 3.2e-15 against 3.5e-15 and 7e-7 against 2.5e-6.  The scale of a column is
// known beforehand: the squares of its entries in the factor add up to what stands on the diagonal.  If they come to more (the
// matrix is not positive definite) or to no number at all, sums says so and the update writes NaN, which the next pivot finds.
namespace {
struct Slab {
    int Fp, nt;
    size_t plane, expo, scale, sums, planes, results, bytes;
};
Slab slab_layout(int rows, int n) {      // n: columns from the slab's first
    Slab s;
    s.nt = (n + 255) / 256;
    s.Fp = s.nt * 256;
    s.plane = (size_t)rows * s.Fp;
    auto up = [](size_t v) { return (v + 1023) / 1024 * 1024; };
    s.expo = 1024;
    s.scale = s.expo + up((size_t)s.Fp * 4);
    s.sums = s.scale + up((size_t)s.Fp * 8);
    s.planes = s.sums + up((size_t)s.Fp * 8);
    s.results = s.planes + CHOL_MODULI * s.plane;
    s.bytes = s.results + ((size_t)1 << 30);
    return s;
}

__global__ __launch_bounds__(256) void diagonal_scales_kernel(const double* __restrict__ A, long long ld, int n, int Fp,
                                                              double* __restrict__ scale, int* __restrict__ expo,
                                                              double* __restrict__ sums, int* __restrict__ flag) {
    const int f = blockIdx.x * 256 + threadIdx.x;
    if (f == 0) *flag = 0;
    if (f >= Fp) return;
    const double a = f < n ? A[(size_t)f * ld + f] : 1.0;
    const bool fine = a > 0.0 && a <= 1.7976931348623157e308;
    int x = 0;
    if (fine) (void)frexp(a * 0.50000005, &x);              // (half of it, so that the margin never overflows)
    const int e = fine ? (x + 2) >> 1 : 0;                  // sqrt(a) < 2^e
    expo[f] = e;
    scale[f] = ldexp(1.0, GAMMA<CHOL_MODULI> - e);
    sums[f] = fine ? 0.0 : __builtin_nan("");
}
}  // namespace

size_t qmll_internal_slab_bytes(int rows, int n) { return slab_layout(rows, n).bytes; }

// A: the slab's first diagonal entry, n columns from there; before the slab's first panel
int qmll_internal_slab_begin(const double* A, long long ld, int rows, int n, void* workspace, const char* who, hipStream_t stream) {
    const Slab s = slab_layout(rows, n);
    char* ws = (char*)workspace;
    hipLaunchKernelGGL(diagonal_scales_kernel, dim3(s.Fp / 256), dim3(256), 0, stream, A, ld, n, s.Fp, (double*)(ws + s.scale),
                       (int*)(ws + s.expo), (double*)(ws + s.sums), (int*)ws);
    QMLL_CHECK_LAUNCH(who);
    return QMLL_OK;
}

// rows k0 .. k0 + m of the slab (multiples of 64) are final: their residues from column f0 (a multiple of 64) on
int qmll_internal_slab_rows(const double* A, long long ld, int rows, int n, int k0, int m, int f0, void* workspace, const char* who,
                            hipStream_t stream) {
    const Slab s = slab_layout(rows, n);
    char* ws = (char*)workspace;
    if (f0 >= n) return QMLL_OK;
    hipLaunchKernelGGL(residues_kernel<CHOL_MODULI>, dim3((s.Fp - f0) / 64, m / 64), dim3(256), 0, stream, A + (size_t)k0 * ld, ld, m, n, s.Fp, f0,
                       k0 / 64, (const double*)(ws + s.scale), (const int*)ws, (signed char*)(ws + s.planes), s.plane,
                       (double*)(ws + s.sums));
    QMLL_CHECK_LAUNCH(who);
    return QMLL_OK;
}

// the update by the slab's first k rows (a multiple of 128) of the tiles behind row and column i0 (a multiple of 256), of the
// next `band` rows of 256 only if that is not 0
int qmll_internal_slab_update(double* A, long long ld, int rows, int n, int k, int i0, int band, void* workspace, const char* who,
                              hipStream_t stream) {
    const Slab s = slab_layout(rows, n);
    char* ws = (char*)workspace;
    const hipError_t lds = allow_stages<CHOL_MODULI>();
    QMLL_REQUIRE(lds == hipSuccess, QMLL_ERR_LAUNCH, "%s: %s", who, hipGetErrorString(lds));
    const int off = i0 / 256, nt = s.nt - off;
    if (nt <= 0 || k <= 0) return QMLL_OK;
    const int tiles = band ? modular_band_tiles(std::min(band, nt), nt) : nt * (nt + 1) / 2;
    const int launches = (tiles + modular_tiles_at_once(CHOL_MODULI) - 1) / modular_tiles_at_once(CHOL_MODULI), range = (tiles + launches - 1) / launches;
    const int pieces = modular_pieces(CHOL_MODULI, range, k / 64, modular_tiles_at_once(CHOL_MODULI));
    signed char* results = (signed char*)(ws + s.results);
    for (int t0 = 0; t0 < tiles; t0 += range) {
        const int nr = std::min(range, tiles - t0);
        const unsigned items = (unsigned)nr * CHOL_MODULI * pieces;
        hipLaunchKernelGGL(modular_gemm_kernel<CHOL_MODULI>, dim3((items + 255) / 256 * 256), dim3(256), NSTAGE * STAGE, stream,
                           (const signed char*)(ws + s.planes), s.plane, s.Fp, k / 64, pieces, off, std::min(band, nt), s.nt, t0, nr,
                           (const int*)ws, results);
        QMLL_CHECK_LAUNCH(who);
        hipLaunchKernelGGL(reconstruct_kernel<CHOL_MODULI>, dim3((unsigned)nr * REC_PER_TILE), dim3(256), 0, stream, (const signed char*)results, pieces, off,
                           std::min(band, nt), s.nt, t0, nr, n, (const int*)(ws + s.expo), (const double*)(ws + s.sums),
                           (const int*)ws, -1.0, 0, A, ld);
        QMLL_CHECK_LAUNCH(who);
    }
    return QMLL_OK;
}

extern "C" size_t qmll_gram_modular_workspace_bytes(int M, int F) {
    // Below MODULAR_MIN_ROWS rows the bytes out of the products and their reconstruction, 2.3 ms at 16384 features whatever
    // the rows, outweigh the sums: 0.87 (fp64 kernel) against 2.3 ms for 128 rows, 1.60 / 2.64 for 320, 3.64 / 3.20 for
    // 800, 8.6 / 4.7 for 2000; at 1024 features 0.042 / 0.055 for 128 and 0.086 / 0.082 for 320.  The line holds at any width: the fp64 kernel has too few tiles to fill the chip where there
    // are few features, and each of them a long sum, which the integer products cut into row ranges.  us, fp64 kernel / integer
    // products, 768 rows and 32000: 24 features 168 / 89 and 4872 / 201, 256 (one padded tile) 162 / 98 and 4465 / 222, 512
    // 162 / 102 and 4481 / 285, 1024 227 / 97 and 4554 / 497, 2048 246 / 125 and 4650 / 1102, 4096 437 / 297 and 9290 / 3552;
    // 2048 rows 361 / 124, 410 / 136, 417 / 127, 417 / 114, 423 / 158 and 859 / 427.
    if (M < MODULAR_MIN_ROWS || F <= 0) return 0;
    return modular_plan(M, F).bytes;
}

static int gram_modular(const char* who, const double* Z, const double* y, int M, int F, int overwrite, double* ZTZ, double* ZTy,
                        void* workspace, size_t workspace_bytes, qmll_stream_t stream) {
    QMLL_REQUIRE(M >= 0 && F > 0, QMLL_ERR_INVALID, "%s: bad size M=%d F=%d", who, M, F);
    QMLL_REQUIRE(M > 0 || !overwrite, QMLL_ERR_INVALID, "%s: no rows to write from", who);
    if (M == 0) return QMLL_OK;
    QMLL_REQUIRE(Z && ZTZ && workspace, QMLL_ERR_INVALID, "%s: null pointer", who);
    QMLL_REQUIRE((y == nullptr) == (ZTy == nullptr), QMLL_ERR_INVALID, "%s: y and ZTy must both be given or both be NULL", who);
    const size_t need = modular_plan(M, F).bytes;
    QMLL_REQUIRE(workspace_bytes >= need && reinterpret_cast<uintptr_t>(workspace) % 16 == 0, QMLL_ERR_INVALID,
                 "%s: needs %zu bytes of workspace, 16-byte aligned", who, need);
    return modular_syrk(Z, F, y, M, F, ZTZ, F, 1.0, overwrite, ZTy, workspace, who, (hipStream_t)stream);
}

extern "C" int qmll_gram_modular_f64(const double* Z, const double* y, int M, int F, double* ZTZ, double* ZTy, void* workspace,
                                     size_t workspace_bytes, qmll_stream_t stream) {
    return gram_modular("qmll_gram_modular_f64", Z, y, M, F, 0, ZTZ, ZTy, workspace, workspace_bytes, stream);
}

extern "C" int qmll_gram_modular_write_f64(const double* Z, const double* y, int M, int F, double* ZTZ, double* ZTy, void* workspace,
                                           size_t workspace_bytes, qmll_stream_t stream) {
    return gram_modular("qmll_gram_modular_write_f64", Z, y, M, F, 1, ZTZ, ZTy, workspace, workspace_bytes, stream);
}
