// Random Fourier features and their derivative rows (fp64, as the reference's training
// route computes them).  Replaces qml_lightning/cuda/random_features_kernel.cu:5-94.
//
// Two kinds of kernels:
//  * thread = feature column f; a workgroup owns 256 consecutive features and a chunk of
//    rows (atoms, or the 3 x TJ derivative rows of one atom), whose fp32 inputs sit in LDS
//    and are read by broadcast, so each W[k,f] load (coalesced over the workgroup) is reused
//    for every row of the chunk.  Any atom order; molecule sums through fp64 atomics.
//  * rff_rows_kernel, for molecule-major atoms: a workgroup owns (molecule, 64 feature columns,
//    up to 63 derivative rows).  Each wavefront keeps its 16 columns of an element's W as MFMA B
//    fragments in registers; per atom the derivative rows plus the atom's own x row (whose
//    product is the sine argument) form one A tile of 16-row blocks in LDS, multiplied with
//    v_mfma_f64_16x16x4_f64; the per-atom product is scaled by the sine column factor and summed
//    over the molecule's atoms in registers, so G is written once and no atomics are needed.
#include <algorithm>
#include <type_traits>

#include "qmll_common.h"

namespace {

constexpr int RT = 256;     // threads = features per workgroup
constexpr int RA = 8;       // atoms per workgroup (features kernel)
constexpr int TJ = 8;       // target atoms per workgroup (derivative kernel)

__global__ __launch_bounds__(RT) void rff_features_kernel(const float* __restrict__ x, const double* __restrict__ W,
                                                           const double* __restrict__ b,
                                                           const int* __restrict__ mol_index, int A, int d, int F,
                                                           int nmol, double* __restrict__ Zf) {
    extern __shared__ float sx[];   // [RA][d]
    const int a0 = blockIdx.x * RA;
    const int na = min(RA, A - a0);
    for (int t = threadIdx.x; t < na * d; t += RT) sx[t] = x[(size_t)a0 * d + t];
    __syncthreads();
    const int f = blockIdx.y * RT + threadIdx.x;
    if (f >= F) return;
    double acc[RA];
#pragma unroll
    for (int r = 0; r < RA; ++r) acc[r] = 0.0;
    for (int k = 0; k < d; ++k) {
        const double w = W[(size_t)k * F + f];
#pragma unroll
        for (int r = 0; r < RA; ++r)
            if (r < na) acc[r] = fma((double)sx[r * d + k], w, acc[r]);
    }
    const double norm = sqrt(2.0 / (double)F);
    const double bf = b[f];
    int cur = -1;
    double run = 0.0;
#pragma unroll
    for (int r = 0; r < RA; ++r) {
        if (r < na) {
            const int mol = mol_index[a0 + r];
            if (mol != cur) {
                if (cur >= 0 && cur < nmol) unsafeAtomicAdd(&Zf[(size_t)cur * F + f], run);
                cur = mol;
                run = 0.0;
            }
            run += norm * cos(acc[r] + bf);
        }
    }
    if (cur >= 0 && cur < nmol) unsafeAtomicAdd(&Zf[(size_t)cur * F + f], run);
}

__global__ __launch_bounds__(RT) void rff_derivative_kernel(const float* __restrict__ x, const float* __restrict__ grad,
                                                             const double* __restrict__ W, const double* __restrict__ b,
                                                             const int* __restrict__ mol_index, int n, int d, int F,
                                                             int nmol, int njc, double* __restrict__ G) {
    extern __shared__ float sm[];   // [d] x row, then [TJ*3][d] derivative rows
    float* sx = sm;
    float* sg = sm + d;
    const size_t a = blockIdx.x / njc;
    const int j0 = (blockIdx.x % njc) * TJ;
    const int nj = min(TJ, n - j0);
    for (int t = threadIdx.x; t < d; t += RT) sx[t] = x[a * d + t];
    for (int t = threadIdx.x; t < nj * 3 * d; t += RT) sg[t] = grad[((a * n + j0) * 3) * d + t];
    __syncthreads();
    const int mol = mol_index[a];
    const int f = blockIdx.y * RT + threadIdx.x;
    if (f >= F || mol < 0 || mol >= nmol) return;
    double s0 = 0.0;
    double acc[TJ * 3];
#pragma unroll
    for (int r = 0; r < TJ * 3; ++r) acc[r] = 0.0;
    for (int k = 0; k < d; ++k) {
        const double w = W[(size_t)k * F + f];
        s0 = fma((double)sx[k], w, s0);
#pragma unroll
        for (int r = 0; r < TJ * 3; ++r)
            if (r < nj * 3) acc[r] = fma((double)sg[r * d + k], w, acc[r]);
    }
    const double fd = sqrt(2.0 / (double)F) * sin(s0 + b[f]);
#pragma unroll
    for (int r = 0; r < TJ * 3; ++r) {
        if (r < nj * 3 && acc[r] != 0.0) {
            const int j = j0 + r / 3, c = r % 3;
            unsafeAtomicAdd(&G[(((size_t)mol * n + j) * 3 + c) * F + f], fd * acc[r]);
        }
    }
}

typedef double double4_t __attribute__((ext_vector_type(4)));

constexpr int MROWS = 64;   // A-tile rows: up to 63 derivative rows + the atom's x row
constexpr int MPAD = 4;     // floats of padding per LDS row: 16 rows x 4 k land in 64 distinct banks

// the elements of a batch (molecule-major atoms within each)
constexpr int RFF_MAXE = 8;
struct RffElements {
    const float* x[RFF_MAXE];      // [A_e, d]
    const float* grad[RFF_MAXE];   // [A_e, 3n, d]
    const void* W[RFF_MAXE];       // [d, F]
    const void* b[RFF_MAXE];       // [F]
    const int* seg[RFF_MAXE];      // first atom of each molecule [nmol + 1]
    int ne;
};

// grid (ceil(F/64), nmol, ceil(max rows / 63)), 256 threads.  All elements of the batch in one launch: G (and, when
// asked for, the energy features, whose argument is the same product) is written once, or read and written once.
// The tile holds as many 16-row blocks as the molecule's rows need (one matrix instruction per block and four k).
// Bound by the fp64 matrix cores: 200 molecules of 3 to 29 atoms, 128 components, 8192 features: 7.3 ms, where a tile
// of 64 rows for every molecule padded to 29 atoms, a launch per element and a kernel of its own for the energy
// features took 16.3 ms (of which the rows left out by the row table are a half).  A column's argument is one value per
// atom, which all four lane groups would work the sine and cosine out of (a tenth of the launch): two or four atoms are
// multiplied first, as the registers allow, and a lane group works them out for one of them (9.0 -> 8.25 ms in a trace, same bits).
// W is fp32 in a model (converted exactly in the registers) or fp64.
template <int D, typename TW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 128 ? 2 : 1))) void rff_rows_kernel(
    RffElements E, const int* __restrict__ row_offsets, int n, int F, int overwrite, double* __restrict__ Ze,
    double* __restrict__ G) {
    constexpr int LD = D + MPAD;
    constexpr int KS = D / 4;                 // MFMA k-steps
    // two tiles: the next atom's is written while this one's is read, one barrier per atom
    __shared__ __attribute__((aligned(16))) float tiles[2][MROWS * LD];

    const int mol = blockIdx.y;
    const int rows3n = 3 * n;
    const size_t grow0 = row_offsets ? (size_t)row_offsets[mol] : (size_t)mol * rows3n;
    const int rows = row_offsets ? row_offsets[mol + 1] - row_offsets[mol] : rows3n;
    const int row0 = blockIdx.z * (MROWS - 1);
    const bool with_energy = Ze != nullptr && blockIdx.z == 0;
    if (row0 >= rows && !with_energy) return;
    const int nrows = max(0, min(MROWS - 1, rows - row0));
    int natoms = 0;
    for (int e = 0; e < E.ne; ++e) natoms += E.seg[e][mol + 1] - E.seg[e][mol];
    if (natoms == 0 && !overwrite) return;

    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int l16 = lane & 15, lk = lane >> 4;
    const int f = blockIdx.x * 64 + wave * 16 + l16;
    const bool fok = f < F;
    const unsigned wcol = lk * F + (fok ? f : F - 1);       // (a column beyond the last computes that one and writes nothing)
    const double norm = sqrt(2.0 / (double)F);
    double zacc = 0.0;

    auto body = [&](auto nbc) {
        constexpr int NB = decltype(nbc)::value;           // 16-row blocks; the x row is the last of them
        constexpr int V4 = (NB * 16 * D / 4 + 255) / 256;  // float4 loads per thread per tile
        constexpr bool AHEAD = D <= 128 || NB <= 3;        // (where the registers last: four blocks of 256 components, 60 molecules of 24, 9370 us, 9970 with it)
        double4_t gacc[NB];
#pragma unroll
        for (int p = 0; p < NB; ++p) gacc[p] = (double4_t){0.0, 0.0, 0.0, 0.0};
        float4 stage[V4];
        auto fetch = [&](int e, int a) {
            const float* ge = E.grad[e] + ((size_t)a * rows3n + row0) * D;
            const float* xe = E.x[e] + (size_t)a * D;
#pragma unroll
            for (int v = 0; v < V4; ++v) {
                const int idx = v * 256 + threadIdx.x;
                const int row = idx / (D / 4), c4 = idx % (D / 4);
                float4 val = make_float4(0.f, 0.f, 0.f, 0.f);
                if (row < nrows)
                    val = *reinterpret_cast<const float4*>(ge + (size_t)row * D + c4 * 4);
                else if (row == NB * 16 - 1)
                    val = *reinterpret_cast<const float4*>(xe + c4 * 4);
                stage[v] = val;
            }
        };
        // the molecule's atoms element by element; (e, a) is the atom whose rows are in flight
        int e = 0, a = 0, aend = 0;
        auto settle = [&]() {                               // the next element that has atoms, when this one is done
            while (a >= aend && e < E.ne) {
                ++e;
                if (e < E.ne) {
                    a = E.seg[e][mol];
                    aend = E.seg[e][mol + 1];
                }
            }
        };
        e = -1;
        settle();
        if (e < E.ne) fetch(e, a);
        int cur = -1;
        TW wreg[KS];
        double bf = 0.0;
        // the atoms in groups of NG: the sine and cosine of a column are worked out once per group, a lane group per atom
        constexpr int NG = (NB <= 2 ? 4 : 2) / (sizeof(TW) == 4 ? 1 : 2);      // (what fits 256 registers)
        for (int done = 0; done < natoms; done += NG) {
            double4_t pacc[NG][NB];
            double arg = 0.0;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                if (done + g >= natoms) break;
                const int el = e;
                float* tile = tiles[(done + g) & 1];
#pragma unroll
                for (int v = 0; v < V4; ++v) {
                    const int idx = v * 256 + threadIdx.x;
                    const int row = idx / (D / 4), c4 = idx % (D / 4);
                    if (V4 * 256 == NB * 16 * D / 4 || row < NB * 16)
                        *reinterpret_cast<float4*>(&tile[row * LD + c4 * 4]) = stage[v];
                }
                __syncthreads();
                if (el != cur) {   // B fragments of this wavefront's 16 columns, all of K, resident for the element's atoms
                    const TW* We = static_cast<const TW*>(E.W[el]);
#pragma unroll
                    for (int kk = 0; kk < KS; ++kk) wreg[kk] = (We + (size_t)(kk * 4) * F)[wcol];
                    bf = (double)static_cast<const TW*>(E.b[el])[fok ? f : F - 1];
                    cur = el;
                }
                ++a;
                settle();
                if (e < E.ne) fetch(e, a);   // in flight during the MFMAs

#pragma unroll
                for (int p = 0; p < NB; ++p) pacc[g][p] = (double4_t){0.0, 0.0, 0.0, 0.0};
                // the operands of two steps are read beside the products of the two before: read where they are used, they kept a
                // wavefront waiting for LDS every eight instructions (400 molecules of 10, 200 of 21 and 120 of 29 atoms at 8192 features 5340 -> 5085 us, 9480 -> 9045, 11757 -> 11333)
                float now[NB][2], next[NB][2];
                auto read = [&](int kk, float (&to)[NB][2]) {
#pragma unroll
                    for (int p = 0; p < NB; ++p)
#pragma unroll
                        for (int q = 0; q < 2; ++q) to[p][q] = tile[(p * 16 + l16) * LD + (kk + q) * 4 + lk];
                };
                read(0, now);
#pragma unroll
                for (int kk = 0; kk < KS; kk += 2) {
                    if (kk + 2 < KS) read(kk + 2, next);
                    if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int p = 0; p < NB; ++p)
                            pacc[g][p] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)now[p][q], (double)wreg[kk + q], pacc[g][p], 0, 0, 0);
                    if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int p = 0; p < NB; ++p)
#pragma unroll
                        for (int q = 0; q < 2; ++q) now[p][q] = next[p][q];
                }
                // accumulator register r of a 16x16 block holds row lane/16 + 4r, column lane%16:
                // the x row (the last of the tile) is register 3 of the last block in lanes 48..63
                const double s0 = __shfl(pacc[g][NB - 1][3], 48 + l16, 64) + bf;
                if ((lk & (NG - 1)) == g) arg = s0;
            }
            double sn, cs;
            sincos(arg, &sn, &cs);
            sn *= norm;
            cs *= norm;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                if (done + g >= natoms) break;
                zacc += __shfl(cs, 16 * g + l16, 64);
                const double fd = __shfl(sn, 16 * g + l16, 64);
#pragma unroll
                for (int p = 0; p < NB; ++p) gacc[p] += fd * pacc[g][p];
            }
        }
        if (!fok) return;
        if (with_energy && lk == 0) {
            double* z = Ze + (size_t)mol * F + f;
            *z = overwrite ? zacc : *z + zacc;
        }
#pragma unroll
        for (int p = 0; p < NB; ++p) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = p * 16 + lk + 4 * r;
                if (row < nrows) {
                    double* dst = G + (grow0 + row0 + row) * F + f;
                    *dst = overwrite ? gacc[p][r] : *dst + gacc[p][r];
                }
            }
        }
    };
    switch ((nrows + 16) / 16) {
        case 1: body(std::integral_constant<int, 1>{}); break;
        case 2: body(std::integral_constant<int, 2>{}); break;
        case 3: body(std::integral_constant<int, 3>{}); break;
        default: body(std::integral_constant<int, 4>{}); break;
    }
}

template <typename TW>
void launch_rff_rows(const RffElements& E, const int* row_offsets, int max_rows, int n, int d, int F, int nmol, int overwrite,
                     double* Ze, double* G, hipStream_t stream) {
    const dim3 grid((F + 63) / 64, nmol, max_rows > 0 ? (max_rows + MROWS - 2) / (MROWS - 1) : 1);
    if (d == 64)
        hipLaunchKernelGGL((rff_rows_kernel<64, TW>), grid, dim3(256), 0, stream, E, row_offsets, n, F, overwrite, Ze, G);
    else if (d == 128)
        hipLaunchKernelGGL((rff_rows_kernel<128, TW>), grid, dim3(256), 0, stream, E, row_offsets, n, F, overwrite, Ze, G);
    else
        hipLaunchKernelGGL((rff_rows_kernel<256, TW>), grid, dim3(256), 0, stream, E, row_offsets, n, F, overwrite, Ze, G);
}


// ---- fused predict path ------------------------------------------------------------------
// e[a] = sqrt(2/F) sum_f alpha_f cos(x_a . W_t[:,f] + b_t[f]),  gx[a,:] = d e[a] / d x_a, for
// element-sorted rows x [A,d] (tiles of 128 atoms share the element t, so one W).  Replaces
// the per-element matmul + cos + index_add + matmul(alpha) of the reference's TorchScript
// forward (qml_lightning/models/random_features.py:88-100) and its autograd transpose
// without ever writing the [atoms, F] feature matrix.
//
// Two chained matrix-core products per 32-feature chunk of W (staged in LDS):
// S^T[f,a] = W^T x^T  ->  P[f,a] = -norm alpha_f sin(S + b_f)  ->  GX^T[k,a] += W P.
// Everything is kept transposed so that the accumulator registers of the first product (row
// = feature, column = atom) are exactly the B operand the second one needs (contraction
// index = feature): P never leaves the registers.  x^T (B operand of the first product)
// stays in registers for the whole kernel, GX^T in accumulators.
typedef float f4_t __attribute__((ext_vector_type(4)));

constexpr int RE_T = 256;        // threads: 4 wavefronts x 32 atoms
constexpr int RE_M = 128;        // atoms per workgroup
constexpr int RE_FC = 32;        // features per staged chunk (one block of 32 rows)

// The products run on the half-precision matrix cores, whose fp16 instructions do thirteen times the flops per clock of
// v_mfma_f32_32x32x2_f32: each fp32 operand is split into two fp16 parts (hi = the value
// rounded to fp16, lo = the rounded rest: 22 bits together) and a product becomes three matrix
// instructions, hi.hi + hi.lo + lo.hi, accumulated in fp32; lo.lo is below the rounding of the sum.
// The instruction is the 16 x 16 x 32 one: on operands with all their bits in use the card's power holds a loop of
// nothing but the 32 x 32 x 16 form to 1.62 PFLOP/s and of this one to 1.90 (2.46 and 2.48 on zeros), and here the clock
// rises from 1.60 to 1.74 GHz.  86016 atoms, 32768 features, 128 components with the gradient: 4.35 ms with the larger form,
// 3.80 with this one; energies only 2.35 / 2.08; 64 components, 16384 features 1.31 / 1.10 and 0.65 / 0.60.  What is left is
// issue as much as power: beside vector work of another wavefront a matrix instruction of either form takes about ten clocks
// of the SIMD's issue, which makes 2000 clocks per wavefront and chunk with the 1050 of the vector instructions.
// fp16 has five exponent bits, so every operand is scaled by a power of two first (exact): x by the
// wavefront's 2^kx (largest |x| of its 32 atoms to [2^13, 2^14)), alpha by the workgroup's 2^kp (largest
// |alpha| norm of its feature range), every chunk of W by its own 2^kw (largest |W| of the chunk); the
// sine argument, the chunk's contribution to the gradient and the outputs take the inverse factors.
// fp16 subnormals are kept by the matrix cores, so small entries beside large ones lose only bits
// below 2^-38 of the largest.
//
// W is a constant of the model, so it is split ONCE (rff_presplit_kernel) into the very bytes the
// predict kernel wants in LDS: per element and 32-feature chunk an image holding the chunk twice,
// as A operands of the first product (rows = features, 32 k per step) and of the second (rows = k, the
// chunk's 32 features), the features in the order in which the first product's accumulators hold them
// (lane group g: 4 g + 0..3 of either tile of 16), so the split P goes straight from registers into the
// B operand; hi and lo parts each, every operand 1 KB in the order of the lanes.  The predict kernel then moves an image into LDS with direct
// global-to-LDS loads (no registers, no vector instructions), the next chunk's while this one is
// multiplied.
template <int D>
struct RffImage {
    static constexpr int OP = 512;                   // halves of one operand: 64 lanes x 8
    static constexpr int KS = D / 32, KT = D / 16;   // contraction steps of the first product, row tiles of the second
    // first product, operand (part, feature tile, step): lane (i, g) holds W[32 step + 8 g + 0..7][16 tile + i]; second product,
    // operand (part, row tile): W[16 tile + i][features 4 g + 0..3 and 16 + 4 g + 0..3]
    __host__ __device__ static constexpr int w1(int part, int tile, int step) { return ((part * 2 + tile) * KS + step) * OP; }
    __host__ __device__ static constexpr int w2(int part, int tile) { return (4 * KS + part * KT + tile) * OP; }
    static constexpr int HALVES = (4 * KS + 2 * KT) * OP;
    static constexpr int BYTES = HALVES * 2;         // 32768 (D = 128), 16384 (D = 64)
    static constexpr int BLOCKS = BYTES / 1024;      // 1 KiB = one operand = one wavefront's 64 x 16-byte load
    static_assert(BLOCKS % 4 == 0, "the same number for each of four wavefronts");
};

// One workgroup per (chunk, element): the chunk's power of two, then the image through LDS.
template <int D>
__global__ __launch_bounds__(RE_T) void rff_presplit_kernel(const float* __restrict__ W, int F, _Float16* __restrict__ images,
                                                            int* __restrict__ exponents) {
    using Img = RffImage<D>;
    constexpr int NP = D / 64;                // pairs of adjacent k rows staged per thread
    __shared__ __attribute__((aligned(16))) _Float16 img[Img::HALVES];
    __shared__ float swmax[RE_T / 64];
    const int chunk = blockIdx.x, type = blockIdx.y, nchunks = gridDim.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float* Wt = W + (size_t)type * D * F;
    const int f0 = chunk * RE_FC;
    // thread -> features sf .. sf+3 of the rows k0 = 2 (tid / 8) + 64 p and k0 + 1
    const int sf = (tid & 7) * 4, skp = 2 * (tid >> 3);
    float4 stage[NP][2];
    float m = 0.0f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            stage[p][r] = *reinterpret_cast<const float4*>(Wt + (size_t)(skp + 64 * p + r) * F + f0 + sf);
            m = fmaxf(fmaxf(fmaxf(m, fabsf(stage[p][r].x)), fmaxf(fabsf(stage[p][r].y), fabsf(stage[p][r].z))),
                      fabsf(stage[p][r].w));
        }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if (lane == 0) swmax[wave] = m;
    __syncthreads();
    const int kw = scale_exponent(fmaxf(fmaxf(swmax[0], swmax[1]), fmaxf(swmax[2], swmax[3])));
    const float sw = pow2i(kw);
    if (tid == 0) exponents[type * nchunks + chunk] = kw;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int k0 = skp + 64 * p;
        const float w0[4] = {stage[p][0].x * sw, stage[p][0].y * sw, stage[p][0].z * sw, stage[p][0].w * sw};
        const float w1[4] = {stage[p][1].x * sw, stage[p][1].y * sw, stage[p][1].z * sw, stage[p][1].w * sw};
        half4_t r0h, r0l, r1h, r1l;
        // rows k0, k0 + 1 among the 32 of a step, features sf .. sf + 3 among the 16 of a tile and among a lane's eight
        const int at1 = ((k0 & 31) >> 3) * 128 + (k0 & 7), at2 = ((sf & 15) >> 2) * 128 + (sf >> 4) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            _Float16 a, c;
            split_f16(w0[e], a, c);
            r0h[e] = a; r0l[e] = c;
            split_f16(w1[e], a, c);
            r1h[e] = a; r1l[e] = c;
            const int to = at1 + ((sf + e) & 15) * 8;
            *reinterpret_cast<half2_t*>(&img[Img::w1(0, sf >> 4, k0 >> 5) + to]) = (half2_t){r0h[e], r1h[e]};
            *reinterpret_cast<half2_t*>(&img[Img::w1(1, sf >> 4, k0 >> 5) + to]) = (half2_t){r0l[e], r1l[e]};
        }
        *reinterpret_cast<half4_t*>(&img[Img::w2(0, k0 >> 4) + at2 + (k0 & 15) * 8]) = r0h;
        *reinterpret_cast<half4_t*>(&img[Img::w2(1, k0 >> 4) + at2 + (k0 & 15) * 8]) = r0l;
        *reinterpret_cast<half4_t*>(&img[Img::w2(0, k0 >> 4) + at2 + (k0 & 15) * 8 + 8]) = r1h;
        *reinterpret_cast<half4_t*>(&img[Img::w2(1, k0 >> 4) + at2 + (k0 & 15) * 8 + 8]) = r1l;
    }
    __syncthreads();
    float4* dst = reinterpret_cast<float4*>(images + (size_t)(type * nchunks + chunk) * Img::HALVES);
    for (int t = tid; t < Img::BYTES / 16; t += RE_T) dst[t] = reinterpret_cast<const float4*>(img)[t];
}

// tile `tile` of RE_M atoms of one element; false past the last
__device__ __forceinline__ bool find_tile(const int* __restrict__ type_offsets, int ne, int tile, int& type, int& row0, int& rows) {
    for (int t = 0; t < ne; ++t) {
        const int o0 = type_offsets[t], o1 = type_offsets[t + 1], nt = (o1 - o0 + RE_M - 1) / RE_M;
        if (tile < nt) {
            type = t;
            row0 = o0 + tile * RE_M;
            rows = min(RE_M, o1 - row0);
            return true;
        }
        tile -= nt;
    }
    return false;
}

// a part of a tile's result: its energies, then (with the gradient) its rows
__host__ __device__ constexpr size_t part_floats(int d, bool with_grad) { return (size_t)RE_M * (with_grad ? d + 1 : 1); }

template <int D, bool WITH_GRAD>
__global__ __launch_bounds__(RE_T) __attribute__((amdgpu_waves_per_eu(2))) void rff_energy_sorted_f16_kernel(
    const float* __restrict__ x, const int* __restrict__ type_offsets, const int* __restrict__ sorted_slots,
    const _Float16* __restrict__ images, const int* __restrict__ exponents, const float* __restrict__ b,
    const float* __restrict__ alpha, int ne, int F, int nwhole, int nparts, float norm, float* __restrict__ parts,
    float* __restrict__ e_slots,
    float* __restrict__ gx) {
    using Img = RffImage<D>;
    constexpr int KS = Img::KS, KT = Img::KT;
    // two images, this chunk's and the next one's, as two arrays of their own: the compiler then knows
    // that the loads into one do not touch what is read from the other and does not wait for them
    __shared__ __attribute__((aligned(16))) _Float16 simg0[Img::HALVES], simg1[Img::HALVES];
    __shared__ __attribute__((aligned(16))) float sba[2 * 2 * RE_FC];     // [2][2][RE_FC]: b / 2 pi, alpha norm 2^kp of the two chunks

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = lane & 15, g = lane >> 4;
    const int nchunks = F / RE_FC;
    // workgroups below `whole` take a tile's chunks all, the others a share of 1 / nparts of them
    const bool whole = (int)blockIdx.x < nwhole;
    const int piece = whole ? 0 : (int)blockIdx.x - nwhole;
    const int c0 = whole ? 0 : (int)((long long)nchunks * (piece % nparts) / nparts);
    const int c1 = whole ? nchunks : (int)((long long)nchunks * (piece % nparts + 1) / nparts);
    int type, row0, rows;
    if (!find_tile(type_offsets, ne, whole ? (int)blockIdx.x : nwhole + piece / nparts, type, row0, rows)) return;
    float* part_out = parts ? parts + (size_t)piece * part_floats(D, WITH_GRAD) : nullptr;
    const float* bt = b + (size_t)type * F;
    const int arow = 32 * wave + i;                      // this lane's atoms: arow and arow + 16
    const int fbeg = c0 * RE_FC, fend = c1 * RE_FC;
    // a scalar base and one per-lane offset: the loads then need no per-lane 64-bit addresses
    const unsigned char* img0 = reinterpret_cast<const unsigned char*>(images) + (size_t)type * nchunks * Img::BYTES;
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);
    const unsigned lane16 = (unsigned)lane * 16u;
    const int* kws = exponents + type * nchunks;
    // chunk `c` of this element into LDS copy `par`: every wavefront moves the 1 KiB blocks wave, wave + 4, ...
    // (64 lanes x 16 bytes per instruction, written to LDS at block start + 16 lane)
    auto dma = [&](int c, _Float16* to) {
        const unsigned char* src = img0 + (size_t)c * Img::BYTES;
        unsigned char* dst = reinterpret_cast<unsigned char*>(to);
#pragma unroll
        for (int u0 = 0; u0 < Img::BLOCKS; u0 += RE_T / 64) {
            const int u = u0 + wave_s;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + u * 1024 + lane16),
                                             (__attribute__((address_space(3))) void*)(dst + u * 1024), 16, 0, 0);
        }
    };
    dma(fbeg / RE_FC, simg0);

    // x^T as the B operand of the first product: step j contracts k = 32 j + 8 g + (0..7)
    half8_t xh[2][KS], xl[2][KS];
    float inv_sx;
    {
        float xv[2][KS][8];
        float m = 0.0f;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const bool aok = arow + 16 * t < rows;
            const float* xr = x + (size_t)(row0 + (aok ? arow + 16 * t : 0)) * D + 8 * g;
#pragma unroll
            for (int j = 0; j < KS; ++j) {
                const float4 v0 = aok ? *reinterpret_cast<const float4*>(xr + 32 * j) : make_float4(0.f, 0.f, 0.f, 0.f);
                const float4 v1 = aok ? *reinterpret_cast<const float4*>(xr + 32 * j + 4) : make_float4(0.f, 0.f, 0.f, 0.f);
                xv[t][j][0] = v0.x; xv[t][j][1] = v0.y; xv[t][j][2] = v0.z; xv[t][j][3] = v0.w;
                xv[t][j][4] = v1.x; xv[t][j][5] = v1.y; xv[t][j][6] = v1.z; xv[t][j][7] = v1.w;
#pragma unroll
                for (int q = 0; q < 8; ++q) m = fmaxf(m, fabsf(xv[t][j][q]));
            }
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        if (__builtin_expect(not_finite(m), 0)) {        // an infinity among the rows: the largest finite entry
            m = 0.0f;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < KS; ++j)
#pragma unroll
                    for (int q = 0; q < 8; ++q) m = fmaxf(m, finite_abs(xv[t][j][q]));
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        }
        const int kx = scale_exponent(m);
        const float sx = pow2i(kx);
        inv_sx = pow2i(-kx);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < KS; ++j)
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    _Float16 a, c;
                    split_f16(xv[t][j][q] * sx, a, c);
                    xh[t][j][q] = a;
                    xl[t][j][q] = c;
                }
    }
    // the workgroup's alpha scale (every wavefront finds the same value)
    float sp, inv_sp;
    {
        float m = 0.0f;
        for (int f = fbeg + lane; f < fend; f += 64) m = fmaxf(m, fabsf(alpha[f]));
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        const int kp = scale_exponent(m * norm);
        sp = pow2i(kp);
        inv_sp = pow2i(-kp);
    }
    if (tid < RE_FC) {
        sba[tid] = bt[fbeg + tid] * 0.15915494309189535f;
        sba[RE_FC + tid] = alpha[fbeg + tid] * norm * sp;
    }

    const f4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f4_t gacc[KT][2];
    if constexpr (WITH_GRAD) {
#pragma unroll
        for (int k = 0; k < KT; ++k)
#pragma unroll
            for (int t = 0; t < 2; ++t) gacc[k][t] = zero;
    }
    float energy[2] = {0.0f, 0.0f};

    // one chunk: `img` holds it, the next one is loaded into `other`
    auto round = [&](int f0, int par, const _Float16* img, _Float16* other) {
        const bool more = f0 + RE_FC < fend;
        // this chunk's image has landed (every wavefront waits for its own loads, then for the others),
        // and the other copy, read in the round before, is free
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        // b and alpha of the next chunk are requested before its image so that waiting for them does
        // not wait for the image; they go to LDS at the end of the round
        float bnext = 0.0f, anext = 0.0f;
        if (more && tid < RE_FC) {
            bnext = bt[f0 + RE_FC + tid];
            anext = alpha[f0 + RE_FC + tid];
        }
        if (more) dma(f0 / RE_FC + 1, other);
        const _Float16* mine = img + lane * 8;
        auto operand = [&](int at) { return *reinterpret_cast<const half8_t*>(mine + at); };
        const float* sb = sba + par * 2 * RE_FC;
        const float* sa = sb + RE_FC;
        const int kw = kws[f0 / RE_FC];
        const float inv_sw = pow2i(-kw);

        // first product: 2^(kx + kw) S^T (32 features x 32 atoms)
        const float inv_sxw = inv_sx * inv_sw;
        f4_t sacc[2][2];                                 // [feature tile][atom tile]
        // (the products with a low part first, while the sum is small: only the KS others round at its full size.  Gradients of 1008 atoms,
        // d = 128, 8192 features against 64 bits, arguments of 2.3 / 4.5 / 6.8 radians: 3.9e-7 / 6.0e-7 / 8.3e-7; the three of a step
        // one behind the other 4.7e-7 / 7.9e-7 / 1.13e-6.  32768 features, 4032 atoms take 240 us either way.)
        half8_t ah[KS][2];
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            const half8_t al[2] = {operand(Img::w1(1, 0, j)), operand(Img::w1(1, 1, j))};
            ah[j][0] = operand(Img::w1(0, 0, j));
            ah[j][1] = operand(Img::w1(0, 1, j));
#pragma unroll
            for (int u = 0; u < 4; ++u)
                sacc[u >> 1][u & 1] =
                    __builtin_amdgcn_mfma_f32_16x16x32_f16(al[u >> 1], xh[u & 1][j], j == 0 ? zero : sacc[u >> 1][u & 1], 0, 0, 0);
#pragma unroll
            for (int u = 0; u < 4; ++u)
                sacc[u >> 1][u & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[j][u >> 1], xl[u & 1][j], sacc[u >> 1][u & 1], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < KS; ++j)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                sacc[u >> 1][u & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[j][u >> 1], xh[u & 1][j], sacc[u >> 1][u & 1], 0, 0, 0);
        // accumulator register r of tile (u, t): feature 16 u + 4 g + r of the chunk, atom 16 t + i.  The sine
        // argument is formed in REVOLUTIONS (b arrives divided by 2 pi, the product takes 1 / 2 pi with its
        // inverse scales): v_sin_f32 / v_cos_f32 reduce the range themselves up to 256 revolutions; the
        // rounding of the argument, |arg| 6e-8 radians, is that of an fp32 argument in radians.  Beyond
        // 1500 radians whole revolutions are taken off first (u - rint(u) is exact in fp32).
        constexpr float UMAX = 1500.0f * 0.15915494309189535f;
        const float crev = inv_sxw * 0.15915494309189535f;
        float umax = 0.0f;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const f4_t bv = *reinterpret_cast<const f4_t*>(&sb[16 * u + 4 * g]);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sacc[u][t][e] = fmaf(sacc[u][t][e], crev, bv[e]);
                    umax = fmaxf(umax, fabsf(sacc[u][t][e]));
                }
        }
        if (__builtin_expect(__any(umax > UMAX), 0)) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (fabsf(sacc[u >> 1][u & 1][e]) > UMAX) sacc[u >> 1][u & 1][e] -= rintf(sacc[u >> 1][u & 1][e]);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const f4_t av = *reinterpret_cast<const f4_t*>(&sa[16 * u + 4 * g]);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float arg = sacc[u][t][e];
                    const float sn = __builtin_amdgcn_sinf(arg), cs = __builtin_amdgcn_cosf(arg);
                    energy[t] = fmaf(av[e], cs, energy[t]);
                    sacc[u][t][e] = -av[e] * sn;         // 2^kp P
                }
        }
        if constexpr (WITH_GRAD) {
            // at d = 128 the kernel takes all 256 registers: without this line the compiler keeps the arguments of the cosines
            // across the second product and spills for it, and a reload waits for the next image too.  The
            // second product goes ahead of the other wavefront's vector instructions: 86016 atoms, 32768 features
            // 4.01 -> 3.82 ms; the same around the first product or around the sines gave nothing
            if constexpr (D == 128) {
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_setprio(1);
            }
            // second product: 2^kp GX^T[k, a] += 2^-kw sum_f 2^kw W[k, f] 2^kp P[f, a]; one step contracts the
            // chunk's 32 features, a lane's eight in the order of its registers.  The chunk's contribution is summed from zero and
            // added to the running sums by the vector unit: the matrix instruction aligns its products
            // to the accumulator it is given, and against a sum over a thousand chunks their low bits
            // would be cut off
            half8_t ph[2], pl[2];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int q = 0; q < 8; q += 2) {
                    half2_t a, c;
                    split_pair(sacc[q >> 2][t][q & 3], sacc[q >> 2][t][(q & 3) + 1], a, c);
                    ph[t][q] = a[0];
                    ph[t][q + 1] = a[1];
                    pl[t][q] = c[0];
                    pl[t][q + 1] = c[1];
                }
#pragma unroll
            for (int k = 0; k < KT; ++k) {
                const half8_t ah = operand(Img::w2(0, k)), al = operand(Img::w2(1, k));
                f4_t part[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) part[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, ph[t], zero, 0, 0, 0);
#pragma unroll
                for (int t = 0; t < 2; ++t) part[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, pl[t], part[t], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < 2; ++t) part[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, ph[t], part[t], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) gacc[k][t][r] = fmaf(part[t][r], inv_sw, gacc[k][t][r]);
            }
        }
        if constexpr (WITH_GRAD && D == 128) __builtin_amdgcn_s_setprio(0);
        // (used here and no earlier: the compiler waits for them right after their loads otherwise)
        asm volatile("" : "+v"(bnext), "+v"(anext)::"memory");
        if (more && tid < RE_FC) {
            float* nb = sba + (par ^ 1) * 2 * RE_FC;
            nb[tid] = bnext * 0.15915494309189535f;
            nb[RE_FC + tid] = anext * norm * sp;
        }
    };
    for (int f0 = fbeg; f0 < fend; f0 += 2 * RE_FC) {
        round(f0, 0, simg0, simg1);
        if (f0 + RE_FC < fend) round(f0 + RE_FC, 1, simg1, simg0);
    }

#pragma unroll
    for (int t = 0; t < 2; ++t) {
        float e = energy[t];
        e += __shfl_xor(e, 16, 64);
        e += __shfl_xor(e, 32, 64);
        e *= inv_sp;
        const int row = arow + 16 * t;
        if (row >= rows) continue;
        if (whole || part_out) {
            if (g == 0) {
                if (whole) e_slots[sorted_slots[row0 + row]] = e;
                else part_out[row] = e;
            }
            if constexpr (WITH_GRAD) {
                float* gr = (whole ? gx + (size_t)row0 * D : part_out + RE_M) + (size_t)row * D + 4 * g;
#pragma unroll
                for (int k = 0; k < KT; ++k) *reinterpret_cast<f4_t*>(gr + 16 * k) = gacc[k][t] * inv_sp;
            }
        } else {
            // no workspace: the parts add into zero-filled outputs
            if (g == 0) atomicAdd(&e_slots[sorted_slots[row0 + row]], e);
            if constexpr (WITH_GRAD) {
                float* gr = gx + (size_t)(row0 + row) * D + 4 * g;
#pragma unroll
                for (int k = 0; k < KT; ++k)
#pragma unroll
                    for (int r = 0; r < 4; ++r) atomicAdd(gr + 16 * k + r, gacc[k][t][r] * inv_sp);
            }
        }
    }
}

// the parts of the tiles nwhole + blockIdx.x, added up in order; grid (tiles, column slices).  HBM bound.
template <int D, bool WITH_GRAD>
__global__ __launch_bounds__(256) void rff_sum_parts_kernel(const int* __restrict__ type_offsets, const int* __restrict__ sorted_slots,
                                                            int ne, int nwhole, int nparts, const float* __restrict__ parts,
                                                            float* __restrict__ e_slots, float* __restrict__ gx) {
    constexpr size_t SLOT = part_floats(D, WITH_GRAD);
    int type, row0, rows;
    if (!find_tile(type_offsets, ne, nwhole + (int)blockIdx.x, type, row0, rows)) return;
    const float* src = parts + (size_t)blockIdx.x * nparts * SLOT;
    if (blockIdx.y == 0 && (int)threadIdx.x < rows) {
        float v = 0.0f;
#pragma unroll 8
        for (int k = 0; k < nparts; ++k) v += src[k * SLOT + threadIdx.x];
        e_slots[sorted_slots[row0 + threadIdx.x]] = v;
    }
    if constexpr (WITH_GRAD) {
        for (int t = blockIdx.y * 256 + threadIdx.x; t < rows * (D / 4); t += gridDim.y * 256) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
            for (int k = 0; k < nparts; ++k) {
                const float4 w = *reinterpret_cast<const float4*>(src + k * SLOT + RE_M + 4 * t);
                v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w;
            }
            *reinterpret_cast<float4*>(gx + (size_t)row0 * D + 4 * t) = v;
        }
    }
}

__global__ void zero_fill_kernel(float* __restrict__ p, size_t n) {
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) p[t] = 0.0f;
}

// rows past the last atom of a known element carry a zero gradient
__global__ void zero_tail_rows_kernel(const int* __restrict__ type_offsets, int ne, int A, int d, float* __restrict__ gx) {
    const int total = type_offsets[ne];
    const size_t n = (size_t)(A - total) * d;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x)
        gx[(size_t)total * d + t] = 0.0f;
}

}  // namespace

extern "C" int qmll_rff_features(const float* x, const double* W, const double* b, const int* mol_index, int A, int d,
                                 int F, int nmol, double* Zf, qmll_stream_t stream) {
    QMLL_REQUIRE(A >= 0 && d > 0 && F > 0 && nmol >= 0, QMLL_ERR_INVALID, "qmll_rff_features: bad size A=%d d=%d F=%d", A,
                 d, F);
    if (A == 0) return QMLL_OK;
    QMLL_REQUIRE(x && W && b && mol_index && Zf, QMLL_ERR_INVALID, "qmll_rff_features: null pointer");
    QMLL_REQUIRE((size_t)RA * d * sizeof(float) <= 64 * 1024, QMLL_ERR_INVALID, "qmll_rff_features: d=%d too large", d);
    QMLL_REQUIRE((F + RT - 1) / RT <= 65535, QMLL_ERR_INVALID, "qmll_rff_features: F=%d too large", F);
    dim3 grid((A + RA - 1) / RA, (F + RT - 1) / RT);
    hipLaunchKernelGGL(rff_features_kernel, grid, dim3(RT), (size_t)RA * d * sizeof(float), (hipStream_t)stream, x, W, b,
                       mol_index, A, d, F, nmol, Zf);
    QMLL_CHECK_LAUNCH("qmll_rff_features");
    return QMLL_OK;
}

extern "C" int qmll_rff_derivative_features(const float* x, const float* grad, const double* W, const double* b,
                                            const int* mol_index, const int* seg_offsets, int A, int n, int d, int F,
                                            int nmol, double* G, qmll_stream_t stream) {
    QMLL_REQUIRE(A >= 0 && n >= 0 && d > 0 && F > 0 && nmol >= 0, QMLL_ERR_INVALID,
                 "qmll_rff_derivative_features: bad size A=%d n=%d d=%d F=%d", A, n, d, F);
    if (A == 0 || n == 0 || nmol == 0) return QMLL_OK;
    QMLL_REQUIRE(x && grad && W && b && (mol_index || seg_offsets) && G, QMLL_ERR_INVALID,
                 "qmll_rff_derivative_features: null pointer");
    if (seg_offsets && (d == 64 || d == 128 || d == 256)) {
        QMLL_REQUIRE(nmol <= 65535 && (3 * n + MROWS - 2) / (MROWS - 1) <= 65535, QMLL_ERR_INVALID,
                     "qmll_rff_derivative_features: grid too large (nmol=%d n=%d)", nmol, n);
        RffElements E = {};
        E.ne = 1;
        E.x[0] = x;
        E.grad[0] = grad;
        E.W[0] = W;
        E.b[0] = b;
        E.seg[0] = seg_offsets;
        launch_rff_rows<double>(E, nullptr, 3 * n, n, d, F, nmol, 0, nullptr, G, (hipStream_t)stream);
        QMLL_CHECK_LAUNCH("qmll_rff_derivative_features");
        return QMLL_OK;
    }
    QMLL_REQUIRE(mol_index, QMLL_ERR_INVALID,
                 "qmll_rff_derivative_features: mol_index is needed when d=%d is not 64, 128 or 256", d);
    const size_t lds = (size_t)(1 + TJ * 3) * d * sizeof(float);
    QMLL_REQUIRE(lds <= 64 * 1024, QMLL_ERR_INVALID, "qmll_rff_derivative_features: d=%d too large", d);
    const int njc = (n + TJ - 1) / TJ;
    QMLL_REQUIRE((long long)A * njc < 2147483647LL && (F + RT - 1) / RT <= 65535, QMLL_ERR_INVALID,
                 "qmll_rff_derivative_features: grid too large");
    dim3 grid((unsigned)(A * njc), (F + RT - 1) / RT);
    hipLaunchKernelGGL(rff_derivative_kernel, grid, dim3(RT), lds, (hipStream_t)stream, x, grad, W, b, mol_index, n, d, F,
                       nmol, njc, G);
    QMLL_CHECK_LAUNCH("qmll_rff_derivative_features");
    return QMLL_OK;
}

extern "C" int qmll_rff_rows(const qmll_rff_element* elements, int ne, const int* row_offsets, int max_rows, int n, int d, int F,
                             int nmol, int overwrite, double* Ze, double* G, qmll_stream_t stream) {
    QMLL_REQUIRE(n >= 0 && nmol >= 0 && ne >= 0 && F > 0 && max_rows >= 0 && max_rows <= 3 * (long long)n, QMLL_ERR_INVALID,
                 "qmll_rff_rows: bad size n=%d nmol=%d ne=%d F=%d max_rows=%d", n, nmol, ne, F, max_rows);
    QMLL_REQUIRE(ne <= RFF_MAXE, QMLL_ERR_INVALID, "qmll_rff_rows: at most %d elements per call (got %d)", RFF_MAXE, ne);
    QMLL_REQUIRE(d == 64 || d == 128 || d == 256, QMLL_ERR_INVALID, "qmll_rff_rows: d=%d is not 64, 128 or 256", d);
    if (n == 0 || nmol == 0 || (ne == 0 && !overwrite)) return QMLL_OK;
    QMLL_REQUIRE((G || max_rows == 0) && (elements || ne == 0), QMLL_ERR_INVALID, "qmll_rff_rows: null pointer");
    QMLL_REQUIRE(nmol <= 65535 && (max_rows + MROWS - 2) / (MROWS - 1) <= 65535, QMLL_ERR_INVALID,
                 "qmll_rff_rows: grid too large (nmol=%d n=%d)", nmol, n);
    RffElements E = {};
    E.ne = ne;
    for (int e = 0; e < ne; ++e) {
        QMLL_REQUIRE(elements[e].x && elements[e].grad && elements[e].W && elements[e].b && elements[e].seg_offsets,
                     QMLL_ERR_INVALID, "qmll_rff_rows: null pointer in element %d", e);
        E.x[e] = elements[e].x;
        E.grad[e] = elements[e].grad;
        E.W[e] = elements[e].W;
        E.b[e] = elements[e].b;
        E.seg[e] = elements[e].seg_offsets;
    }
    launch_rff_rows<float>(E, row_offsets, max_rows, n, d, F, nmol, overwrite, Ze, G, (hipStream_t)stream);
    QMLL_CHECK_LAUNCH("qmll_rff_rows");
    return QMLL_OK;
}

// bytes of the pre-split form of W [ne, d, F]: the images, then one exponent per image
static size_t rff_image_bytes(int d) { return d == 64 ? (size_t)RffImage<64>::BYTES : (size_t)RffImage<128>::BYTES; }

extern "C" size_t qmll_rff_presplit_bytes(int ne, int d, int F) {
    if (ne <= 0 || F <= 0 || F % RE_FC != 0 || (d != 64 && d != 128)) return 0;
    const size_t n = (size_t)ne * (F / RE_FC);
    return n * rff_image_bytes(d) + n * sizeof(int);
}

extern "C" int qmll_rff_presplit(const float* W, int ne, int d, int F, void* out, size_t out_bytes, qmll_stream_t stream) {
    QMLL_REQUIRE(ne > 0 && F > 0, QMLL_ERR_INVALID, "qmll_rff_presplit: bad size ne=%d F=%d", ne, F);
    QMLL_REQUIRE(d == 64 || d == 128, QMLL_ERR_INVALID, "qmll_rff_presplit: d=%d is not 64 or 128", d);
    QMLL_REQUIRE(F % RE_FC == 0, QMLL_ERR_INVALID, "qmll_rff_presplit: F=%d is not a multiple of %d", F, RE_FC);
    QMLL_REQUIRE(W && out, QMLL_ERR_INVALID, "qmll_rff_presplit: null pointer");
    QMLL_REQUIRE(out_bytes >= qmll_rff_presplit_bytes(ne, d, F), QMLL_ERR_INVALID,
                 "qmll_rff_presplit: output of %zu bytes, %zu are needed", out_bytes, qmll_rff_presplit_bytes(ne, d, F));
    QMLL_REQUIRE((((uintptr_t)W | (uintptr_t)out) & 15) == 0, QMLL_ERR_INVALID,
                 "qmll_rff_presplit: W and the output must be 16-byte aligned");
    const int nchunks = F / RE_FC;
    QMLL_REQUIRE(ne <= 65535, QMLL_ERR_INVALID, "qmll_rff_presplit: ne=%d too large", ne);
    _Float16* images = (_Float16*)out;
    int* exponents = (int*)((char*)out + (size_t)ne * nchunks * rff_image_bytes(d));
    const dim3 grid(nchunks, ne);
    if (d == 64)
        hipLaunchKernelGGL(rff_presplit_kernel<64>, grid, dim3(RE_T), 0, (hipStream_t)stream, W, F, images, exponents);
    else
        hipLaunchKernelGGL(rff_presplit_kernel<128>, grid, dim3(RE_T), 0, (hipStream_t)stream, W, F, images, exponents);
    QMLL_CHECK_LAUNCH("qmll_rff_presplit");
    return QMLL_OK;
}

// How the tiles of a launch (128 atoms of one element each) are shared out.  Two workgroups fit a CU (two wavefronts per SIMD; four
// at d = 64 without the gradient) and all walk the chunks of W at the same pace, which is what lets the workgroups of an
// XCD share its L2: W's images are 116 MB at 32768 features, and shares that begin anywhere in W, though of equal size, were bound by their traffic (86016 atoms: 5.4 ms).  So
// as many full rounds of 512 tiles as there are run whole, and each tile of the rest is cut into nparts ranges of chunks.
// In units of one chunk (2.4 us with 512 workgroups resident): a part costs three more for its x and alpha, a launch more
// three, and 72 parts written and read back one.
// The parts used to be added into zero-filled outputs with atomics, 4 bytes each at a stride of a row, which took 2 to 3 ms per
// launch whatever its work.  Measured with the gradient, atomics -> parts: d = 128, 32768 features, 86016 atoms 4.99 -> 4.53 ms, 10000
// atoms 2.06 -> 0.58, 300 atoms 146 -> 67 us; 2048 features, 33000 atoms 3.27 ms -> 173 us; d = 64, 8192 features, 4000 atoms
// 434 -> 55 us.  Energies only, where an atom adds one float a part, they stay up to 4096 of them (added): then the launch that
// sums the parts costs more.  Parts / atomics: d = 128, 1024 features (8 parts), 21 atoms 10.4 / 8.2 us, 512 atoms 11.6 / 10.6; 2048 features
// (16), 21 atoms 10.3 / 8.3, 128 atoms 10.9 / 9.9, 512 atoms 12.1 / 12.7; 8192 features (64), 21 atoms 12.1 / 10.0, 64 atoms 12.4 / 12.4, 256 atoms
// 13.5 / 20.3; 32768 features, 21 atoms 26.4 / 23.3, 128 atoms 26.9 / 29.1; d = 64 alike.
struct RffSplit { int nwhole, ntail, nparts; bool added; };
static RffSplit rff_split(int A, int ne, int d, int F, bool with_grad) {
    const int SLOTS = (d == 64 && !with_grad ? 4 : 2) * 256;
    const int tiles = (A + RE_M - 1) / RE_M + ne, nchunks = F / RE_FC;      // at most: every element's last tile may be partial
    RffSplit p = {tiles / SLOTS * SLOTS, tiles % SLOTS, 1, false};
    double best = nchunks + 3.0;
    for (int k = 2; k <= 64 && nchunks / k >= 4; ++k) {
        const int pieces = p.ntail * k;
        const double cost = ((pieces + SLOTS - 1) / SLOTS) * ((nchunks + k - 1) / k + 3.0) + 3.0 + pieces / 72.0;
        if (cost < best) {
            best = cost;
            p.nparts = k;
        }
    }
    if (p.nparts == 1) {
        p.nwhole = tiles;
        p.ntail = 0;
    }
    p.added = !with_grad && p.ntail > 0 && (long long)A * p.nparts <= 4096;
    return p;
}

extern "C" size_t qmll_rff_energy_workspace_bytes(int A, int ne, int d, int F, int with_grad) {
    if (A <= 0 || ne <= 0 || d <= 0 || F < RE_FC) return 0;
    const RffSplit p = rff_split(A, ne, d, F, with_grad != 0);
    return p.added ? 0 : (size_t)p.ntail * p.nparts * part_floats(d, with_grad) * sizeof(float);
}

extern "C" int qmll_rff_energy_shares(const float* x, const int* type_offsets, const int* sorted_slots, const void* W_split,
                                      const float* b, const float* alpha, int A, int ne, int d, int F, float* work,
                                      size_t work_bytes, float* e_slots, float* gx, qmll_stream_t stream) {
    QMLL_REQUIRE(A >= 0 && ne > 0 && d > 0 && F > 0, QMLL_ERR_INVALID, "qmll_rff_energy_sorted: bad size A=%d ne=%d d=%d F=%d",
                 A, ne, d, F);
    QMLL_REQUIRE(d == 64 || d == 128, QMLL_ERR_INVALID, "qmll_rff_energy_sorted: d=%d is not 64 or 128", d);
    QMLL_REQUIRE(F % RE_FC == 0, QMLL_ERR_INVALID, "qmll_rff_energy_sorted: F=%d is not a multiple of %d", F, RE_FC);
    if (A == 0) return QMLL_OK;
    QMLL_REQUIRE(x && type_offsets && sorted_slots && W_split && b && alpha && e_slots, QMLL_ERR_INVALID,
                 "qmll_rff_energy_sorted: null pointer");
    QMLL_REQUIRE((((uintptr_t)x | (uintptr_t)W_split | (uintptr_t)work | (uintptr_t)gx) & 15) == 0, QMLL_ERR_INVALID,
                 "qmll_rff_energy_sorted: x, W_split, work and gx must be 16-byte aligned");
    QMLL_REQUIRE(!work || work_bytes >= qmll_rff_energy_workspace_bytes(A, ne, d, F, gx != nullptr), QMLL_ERR_INVALID,
                 "qmll_rff_energy_sorted: workspace of %zu bytes, %zu are needed", work_bytes,
                 qmll_rff_energy_workspace_bytes(A, ne, d, F, gx != nullptr));
    const _Float16* images = (const _Float16*)W_split;
    const int* exponents = (const int*)((const char*)W_split + (size_t)ne * (F / RE_FC) * rff_image_bytes(d));
    const float norm = sqrtf(2.0f / (float)F);
    hipStream_t st = (hipStream_t)stream;
    const RffSplit p = rff_split(A, ne, d, F, gx != nullptr);
    if (p.added) work = nullptr;
    if (!work && p.ntail && gx) {
        hipLaunchKernelGGL(zero_fill_kernel, dim3(1024), dim3(256), 0, st, gx, (size_t)A * d);
        QMLL_CHECK_LAUNCH("qmll_rff_energy_sorted");
    }
    auto launch = [&](auto dc, auto gc) {
        constexpr int DD = decltype(dc)::value;
        constexpr bool GG = decltype(gc)::value;
        hipLaunchKernelGGL((rff_energy_sorted_f16_kernel<DD, GG>), dim3(p.nwhole + p.ntail * p.nparts), dim3(RE_T), 0, st, x, type_offsets,
                           sorted_slots, images, exponents, b, alpha, ne, F, p.nwhole, p.nparts, norm, work, e_slots, gx);
        if (work && p.ntail)
            hipLaunchKernelGGL((rff_sum_parts_kernel<DD, GG>), dim3(p.ntail, GG ? 8 : 1), dim3(256), 0, st, type_offsets, sorted_slots,
                               ne, p.nwhole, p.nparts, work, e_slots, gx);
    };
    auto by_grad = [&](auto dc) {
        if (gx) launch(dc, std::true_type{});
        else launch(dc, std::false_type{});
    };
    if (d == 64) by_grad(std::integral_constant<int, 64>{});
    else by_grad(std::integral_constant<int, 128>{});
    QMLL_CHECK_LAUNCH("qmll_rff_energy_sorted");
    if (gx) {
        hipLaunchKernelGGL(zero_tail_rows_kernel, dim3(64), dim3(256), 0, st, type_offsets, ne, A, d, gx);
        QMLL_CHECK_LAUNCH("qmll_rff_energy_sorted");
    }
    return QMLL_OK;
}

extern "C" int qmll_rff_energy_sorted(const float* x, const int* type_offsets, const int* sorted_slots, const void* W_split,
                                      const float* b, const float* alpha, int A, int ne, int d, int F, float* e_slots,
                                      float* gx, qmll_stream_t stream) {
    return qmll_rff_energy_shares(x, type_offsets, sorted_slots, W_split, b, alpha, A, ne, d, F, nullptr, 0, e_slots, gx, stream);
}
