// Fused SORF energy and gradient on element-sorted rows (the contract of qmll_sorf_energy_sorted) with the in-row part of
// the Walsh-Hadamard transforms on the half-precision matrix cores, for d = 64, 128 or 256 and one or two transforms per stack.
//
// H_d = H_{d/16} (x) H_16.  A wavefront carries 16 atoms through a stack.  v_mfma_f32_16x16x32_f16 multiplies the
// +-1 block H_16 (exact in fp16) with a 16 x 16 block of the vectors (index within the block x atom), each fp32 entry
// as two fp16 parts side by side along k: 16 high parts and 16 low parts fill its k = 32, so ONE instruction is one
// 16-point transform of 16 atoms with fp32 accumulation.  Its accumulators hold, per lane, four entries of one atom
// (rows 4 (lane / 16) .. + 3); with d/16 of them a lane holds the remaining log2(d/16) index bits in its own registers,
// where they are plain additions, and the accumulator layout is the operand layout of the transposed transform (a
// lane's four entries, high and low, are its eight k values), so nothing ever crosses lanes.
//
// The first operand of a stack never changes but for the signs of its diagonal: x is split once per atom, and the
// signs go into the H_16 block, which is prepared per call (sorf_prepare_kernel: a block per (element, stack, transform), the
// diagonal must hold +-1) and moved into LDS by direct loads, a round ahead.  The gradient is split per stack (a
// conversion, a mixed-precision subtraction and a conversion per value); both parts are rounded to nearest, 23 bits
// together, one less than fp32: the largest error of an operand is 2^-23 of its binade, the root mean square 0.7 x 2^-24.
// What that adds is taken off elsewhere, in the forms: bias is reduced to a quarter of a revolution in fp64 (the argument's
// rounding is the largest error of either kernel) and the constant factors are rounded once.  Against fp64, root mean square of energies
// / gradients, rows kernel -> this one, relative: d = 128, 128 stacks 3.7e-7 / 3.1e-7 -> 2.3e-7 / 2.2e-7, two transforms, 32 stacks
// 3.1e-7 / 3.1e-7 -> 2.4e-7 / 2.4e-7; with arguments twice as large and falling components 4.7e-7 / 4.6e-7 -> 4.2e-7 / 4.3e-7 at most.
// (The accumulators that start from the bias round it with every partial sum: reduced to a half revolution only, energies and gradients
// of 512 rows were 2.7e-7 / 2.5e-7 where the fma had given 2.5e-7 / 2.3e-7, three draws; to a quarter 2.4e-7 / 2.3e-7.)
// Power-of-two scales keep everything in fp16's range: x per atom
// (sum |x| to [2^13, 2^14), which bounds every partial transform), alpha per call.  With one transform x has a fixed scale, whose
// inverse is in the H_16 blocks, so that the accumulators hold revolutions and can start from the bias behind the inverse of the
// register part's stages: the fma that scaled and added it, 32 per stack, is gone (131072 atoms, 64 stacks, energies only 248 -> 226 us;
// with the gradient 86016 atoms, 128 stacks 630 -> 624).
//
// Instruction issue bounds it, as it does the kernel without matrix instructions (sorf_energy_rows_kernel, which at
// d = 128 spends 162 vector instructions per 4 atoms and stack, 64 of them cross-lane ones at half rate): here 16 atoms
// and a stack take 275 plain, 64 conversion and 64 transcendental vector instructions and 16 matrix instructions, and
// the matrix instructions take issue time of their own (giving one butterfly stage of either side to them leaves the
// time as it was, giving them two makes it 16 % longer).  Two tiles of atoms per wavefront, one stack per barrier,
// eight wavefronts per workgroup and four wavefronts per SIMD (with spills) were measured too: 0 to 4 % slower.
//
// A tile (64 atoms of one element) through all stacks is too coarse a unit: with the three workgroups a CU holds, the last
// of two rounds of tiles left most of the chip idle.  A workgroup takes an equal share of all (tile, round of stacks) units
// instead; of a tile that two or more shares meet in the first writes its sums where they belong, the others theirs into a
// part each, which sorf_parts_kernel adds in order.
// Measured with the gradient / energies only, rows kernel -> this call, at d = 128, 128 stacks: 86016 atoms 764 -> 653 us / 456 -> 305;
// 24000 atoms 222 -> 214 / 133 -> 108; two transforms, 32 stacks, 33000 atoms 148 -> 143 / 78 -> 75, 86016 atoms 369 -> 314 / 194 -> 148;
// d = 64, 128 stacks, 86016 atoms 360 -> 309 / 230 -> 147.  Of that 5 us go to the forms and 3 to 4 to the launch behind.  (These
// are from before the precedence below and the accumulators that start from the bias.)
//
// d = 256: with all of 16 vectors the registers leave two wavefronts per SIMD, which take 890 us for 41796 atoms, 128 stacks where the rows
// kernel takes 822.  So the sixteen columns are eight atoms times the two halves of their vectors: the registers, and three wavefronts per SIMD, are
// those of d = 128, and the eighth index bit is one more stage between lanes eight apart, an addition that reads its partner through the DPP
// network.  The halves have diagonals of their own and share the H_16 block, which is plain and stays in registers: the signs are flipped in the
// split operand, an exclusive or per register.  622 us; energies only 447 -> 295; two transforms, 32 stacks 596 -> 322 / 207 -> 169.
#include <algorithm>
#include <type_traits>

#include "qmll_common.h"

namespace {

typedef float f4_t __attribute__((ext_vector_type(4)));
typedef int int4_t __attribute__((ext_vector_type(4)));

constexpr int SM_WAVES = 4;                  // wavefronts per workgroup
// d = 256: the sixteen columns of a wavefront's operands are eight atoms times the two halves of their vectors
__host__ __device__ constexpr int column_halves(int d) { return d == 256 ? 2 : 1; }
__host__ __device__ constexpr int tile_atoms(int d) { return 16 * SM_WAVES / column_halves(d); }
constexpr float INV2PI = 0.15915494309189535f;
constexpr float UMAX = 1500.0f * INV2PI;     // beyond, whole revolutions are taken off the sine argument first
// One transform: x (in revolutions) goes times 2^SM_EXP into its two fp16 parts: an entry is then off by 2^-33 at most beside its 23
// bits, and atoms of sum |x| up to 128 revolutions fit.  Beside an ordinary bias that is far below the rounding of an argument; where
// some stack's bias is small (below a sixteenth of a revolution in the mean; phases drawn evenly have an eighth), an atom whose entries
// are below SM_LEAST in the mean has a power of two of its own, as those beyond 128 have (no bias and sum |x| = 2e-3 revolutions at
// d = 128: gradients 3.2e-6 off with the common one, 3.1e-7 so).
constexpr int SM_EXP = 8;
constexpr float SM_LEAST = 1.0f / 512, SMALL_BIAS = 1.0f / 16;

// stacks per buffer: one barrier for so many (and at least 3 workgroups in LDS)
constexpr int stacks_per_round(int d, int T) { return d * T <= 128 || d == 256 ? 2 : 1; }
constexpr int SM_CUS = 256;

// index bits of a vector that are not in its 16-point blocks
template <int D>
constexpr int block_bits() { return D == 64 ? 2 : D == 128 ? 3 : 4; }

// where entry k of a vector stands in the rows that a stack reads from LDS: at d = 256 the two halves of a block side by side, as the
// lanes of a wavefront read them at the same time
template <int D>
__device__ __forceinline__ int row_place(int k) {
    return D == 256 ? (k & 0x70) << 1 | (k >> 7) << 4 | (k & 15) : k;
}
// bytes per (element, stack) of the forms that the first operands come from
__host__ __device__ constexpr int image_bytes(int d, int T) { return d == 256 ? T * 1536 : T * d * 64; }

// one 16-point block operand: half t of lane (i, q) is sign * H_16[i][4q + t % 4]
__device__ __forceinline__ bool h16_negative(int i, int h) { return __popc(i & h) & 1; }

// What a launch needs of the model beside its tensors.  Made by every call (sorf_prepare_kernel, 4 us of 150 and more up to 128 stacks): nothing
// is kept that a write to the tensors could leave behind, and no other stream or captured graph has to wait for it.
struct Forms {
    half8_t* images;      // [ne][S][T][NB][64 lanes]: the H_16 blocks behind the signs of their diagonal.  d = 256: [ne][S], of the
                          // diagonals [T][256] in the order of row_place, then the sign bits of the halves [T][4][half, lane / 16][16 bytes]
    float* largest;       // [ne][S]: the largest entry of H D_1 H (one transform: 1, or 2 where the stack's bias is small), infinite where a
                          // diagonal is not +-1
    // Bias in revolutions, reduced to a quarter either way in fp64: the smaller the argument, the less its rounding.  What is taken off is
    // whole halves, and the sign that an odd number of them gives cosine and sine is alpha's.
    float* bias;          // [ne][S][d]; with one transform what its accumulators start from, of which the stages over the block index make that;
                          // this and alpha in the order of row_place
    float* alpha;         // [ne][S][d] +-2^k alpha with the largest entry at [2^13, 2^14) / NB (a transform's register part sums NB of them),
                          // then 2^-k
    float* pieces;        // [alpha_pieces]: the largest entry of each piece of alpha
    int* unfit;           // 1: some diagonal is not +-1, and sorf_energy_rows_kernel takes the call
};

__device__ __forceinline__ float workgroup_max(float m, float* wmax) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
    m = wmax[0];
    for (int w = 1; w < (int)blockDim.x >> 6; ++w) m = fmaxf(m, wmax[w]);
    return m;
}

// The call's scale of alpha comes from its largest entry, which every workgroup of sorf_prepare_kernel has to know.  Up to ALPHA_ALONE
// entries each looks through all of alpha itself; that is S workgroups' reads of S D entries, and beyond a launch ahead finds the largest
// of every ALPHA_PIECE of them and the workgroups look through those.  Whole calls of four elements at d = 128, alone / so: 512 stacks, 3000
// atoms 163 / 154 us, energies only 98 / 88; 2048 stacks, 1500 atoms 526 / 292 and 397 / 161; 256 stacks (32768 entries) 127 / 128.
constexpr int PREP_THREADS = 512;
constexpr int ALPHA_ALONE = 32768, ALPHA_PIECE = 8192;
__host__ __device__ constexpr int alpha_pieces(int S, int D) { return (int)(((long long)S * D + ALPHA_PIECE - 1) / ALPHA_PIECE); }
__global__ __launch_bounds__(PREP_THREADS) void sorf_alpha_pieces_kernel(const float* __restrict__ alpha, int n, float* __restrict__ largest) {
    __shared__ float wmax[PREP_THREADS / 64];
    const int begin = blockIdx.x * ALPHA_PIECE, end = n - begin < ALPHA_PIECE ? n : begin + ALPHA_PIECE;
    float m = 0.0f;
#pragma unroll 8
    for (int t = begin + threadIdx.x; t < end; t += PREP_THREADS) m = fmaxf(m, finite_abs(alpha[t]));
    m = workgroup_max(m, wmax);
    if (threadIdx.x == 0) largest[blockIdx.x] = m;
}

// a workgroup per (element, stack).  bias and alpha may both be null: the images and bounds alone.  The blocks are +-factor.
template <int D, int T>
__global__ __launch_bounds__(PREP_THREADS) void sorf_prepare_kernel(const float* __restrict__ Dmat, const float* __restrict__ bias,
                                                                    const float* __restrict__ alpha, int S, float factor, Forms f) {
    constexpr int NB = D / 16;
    constexpr bool HALVES = D == 256;
    __shared__ float wmax[PREP_THREADS / 64];
    __shared__ float h[D];
    const int tid = threadIdx.x;
    const int e = blockIdx.x / S, s = blockIdx.x - e * S;
    bool unfit = false;
#pragma unroll
    for (int m = 0; m < T; ++m) {
        const float* row = Dmat + (((size_t)e * T + m) * S + s) * D;
        if constexpr (HALVES) {
            char* image = (char*)f.images + ((size_t)e * S + s) * image_bytes(D, T);
            if (tid < D) {
                // the second half of a transform's result has its sign pending, which the next diagonal takes
                const float sd = row[tid], v = m > 0 && tid >= D / 2 ? -sd : sd;
                unfit |= !(fabsf(sd) == 1.0f);
                reinterpret_cast<float*>(image)[m * D + row_place<D>(tid)] = v;
                // blocks 2 j and 2 j + 1 of a half next to each other, four sign bits of 16 each
                const int b = (tid >> 4) & 7, q = (tid >> 2) & 3;
                reinterpret_cast<unsigned short*>(image + T * D * 4 + m * 512)[((b >> 1) * 8 + (tid >> 7) * 4 + q) * 8 + (b & 1) * 4 + (tid & 3)] =
                    v < 0.0f ? 0x8000 : 0;
            }
            continue;
        }
        half8_t* dst = f.images + (((size_t)e * S + s) * T + m) * NB * 64;
        for (int t = tid; t < NB * 64; t += PREP_THREADS) {
            const int b = t >> 6, lane = t & 63, i = lane & 15, q = lane >> 4;
            half8_t v;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float sd = row[16 * b + 4 * q + r], v1 = sd * factor;
                const _Float16 hv = (_Float16)(h16_negative(i, 4 * q + r) ? -v1 : v1);
                v[r] = hv;
                v[r + 4] = hv;
                unfit |= !(fabsf(sd) == 1.0f);
            }
            dst[t] = v;
        }
    }
    float largest = 1.0f;
    if constexpr (T == 2) {
        // entry (i, j) of H D_1 H is entry i ^ j of the transform of D_1's diagonal
        if (tid < D) h[tid] = Dmat[(((size_t)e * T + 1) * S + s) * D + tid];
        for (int o = 1; o < D; o <<= 1) {
            __syncthreads();
            if (tid < D / 2) {
                const int a = (tid & ~(o - 1)) << 1 | (tid & (o - 1));
                const float x = h[a], y = h[a + o];
                h[a] = x + y;
                h[a + o] = x - y;
            }
        }
        __syncthreads();
        largest = workgroup_max(tid < D ? fabsf(h[tid]) : 0.0f, wmax);
    }
    const bool any_unfit = __syncthreads_or(unfit);
    if (bias != nullptr) {
        __shared__ double rev[D];
        const size_t at = ((size_t)e * S + s) * D + tid, to = ((size_t)e * S + s) * D + row_place<D>(tid & (D - 1));
        const float mine = tid < D ? alpha[s * D + tid] : 0.0f;
        bool odd = false;
        if (tid < D) {
            const double b = (double)bias[at], n = rint(b * 0.31830988618379067154);
            odd = n != 2.0 * rint(0.5 * n);
            rev[tid] = fma(b, 0.15915494309189533577, -0.5 * n);
        }
        float m = 0.0f;                  // the call's scale of alpha: every workgroup finds the same value
        const float* from = S * D > ALPHA_ALONE ? f.pieces : alpha;
        const int entries = S * D > ALPHA_ALONE ? alpha_pieces(S, D) : S * D;
#pragma unroll 8
        for (int t = tid; t < entries; t += PREP_THREADS) m = fmaxf(m, finite_abs(from[t]));
        m = workgroup_max(m, wmax);      // (its barriers are also those between the writes of rev and the reads)
        if constexpr (T == 1) {
            float sum = 0.0f;
            if (tid < 64)
                for (int t = tid; t < D; t += 64) sum += fabsf((float)rev[t]);
            sum = wave_sum(sum);         // (of the first wavefront)
            if (sum < D * SMALL_BIAS) largest = 2.0f;
        }
        const int k = max(scale_exponent(m) - block_bits<D>(), -126);
        if (tid < D) {
            double v = rev[tid];
            if constexpr (T == 1) {      // the stages over the block index are their own inverse but for the factor NB
                v = 0.0;
#pragma unroll
                for (int b = 0; b < NB; ++b) v += h16_negative(tid >> 4, b) ? -rev[16 * b + (tid & 15)] : rev[16 * b + (tid & 15)];
                v *= 1.0 / NB;
            } else if (HALVES && tid >= D / 2) {
                v = -v;                  // (the sign that is pending)
            }
            f.bias[to] = (float)v;
            f.alpha[to] = mine * (odd ? -pow2i(k) : pow2i(k));
        }
        if (blockIdx.x == 0 && tid == 0) f.alpha[(size_t)gridDim.x * D] = pow2i(-k);
    }
    if (tid == 0) f.largest[(size_t)e * S + s] = any_unfit ? HUGE_VALF : largest;
}

// Which wavefront of a SIMD issues first.  A plain vector instruction takes the issue two clocks, a conversion four, a sine or cosine
// eight, and a matrix instruction seven beside either of the latter and all of its sixteen beside plain ones: so the wavefronts whose
// phase has the slow instructions go ahead, and the others fill in with their additions.  Left to themselves they run into the same
// phase together.  86016 atoms, 128 components, 128 stacks with the gradient: all equal 624 us; the sines and cosines ahead 581; these and the
// splits with their matrix instructions 548; the stages between the two above the first ones 539; the adjoint's end above them too,
// and the matrix instructions above the sines 526.  Energies only, 131072 atoms, 64 stacks 226 -> 213; two transforms, 32 stacks, 33000
// atoms 143 -> 122 (127 without the forward's second splits).  The first matrix instructions, whose operands come from LDS, gained nothing.
template <int P>
__device__ __forceinline__ void precedence() {
    __builtin_amdgcn_s_setprio(P);
}

// butterflies over the block index
template <int NB>
__device__ __forceinline__ void block_stages(f4_t (&v)[NB]) {
#pragma unroll
    for (int h = 1; h < NB; h <<= 1) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if ((b & h) == 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float x = v[b][r], y = v[b + h][r];
                    v[b][r] = x + y;
                    v[b + h][r] = x - y;
                }
            }
        }
    }
}

// The butterflies between the two halves of a vector, which lie eight lanes apart: v + c * partner, one instruction.  With c = 1 in the
// first half and -1 in the second the second comes out with the other sign, which stays pending; with -c it is the transposed stage.
// (two registers sets behind one pair of wait states, which the writes before may need)
#define QMLL_HALF_STAGE8(x, y, c)                                                                                                   \
    asm("s_nop 1\n\t"                                                                                                               \
        "v_fmac_f32_dpp %0, %0, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %1, %1, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %2, %2, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %3, %3, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %4, %4, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %5, %5, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %6, %6, %8 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %7, %7, %8 row_ror:8 row_mask:0xf bank_mask:0xf"                                                            \
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3])                            \
        : "v"(c))
template <int NB>
__device__ __forceinline__ void half_stage(f4_t (&v)[NB], float c) {
#pragma unroll
    for (int b = 0; b < NB; b += 2) {
        float x[4] = {v[b][0], v[b][1], v[b][2], v[b][3]}, y[4] = {v[b + 1][0], v[b + 1][1], v[b + 1][2], v[b + 1][3]};
        QMLL_HALF_STAGE8(x, y, c);
        v[b] = (f4_t){x[0], x[1], x[2], x[3]};
        v[b + 1] = (f4_t){y[0], y[1], y[2], y[3]};
    }
}

// four values as the lane's eight k entries of an operand: high parts, then low parts, both rounded to nearest
__device__ __forceinline__ half8_t split4(f4_t v) {
    half2_t h0, h1, l0, l1;
    split_pair(v[0], v[1], h0, l0);
    split_pair(v[2], v[3], h1, l1);
    return (half8_t){h0[0], h0[1], h1[0], h1[1], l0[0], l0[1], l1[0], l1[1]};
}

template <int D, int T>
struct StackBuffer {      // what a stack needs, in LDS
    static constexpr int NB = D / 16;
    half8_t signs[T * NB * 64];
    float diag[T * D];
    float bias[D];        // in revolutions (see Forms)
    float alpha[D];       // scaled
};
template <int T>
struct StackBuffer<256, T> {      // all of it in the order of row_place
    float diag[T * 256];
    int4_t signs[T * 32];
    float bias[256];
    float alpha[256];
};

// Tiles of 64 (d = 256: 32) atoms of one element; a share of the launch is a range of (tile, round of SPB stacks) units, tile after tile.
template <int ATOMS>
__device__ __forceinline__ int tile_count(const int* __restrict__ type_offsets, int ne) {
    int n = 0;
    for (int t = 0; t < ne; ++t) n += (type_offsets[t + 1] - type_offsets[t] + ATOMS - 1) / ATOMS;
    return n;
}
template <int ATOMS>
__device__ __forceinline__ void find_tile(const int* __restrict__ type_offsets, int ne, int tile, int& type, int& row0, int& rows) {
    type = row0 = rows = 0;
    for (int t = 0; t < ne; ++t) {
        const int o0 = type_offsets[t], o1 = type_offsets[t + 1], nt = (o1 - o0 + ATOMS - 1) / ATOMS;
        if (tile < nt) {
            type = t;
            row0 = o0 + tile * ATOMS;
            rows = min(ATOMS, o1 - row0);
            return;
        }
        tile -= nt;
    }
}
// First unit of share g of `nshares`, of which `slots` workgroups are resident at a time; with fewer units than shares the last ones
// are empty.  Where there are two rounds of workgroups, the first takes whole tiles and the equal shares of the second level out what
// is left, so that only those are cut: all tiles cut into equal shares end at the same time, but a tile in parts is written and
// read once more (d = 128, 128 stacks with the gradient, all shares equal / whole tiles first: 60000 atoms 474 / 444 us,
// 86016 653 / 628, 131072 972 / 923, 200000 1467 / 1394).  Not where less than an eighth of a tile a share is left, as few tiles are
// then cut into very many parts: 52300 atoms (a sixteenth) 419 / 435, 49400 (all that is left) 390 / 558; 56000 (a seventh) 444 / 414.
constexpr int LEAST_LEFT = 8;
__device__ __forceinline__ int share_begin(int g, int nshares, int slots, int ntiles, int rounds) {
    const int units = ntiles * rounds;
    int whole = 0, each = 0;                                            // shares of whole tiles, tiles in each
    if (nshares >= 2 * slots) {
        whole = (nshares / slots - 1) * slots;
        each = (ntiles + nshares - 1) / nshares;
        // (at least 1 / LEAST_LEFT of a tile a share is left)
        if ((long long)whole * each * LEAST_LEFT > (long long)ntiles * LEAST_LEFT - (nshares - whole)) whole = each = 0;
    }
    if (g < whole) return g * each * rounds;
    const int left = units - whole * each * rounds, used = min(nshares - whole, left);
    return g - whole >= used ? units : units - left + (int)((long long)left * (g - whole) / used);
}
template <int D, bool WITH_GRAD>
constexpr int RESIDENT = (D >= 128 && WITH_GRAD ? 3 : 4) * SM_CUS;

// (at least two wavefronts per SIMD: with up to 256 registers the compiler lets the matrix instructions write vector
// registers directly; asked for fewer it goes through accumulator registers, a move per value)
template <int D, bool WITH_GRAD, int T>
__global__ __launch_bounds__(64 * SM_WAVES) __attribute__((amdgpu_waves_per_eu(2))) void sorf_energy_matrix_kernel(
    const float* __restrict__ x, const int* __restrict__ type_offsets, const int* __restrict__ out_index,
    const float* __restrict__ Dmat, const half8_t* __restrict__ images, const float* __restrict__ bias_rev,
    const float* __restrict__ alpha_scaled, const float* __restrict__ bounds, int ne, int A, int S, int nshares, float xs, float gscale,
    float normf, float* __restrict__ parts, float* __restrict__ e_slots, float* __restrict__ gx) {
    constexpr int HALVES = column_halves(D), NB = D / (16 * HALVES), WAVE_ATOMS = 16 / HALVES, ATOMS = tile_atoms(D);
    using Buffer = StackBuffer<D, T>;
    // two buffers as two arrays: the compiler then knows that loads into one do not touch what is read from the other
    constexpr int SPB = stacks_per_round(D, T);
    __shared__ __attribute__((aligned(16))) Buffer buf0[SPB], buf1[SPB];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, q = lane >> 4;
    const int atom = col & (WAVE_ATOMS - 1), half = HALVES == 2 ? col >> 3 : 0;
    const int at4 = 16 * half + 4 * q;                                  // this lane's entries of a block, in the order of row_place
    const int rounds = (S + SPB - 1) / SPB;

    const int ntiles = tile_count<ATOMS>(type_offsets, ne);
    if ((int)blockIdx.x >= nshares) {
        // a workgroup beyond the shares: its part of the gradient rows of atoms of unknown elements, which are zero
        if constexpr (WITH_GRAD) {
            const int spare = (int)blockIdx.x - nshares, nspare = (int)gridDim.x - nshares;
            for (int r = type_offsets[ne] + spare; r < A; r += nspare)
                for (int c = tid; c < D; c += 64 * SM_WAVES) gx[(size_t)r * D + c] = 0.0f;
        }
        return;
    }
    const int ubeg = share_begin(blockIdx.x, nshares, RESIDENT<D, WITH_GRAD>, ntiles, rounds);
    const int uend = share_begin(blockIdx.x + 1, nshares, RESIDENT<D, WITH_GRAD>, ntiles, rounds);

    for (int u = ubeg; u < uend;) {
        const int tile = u / rounds, r0 = u - tile * rounds, r1 = min(rounds, r0 + uend - u);
        int type, row0, rows;
        find_tile<ATOMS>(type_offsets, ne, tile, type, row0, rows);
        const bool first_piece = r0 == 0;                               // else a part: only a share's first tile can be one
        if (u != ubeg) __syncthreads();                                 // the buffers of the tile before are free
        u += r1 - r0;
        const int s0 = r0 * SPB, s1 = min(S, r1 * SPB);
        float largest = 0.0f;                                           // entry of H D_1 H of the element
        for (int t = lane; t < S; t += 64) largest = fmaxf(largest, bounds[(size_t)type * S + t]);
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) largest = fmaxf(largest, __shfl_xor(largest, o, 64));
        if (largest == HUGE_VALF) continue;                             // not +-1: the rows kernel behind this one writes all

        const float* Dt = Dmat + (size_t)type * T * S * D;
        const unsigned char* it = reinterpret_cast<const unsigned char*>(images) + (size_t)type * S * image_bytes(D, T);
        const float* bt = bias_rev + (size_t)type * S * D;
        const float* at = alpha_scaled + (size_t)type * S * D;

        // stack s into a buffer: direct global-to-LDS loads of 16 bytes per lane, in 1 KiB blocks shared out over the wavefronts
        auto load16 = [&](const void* src, void* dst) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                             (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
        };
        const unsigned lane16 = (unsigned)lane * 16u;
        auto fetch = [&](int s, Buffer& to) {
            const unsigned char* src = it + (size_t)s * image_bytes(D, T);
            if constexpr (HALVES == 2) {      // a row of 256 floats is one such load
                if (wave == 0) load16(bt + (size_t)s * D + lane * 4, to.bias);
                if (wave == 1) load16(at + (size_t)s * D + lane * 4, to.alpha);
                if (WITH_GRAD && wave == 2) load16(src + lane16, to.diag);
                if (WITH_GRAD && T == 2 && wave == 0) load16(src + 1024 + lane16, to.diag + (T - 1) * D);
                if (wave == 3 && lane < 32 * T) load16(src + T * 1024 + lane16, to.signs);
                return;
            }
            unsigned char* dst = reinterpret_cast<unsigned char*>(to.signs);
#pragma unroll
            for (int u = 0; u < T * NB; u += SM_WAVES) load16(src + (u + wave) * 1024 + lane16, dst + (u + wave) * 1024);
            if (lane < D / 4) {      // a row of D floats
                if (wave == 0) load16(bt + (size_t)s * D + lane * 4, to.bias);
                if (wave == 1) load16(at + (size_t)s * D + lane * 4, to.alpha);
                if constexpr (WITH_GRAD) {
                    if (wave == 2) load16(Dt + (size_t)s * D + lane * 4, to.diag);
                    if (T == 2 && wave == 3) load16(Dt + ((size_t)S + s) * D + lane * 4, to.diag + (T - 1) * D);
                }
            }
        };
        auto fetch_all = [&](int s, Buffer (&to)[SPB]) {
#pragma unroll
            for (int k = 0; k < SPB; ++k)
                if (s + k < s1) fetch(s + k, to[k]);
        };
        fetch_all(s0, buf0);

        const int first = WAVE_ATOMS * wave;                 // of this wavefront's atoms
        const bool live = first < rows;                      // of the whole wavefront
        const bool aok = first + atom < rows;

        // x in revolutions, split behind a power of two
        half8_t xop[NB];
        float inv, to_scale;
        bool wide;
        {
            const float* xr = x + (size_t)(row0 + (aok ? first + atom : 0)) * D + D / 2 * half + 4 * q;
            f4_t xv[NB];
            float sum = 0.0f;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                xv[b] = *reinterpret_cast<const f4_t*>(xr + 16 * b);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    xv[b][r] = aok ? xv[b][r] * xs : 0.0f;
                    sum += fabsf(xv[b][r]);
                }
            }
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            if constexpr (HALVES == 2) sum += __shfl_xor(sum, 8, 64);
            // Every argument is at most sum |x|, times the largest entry of H D_1 H for a second transform, + |bias|: where that
            // stays below UMAX no stack looks at its arguments.  One transform: below the second limit all atoms share one power of
            // two, whose inverse is in the H_16 blocks.  (Rows that are not there are zeros.)
            const float bound = fmaf(sum, largest, 0.5f), least = largest > 1.0f ? D * SM_LEAST : 0.0f;
            wide = __any(!(bound <= UMAX && (T == 2 || (sum < (float)(1 << (15 - SM_EXP)) && (sum >= least || sum == 0.0f)))));
            const int kx = T == 1 && !wide ? SM_EXP : not_finite(sum) ? 0 : scale_exponent(sum);
            const float sx = pow2i(kx);
            inv = pow2i((T == 1 ? SM_EXP : 0) - kx);
            to_scale = pow2i(kx - SM_EXP);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
#pragma unroll
                for (int r = 0; r < 4; ++r) xv[b][r] *= sx;
                xop[b] = split4(xv[b]);
            }
        }
        // the plain H_16 block, and the one behind the second transform's adjoint, scaled back into fp16's range
        constexpr int BACK = 4 + block_bits<D>() - 1;
        half8_t hop, hback, hfirst;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const bool neg = h16_negative(col, 4 * q + (t & 3));
            hop[t] = neg ? (_Float16)-1.0f : (_Float16)1.0f;
            hback[t] = neg ? (_Float16)(-1.0f / (1 << BACK)) : (_Float16)(1.0f / (1 << BACK));
            hfirst[t] = neg ? (_Float16)(-1.0f / (1 << SM_EXP)) : (_Float16)(1.0f / (1 << SM_EXP));
        }
        const float cross = half ? -1.0f : 1.0f;
        float uncross = -cross;
        asm("" : "+v"(uncross));                             // kept in a register
        const f4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
        f4_t acc[NB];
        float energy = 0.0f;
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = zero;

        auto stack = [&](const Buffer& B, auto narrow) __attribute__((always_inline)) {
            const bool look = !decltype(narrow)::value && wide;
            f4_t v[NB];
            // four entries of block b from a row
            auto entries = [&](const float* row, int b) { return *reinterpret_cast<const f4_t*>(row + 16 * HALVES * b + at4); };
            auto bias = [&](int b) { return entries(B.bias, b); };
            // transform m's 16-point blocks of `from` (split) behind its diagonal
            auto blocks = [&](int m, auto from, auto start) __attribute__((always_inline)) {
                if constexpr (HALVES == 2) {
#pragma unroll
                    for (int j = 0; j < NB / 2; ++j) {
                        const int4_t sg = B.signs[m * 32 + j * 8 + half * 4 + q];
#pragma unroll
                        for (int k = 0; k < 2; ++k) {
                            const int b = 2 * j + k;
                            const int4_t flip = {sg[2 * k], sg[2 * k + 1], sg[2 * k], sg[2 * k + 1]};
                            const half8_t op = __builtin_bit_cast(half8_t, __builtin_bit_cast(int4_t, from(b)) ^ flip);
                            v[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(T == 1 ? hfirst : hop, op, start(b), 0, 0, 0);
                        }
                    }
                } else {
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        v[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(B.signs[(m * NB + b) * 64 + lane], from(b), start(b), 0, 0, 0);
                }
            };
            auto stages = [&] {
                block_stages<NB>(v);
                if constexpr (HALVES == 2) half_stage<NB>(v, cross);
            };
            auto transposed_stages = [&] {
                block_stages<NB>(v);
                if constexpr (HALVES == 2) half_stage<NB>(v, uncross);
            };
            if constexpr (T == 1) {
                // The accumulators start not from zero, so that the register part's stages add the bias on the way (an instruction
                // per value less, and one rounding less).
                f4_t c[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b) c[b] = bias(b);
                if (__builtin_expect(look, 0)) {
#pragma unroll
                    for (int b = 0; b < NB; ++b) c[b] *= to_scale;
                }
                blocks(0, [&](int b) { return xop[b]; }, [&](int b) { return c[b]; });
                stages();
            } else {
                blocks(0, [&](int b) { return xop[b]; }, [&](int) { return zero; });
                stages();
                precedence<2>();
                blocks(1, [&](int b) { return split4(v[b]); }, [&](int) { return zero; });
                precedence<0>();
                stages();
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const f4_t bv = bias(b);
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[b][r] = fmaf(v[b][r], inv, bv[r]);
                }
            }
            if (__builtin_expect(look, 0)) {
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float u = T == 1 ? v[b][r] * inv : v[b][r];
                        v[b][r] = fabsf(u) > UMAX ? u - rintf(u) : u;      // exact
                    }
            }
            precedence<2>();
            float part = 0.0f;                               // of this stack: the running sum takes one rounding per stack
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const f4_t av = entries(B.alpha, b);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float u = v[b][r];
                    part = fmaf(av[r], __builtin_amdgcn_cosf(u), part);
                    if constexpr (WITH_GRAD) v[b][r] = av[r] * __builtin_amdgcn_sinf(u);
                }
            }
            energy += part;
            if constexpr (!WITH_GRAD) {
                precedence<0>();
            } else {
                precedence<1>();
                transposed_stages();
                precedence<3>();
                if constexpr (T == 2) {
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        const f4_t dv = entries(B.diag + D, b);
                        v[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hback, split4(v[b]), zero, 0, 0, 0) * dv;
                    }
                    precedence<1>();
                    transposed_stages();
                    precedence<3>();
                }
                // summed from zero and added by the vector unit: the matrix instruction aligns its products to the
                // accumulator it is given, and against a sum over many stacks their low bits would be cut off
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    v[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hop, split4(v[b]), zero, 0, 0, 0);
                precedence<1>();
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const f4_t dv = entries(B.diag, b);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[b][r] = fmaf(v[b][r], dv[r], acc[b][r]);
                }
                precedence<0>();
            }
        };
        auto round = [&](int s, const Buffer (&cur)[SPB], Buffer (&other)[SPB], auto narrow) __attribute__((always_inline)) {
            // these stacks' data has landed (every wavefront waits for its own loads, then for the others), and the
            // other buffer, read in the round before, is free
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            fetch_all(s + SPB, other);
            if (!live) return;
#pragma unroll
            for (int k = 0; k < SPB; ++k)
                if (s + k < s1) stack(cur[k], narrow);
        };
        auto all_rounds = [&](auto narrow) __attribute__((always_inline)) {
            for (int s = s0; s < s1; s += 2 * SPB) {
                round(s, buf0, buf1, narrow);
                if (s + SPB < s1) round(s + SPB, buf1, buf0, narrow);
            }
        };
        // Energies only: the short stack without the two branches (131072 atoms, 64 stacks 238 -> 225 us); with the gradient they cost
        // nothing.
        if (WITH_GRAD || __builtin_expect(__syncthreads_or(wide), 0)) all_rounds(std::false_type{});
        else all_rounds(std::true_type{});

        const float inv_alpha = alpha_scaled[(size_t)ne * S * D];
        energy += __shfl_xor(energy, 16, 64);
        energy += __shfl_xor(energy, 32, 64);
        if constexpr (HALVES == 2) energy += __shfl_xor(energy, 8, 64);
        if (!aok) continue;
        const int in_tile = first + atom;
        if (q == 0 && half == 0) {
            const float e = energy * inv_alpha * normf;
            if (first_piece) e_slots[out_index[row0 + in_tile]] = e;
            else parts[(size_t)blockIdx.x * ATOMS * (WITH_GRAD ? D + 1 : 1) + in_tile] = e;
        }
        if constexpr (WITH_GRAD) {
            const float gs = gscale * inv_alpha * (T == 2 ? (float)(1 << BACK) : 1.0f);
            float* to = first_piece ? gx + (size_t)row0 * D : parts + (size_t)blockIdx.x * ATOMS * (D + 1) + ATOMS;
            float* gr = to + (size_t)in_tile * D + D / 2 * half + 4 * q;
#pragma unroll
            for (int b = 0; b < NB; ++b) *reinterpret_cast<f4_t*>(gr + 16 * b) = acc[b] * gs;
        }
    }
}

// the tiles that were cut: workgroup g adds up the parts of the tile that begins in share g and ends in a later one, in order
// (and the last one says whether the rows kernel has to take the call)
template <int D, bool WITH_GRAD>
__global__ __launch_bounds__(256) void sorf_parts_kernel(const int* __restrict__ type_offsets, const int* __restrict__ out_index, int ne,
                                                         int S, int rounds, const float* __restrict__ parts, Forms f,
                                                         float* __restrict__ e_slots, float* __restrict__ gx) {
    constexpr int ATOMS = tile_atoms(D);
    constexpr size_t SLOT = ATOMS * (WITH_GRAD ? D + 1 : 1);
    const int g = blockIdx.x, nshares = (int)gridDim.x - 1;
    if (g == nshares) {
        bool unfit = false;
        for (int t = threadIdx.x; t < ne * S; t += 256) unfit |= f.largest[t] == HUGE_VALF;
        unfit = __syncthreads_or(unfit);
        if (threadIdx.x == 0) *f.unfit = unfit;
        return;
    }
    const int ntiles = tile_count<ATOMS>(type_offsets, ne);
    constexpr int slots = RESIDENT<D, WITH_GRAD>;
    const int ubeg = share_begin(g, nshares, slots, ntiles, rounds), uend = share_begin(g + 1, nshares, slots, ntiles, rounds);
    if (ubeg == uend) return;
    const int tile = (uend - 1) / rounds, tbeg = tile * rounds, tend = tbeg + rounds;
    if (tbeg < ubeg || tend <= uend) return;
    int last = g + 1;                                    // the share in which the tile ends
    while (share_begin(last + 1, nshares, slots, ntiles, rounds) < tend) ++last;
    int type, row0, rows;
    find_tile<ATOMS>(type_offsets, ne, tile, type, row0, rows);
    const float* next = parts + (size_t)(g + 1) * SLOT;
    const int nparts = last - g;
    for (int t = threadIdx.x; t < rows; t += 256) {
        float* to = e_slots + out_index[row0 + t];
        float v = *to;
        for (int b = 0; b < nparts; ++b) v += next[b * SLOT + t];
        *to = v;
    }
    if constexpr (WITH_GRAD) {
        for (int t = threadIdx.x; t < rows * (D / 4); t += 256) {
            f4_t* to = reinterpret_cast<f4_t*>(gx + (size_t)row0 * D) + t;
            f4_t v = *to;
            for (int b = 0; b < nparts; ++b) v += *reinterpret_cast<const f4_t*>(next + b * SLOT + ATOMS + 4 * t);
            *to = v;
        }
    }
}

}  // namespace

static int matrix_rounds(int T, int S, int d) { return (S + stacks_per_round(d, T) - 1) / stacks_per_round(d, T); }
static long long matrix_units(int A, int ne, int T, int S, int d) {
    return ((long long)(A + tile_atoms(d) - 1) / tile_atoms(d) + ne) * matrix_rounds(T, S, d);
}
// Shares of a launch: as many as workgroups are resident, which then all end at the same time, or twice as many where a share of those
// still has many units and the whole tiles of the first round (share_begin) save parts.  Any other number leaves a round of
// workgroups part empty: four shares per CU where three are resident take 292 us for 33000 atoms at d = 128, 128 stacks with the gradient,
// three 228; 60000 atoms with two transforms, 32 stacks 234 and 201.  One round / two: with the gradient 45000 atoms (30 units a
// share) 297 / 313 us, 65000 (42) 409 / 409, 200000 1166 / 1158; energies only 55300 atoms (27) 191 / 195, 100000 (49) 314 / 304, and at
// d = 256 34000 (33) 265 / 263, 60000 443 / 419.
static long long matrix_shares(long long units, int d, int with_grad) {
    const long long resident = SM_CUS * (d >= 128 && with_grad ? 3 : 4);
    return std::min(units, units >= 2 * resident * (with_grad ? 48 : 32) ? 2 * resident : resident);
}

// the workspace of a call: the forms, every part of them 16-byte aligned, then the parts of the cut tiles; its size for base = null
static size_t matrix_workspace(char* base, int A, int ne, int T, int S, int d, int with_grad, Forms& f, float*& parts) {
    size_t at = 0;
    auto take = [&](size_t bytes) {
        char* p = (char*)((uintptr_t)base + at);
        at += (bytes + 15) / 16 * 16;
        return p;
    };
    f.images = (half8_t*)take((size_t)ne * S * image_bytes(d, T));
    f.largest = (float*)take((size_t)ne * S * sizeof(float));
    f.pieces = (float*)take(alpha_pieces(S, d) * sizeof(float));
    f.unfit = (int*)take(sizeof(int));
    f.bias = (float*)take((size_t)ne * S * d * sizeof(float));
    f.alpha = (float*)take(((size_t)ne * S * d + 1) * sizeof(float));
    parts = (float*)take((size_t)matrix_shares(matrix_units(A, ne, T, S, d), d, with_grad) * tile_atoms(d) * (with_grad ? d + 1 : 1) * sizeof(float));
    return at;
}

static int matrix_shape(int ne, int T, int S, int d) {
    return ne > 0 && S > 0 && (T == 1 || T == 2) && (d == 64 || d == 128 || d == 256) && (long long)ne * S < (1ll << 31) - 1 &&
           (long long)S * d < (1ll << 31);
}

extern "C" size_t qmll_sorf_matrix_workspace_bytes(int A, int ne, int T, int S, int d, int with_grad) {
    Forms f;
    float* parts;
    return A <= 0 || !matrix_shape(ne, T, S, d) ? 0 : matrix_workspace(nullptr, A, ne, T, S, d, with_grad, f, parts);
}

// What this kernel gains per atom and stack has to carry three launches more and the parts of the cut tiles, 25 us with the
// gradient and 15 us without.  Measured, rows kernel / this call, in units of 1e6 below.  With the gradient, one transform: d = 128, 128 stacks
// 10000 atoms (1.3) 100 / 106 us, 12000 (1.5) 117 / 116, 17000 161 / 142, 32 stacks 40000 atoms (1.3) 101 / 102; d = 64 18000 (1.2) 84 / 84;
// d = 256 5000 (1.3) 112 / 120, 7000 (1.8) 151 / 144.  Two transforms, 32 stacks: d = 128 14000 atoms (0.9) 68 / 81, 18000 (1.2) 86 / 88,
// 24000 (1.5) 111 / 101; d = 64 30000 (1.0) 68 / 71, 40000 (1.3) 87 / 79; d = 256, where the rows kernel has few wavefronts per SIMD, 4000
// (0.5) 70 / 78, 6000 (0.8) 101 / 86.  Energies only: d = 128 10000 (1.3) 61 / 64, 12000 (1.5) 71 / 68; d = 64 18000 (1.2) 54 / 53; d = 256
// 5000 (1.3) 63 / 67, 7000 (1.8) 85 / 82; two transforms, d = 128 24000 (1.5) 61 / 63, d = 256 14000 (1.8) 76 / 77.
// The same product of more stacks and fewer atoms makes more forms, and more parts of each tile: with the gradient, d = 128, 256 stacks 6000
// atoms (1.5) 118 / 128, 384 4000 (1.5) 122 / 138, 512 3000 (1.5) 125 / 154 and 3515 (1.8) 160 / 160, 2048 878 (1.8) 175 / 283 and 1318 (2.7)
// 339 / 292; d = 64, 2048 1757 (1.8) 183 / 199; two transforms, d = 128, 128 4687 (1.2) 100 / 112 and 7031 (1.8) 134 / 129, 512 1171 (1.2)
// 188 / 205.  At d = 256 the rows kernel has as few workgroups then: 512 stacks 1171 atoms (1.2) 190 / 167.
extern "C" int qmll_sorf_matrix_pays(int A, int ne, int T, int S, int d, int with_grad) {
    if (!matrix_shape(ne, T, S, d) || matrix_units(A, ne, T, S, d) >= (1ll << 31)) return 0;
    double line = with_grad ? (T == 1 ? 1.5e6 : d == 256 ? 0.75e6 : 1.2e6) : (T == 1 ? 1.5e6 : 1.8e6);
    if (with_grad && d <= 128) line = std::min(2e6, line * pow(std::max(1.0, S / (T == 1 ? 128.0 : 32.0)), 1.0 / 6.0));
    return (double)A * S * T * d / 128.0 >= line;
}

static void launch_prepare(const float* D, const float* bias, const float* alpha, int ne, int T, int S, int d, float factor,
                           const Forms& f, hipStream_t st) {
    const dim3 grid(ne * S), block(PREP_THREADS);
    if (alpha && S * d > ALPHA_ALONE) hipLaunchKernelGGL(sorf_alpha_pieces_kernel, dim3(alpha_pieces(S, d)), block, 0, st, alpha, S * d, f.pieces);
    if (d == 64 && T == 1) hipLaunchKernelGGL((sorf_prepare_kernel<64, 1>), grid, block, 0, st, D, bias, alpha, S, factor, f);
    else if (d == 64) hipLaunchKernelGGL((sorf_prepare_kernel<64, 2>), grid, block, 0, st, D, bias, alpha, S, factor, f);
    else if (d == 128 && T == 1) hipLaunchKernelGGL((sorf_prepare_kernel<128, 1>), grid, block, 0, st, D, bias, alpha, S, factor, f);
    else if (d == 256 && T == 1) hipLaunchKernelGGL((sorf_prepare_kernel<256, 1>), grid, block, 0, st, D, bias, alpha, S, factor, f);
    else if (d == 256) hipLaunchKernelGGL((sorf_prepare_kernel<256, 2>), grid, block, 0, st, D, bias, alpha, S, factor, f);
    else hipLaunchKernelGGL((sorf_prepare_kernel<128, 2>), grid, block, 0, st, D, bias, alpha, S, factor, f);
}

static int signs_shape(int ne, int T, int S, int d) { return matrix_shape(ne, T, S, d) && d <= 128; }

extern "C" size_t qmll_sorf_signs_bytes(int ne, int T, int S, int d) {
    return signs_shape(ne, T, S, d) ? (size_t)ne * S * image_bytes(d, T) + (size_t)ne * S * sizeof(float) : 0;
}

extern "C" int qmll_sorf_signs(const float* D, int ne, int T, int S, int d, void* out, size_t out_bytes, qmll_stream_t stream) {
    QMLL_REQUIRE(signs_shape(ne, T, S, d), QMLL_ERR_INVALID, "qmll_sorf_signs: no kernel takes ne=%d T=%d S=%d d=%d", ne, T, S, d);
    QMLL_REQUIRE(D && out && ((uintptr_t)out & 15) == 0, QMLL_ERR_INVALID, "qmll_sorf_signs: null or misaligned pointer");
    QMLL_REQUIRE(out_bytes >= qmll_sorf_signs_bytes(ne, T, S, d), QMLL_ERR_INVALID, "qmll_sorf_signs: output of %zu bytes, %zu are needed",
                 out_bytes, qmll_sorf_signs_bytes(ne, T, S, d));
    Forms f = {};
    f.images = (half8_t*)out;
    f.largest = (float*)((char*)out + (size_t)ne * S * image_bytes(d, T));
    launch_prepare(D, nullptr, nullptr, ne, T, S, d, 1.0f, f, (hipStream_t)stream);
    QMLL_CHECK_LAUNCH("qmll_sorf_signs");
    return QMLL_OK;
}

extern "C" int qmll_sorf_energy_matrix(const float* x, const int* type_offsets, const int* sorted_slots, const float* D,
                                       const float* bias, const float* alpha, int A, int ne, int d, int S, int T,
                                       float normalisation, void* work, size_t work_bytes, float* e_slots, float* gx,
                                       qmll_stream_t stream) {
    QMLL_REQUIRE(A >= 0 && matrix_shape(ne, T, S, d), QMLL_ERR_INVALID,
                 "qmll_sorf_energy_matrix: bad size A=%d ne=%d T=%d S=%d d=%d", A, ne, T, S, d);
    if (A == 0) return QMLL_OK;
    QMLL_REQUIRE(x && type_offsets && sorted_slots && D && bias && alpha && e_slots, QMLL_ERR_INVALID,
                 "qmll_sorf_energy_matrix: null pointer");
    QMLL_REQUIRE(work && work_bytes >= qmll_sorf_matrix_workspace_bytes(A, ne, T, S, d, gx != nullptr), QMLL_ERR_INVALID,
                 "qmll_sorf_energy_matrix: workspace of %zu bytes, %zu are needed", work ? work_bytes : (size_t)0,
                 qmll_sorf_matrix_workspace_bytes(A, ne, T, S, d, gx != nullptr));
    QMLL_REQUIRE(matrix_units(A, ne, T, S, d) < (1ll << 31), QMLL_ERR_INVALID,
                 "qmll_sorf_energy_matrix: %d atoms times %d stacks are too many for one launch", A, S);
    QMLL_REQUIRE((((uintptr_t)x | (uintptr_t)work | (uintptr_t)D | (uintptr_t)gx) & 15) == 0, QMLL_ERR_INVALID,
                 "qmll_sorf_energy_matrix: x, D, work and gx must be 16-byte aligned");
    Forms f;
    float* parts;
    matrix_workspace((char*)work, A, ne, T, S, d, gx != nullptr, f, parts);
    // x into revolutions, and the factors of the gradient and of the energy, each rounded once
    const double scale = (double)normalisation / (T == 1 ? sqrt((double)d) : (double)d), norm = sqrt(2.0 / ((double)S * d));
    const float xs = (float)(scale * 0.15915494309189533577), gscale = (float)(-scale * norm), normf = (float)norm;
    const int nshares = (int)matrix_shares(matrix_units(A, ne, T, S, d), d, gx != nullptr);
    const dim3 grid(nshares + (gx ? (A >= 65536 ? 64 : (A >> 10) + 1) : 0));
    hipStream_t st = (hipStream_t)stream;
    launch_prepare(D, bias, alpha, ne, T, S, d, T == 1 ? 1.0f / (1 << SM_EXP) : 1.0f, f, st);
    auto launch = [&](auto dc, auto tc, auto gc) {
        constexpr int DD = decltype(dc)::value, TT = decltype(tc)::value;
        constexpr bool GG = decltype(gc)::value;
        hipLaunchKernelGGL((sorf_energy_matrix_kernel<DD, GG, TT>), grid, dim3(64 * SM_WAVES), 0, st, x, type_offsets, sorted_slots, D,
                           f.images, f.bias, f.alpha, f.largest, ne, A, S, nshares, xs, gscale, normf, parts, e_slots, gx);
        hipLaunchKernelGGL((sorf_parts_kernel<DD, GG>), dim3(nshares + 1), dim3(256), 0, st, type_offsets, sorted_slots, ne, S,
                           matrix_rounds(TT, S, DD), parts, f, e_slots, gx);
    };
    auto by_grad = [&](auto dc, auto tc) {
        if (gx) launch(dc, tc, std::true_type{});
        else launch(dc, tc, std::false_type{});
    };
    auto by_d = [&](auto tc) {
        if (d == 64) by_grad(std::integral_constant<int, 64>{}, tc);
        else if (d == 128) by_grad(std::integral_constant<int, 128>{}, tc);
        else by_grad(std::integral_constant<int, 256>{}, tc);
    };
    if (T == 1) by_d(std::integral_constant<int, 1>{});
    else by_d(std::integral_constant<int, 2>{});
    QMLL_CHECK_LAUNCH("qmll_sorf_energy_matrix");
    // diagonals that are not +-1, which only the device knows of: the rows kernel, whose workgroups else return at once
    return qmll_sorf_rows_if(x, type_offsets, sorted_slots, D, bias, alpha, A, ne, d, S, T, normalisation, f.unfit, e_slots, gx, st);
}
