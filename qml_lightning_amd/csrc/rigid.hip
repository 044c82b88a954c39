// Force rows of a training batch without the combinations that vanish identically.
//
// The representation depends on differences of coordinates only, so moving a molecule as a whole leaves every
// feature as it is: of a molecule's 3n force-feature rows (qml_lightning/models/kernel.py:167-170) the three
// sums over the atoms (translations) are zero, and without periodic images so are the three combinations
// sum_i (e_c x (r_i - r)) . G_i (rotations).  Z^T Z and Z^T y do not change when a molecule's rows and targets are
// replaced by Q^T G and Q^T y with an orthogonal Q; with Q the product of the Householder reflections that
// map the vanishing combinations onto the first k rows, those k rows are zero (up to the rounding of the fp32
// representation, which enters Z^T Z squared) and are left out of the Gram product, together with the rows
// of the padded slots: 58 rows instead of 64 per C9H8O4 molecule with its energy row, less than half for molecules
// padded to the largest of a mixed batch.  The rows are linear in the projected Jacobian, so Q acts on that
// (npcas columns) and not on the rows (nfeatures columns).
#include "qmll_common.h"

namespace {

constexpr int NV = 8;   // doubles per row of V: 6 reflections, padded to one 64-byte scalar load

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// One wavefront per molecule.  modes[m] = k: 3 translations, then k - 3 of the three rotations, largest norm
// first (two atoms have two); 0: the molecule's rows stay as they are.  V [B][3n][NV] holds the unit vectors of the reflections I - 2 v v^T,
// T [B][36] the factor of Q = H_0 H_1 .. = I - V T V^T (upper triangular, T_jj = 2).
__global__ __launch_bounds__(64) void rigid_modes_kernel(const float* __restrict__ X, const int* __restrict__ natoms,
                                                         const int* __restrict__ modes, const int* __restrict__ row_offsets,
                                                         int n, double* __restrict__ V, double* __restrict__ T,
                                                         const double* __restrict__ forces, double* __restrict__ targets) {
    const int m = blockIdx.x, lane = threadIdx.x;
    const int nm = min(natoms[m], n), rows = 3 * nm;
    int k = min(max(modes[m], 0), 6);
    if (k > rows) k = rows;
    double* Vm = V + (size_t)m * 3 * n * NV;
    double* Tm = T + (size_t)m * 36;
    const float* Xm = X + (size_t)m * n * 3;
    double c[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        double s = 0.0;
        for (int i = lane; i < nm; i += 64) s += (double)Xm[3 * i + x];
        c[x] = wave_sum_f64(s) / (double)max(nm, 1);
    }
    // the six combinations, as columns of V
    for (int r = lane; r < rows; r += 64) {
        const int i = r / 3, x = r - 3 * i;
        const double dx = (double)Xm[3 * i] - c[0], dy = (double)Xm[3 * i + 1] - c[1], dz = (double)Xm[3 * i + 2] - c[2];
        double* v = Vm + (size_t)r * NV;
#pragma unroll
        for (int t = 0; t < 3; ++t) v[t] = x == t ? 1.0 : 0.0;
        v[3] = x == 1 ? -dz : (x == 2 ? dy : 0.0);      // e_x x d
        v[4] = x == 0 ? dz : (x == 2 ? -dx : 0.0);      // e_y x d
        v[5] = x == 0 ? -dy : (x == 1 ? dx : 0.0);      // e_z x d
        v[6] = v[7] = 0.0;
    }
    __syncthreads();
    for (int j = 0; j < 6; ++j) {
        if (j >= k) {                                    // not a reflection of this molecule
            for (int r = lane; r < rows; r += 64) Vm[(size_t)r * NV + j] = 0.0;
            continue;
        }
        int p = j;
        double best = 0.0;
        for (int q = j; q < (j < 3 ? j + 1 : 6); ++q) {
            double s = 0.0;
            for (int r = j + lane; r < rows; r += 64) s += Vm[(size_t)r * NV + q] * Vm[(size_t)r * NV + q];
            s = wave_sum_f64(s);
            if (q == j || s > best) {
                best = s;
                p = q;
            }
        }
        __syncthreads();
        if (p != j) {
            for (int r = lane; r < rows; r += 64) {
                const double u = Vm[(size_t)r * NV + j];
                Vm[(size_t)r * NV + j] = Vm[(size_t)r * NV + p];
                Vm[(size_t)r * NV + p] = u;
            }
            __syncthreads();
        }
        const double head = Vm[(size_t)j * NV + j];
        const double norm = sqrt(best);
        const double vh = head + (head < 0.0 ? -norm : norm);
        const double len2 = best - head * head + vh * vh;      // |v|^2 of v = w + sign(w_j) |w| e_j
        const double inv = len2 > 0.0 ? 1.0 / sqrt(len2) : 0.0;
        __syncthreads();
        for (int r = lane; r < rows; r += 64) {
            const double w = Vm[(size_t)r * NV + j];
            Vm[(size_t)r * NV + j] = r < j ? 0.0 : (r == j ? vh : w) * inv;
        }
        __syncthreads();
        for (int q = j + 1; q < 6; ++q) {
            double s = 0.0;
            for (int r = j + lane; r < rows; r += 64) s += Vm[(size_t)r * NV + j] * Vm[(size_t)r * NV + q];
            s = 2.0 * wave_sum_f64(s);
            for (int r = j + lane; r < rows; r += 64) Vm[(size_t)r * NV + q] -= s * Vm[(size_t)r * NV + j];
        }
        __syncthreads();
    }
    // T column by column: T_jj = 2, T_{0..j-1, j} = -2 T (V^T v_j)
    double t[6][6];
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) t[i][j] = 0.0;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        double d[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            d[i] = 0.0;
            if (i < j) {
                double s = 0.0;
                for (int r = lane; r < rows; r += 64) s += Vm[(size_t)r * NV + i] * Vm[(size_t)r * NV + j];
                d[i] = wave_sum_f64(s);
            }
        }
        t[j][j] = 2.0;
#pragma unroll
        for (int i = 0; i < 6; ++i)
            if (i < j) {
                double s = 0.0;
#pragma unroll
                for (int l = 0; l < 6; ++l)
                    if (l >= i && l < j) s += t[i][l] * d[l];
                t[i][j] = -2.0 * s;
            }
    }
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j)
            if (lane == 6 * i + j) Tm[lane] = t[i][j];
    if (forces == nullptr || targets == nullptr) return;     // no targets wanted, or no row remains
    // the targets: y - V T^T V^T y, rows k..
    const double* y = forces + (size_t)m * 3 * n;
    double w[6], u[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        double s = 0.0;
        for (int r = lane; r < rows; r += 64) s += Vm[(size_t)r * NV + j] * y[r];
        w[j] = wave_sum_f64(s);
    }
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        u[j] = 0.0;
#pragma unroll
        for (int i = 0; i < 6; ++i)
            if (i <= j) u[j] += t[i][j] * w[i];
    }
    double* out = targets + row_offsets[m];
    for (int r = k + lane; r < rows; r += 64) {
        double v = y[r];
#pragma unroll
        for (int j = 0; j < 6; ++j) v -= Vm[(size_t)r * NV + j] * u[j];
        out[r - k] = v;
    }
}

// Q^T on the projected Jacobian rows of one atom, in place: rows k.. of the molecule's 3 natoms move to the front.
// Thread = column; a column's rows are read twice (the second time from L2: 32 KB per workgroup at 128 components and
// 21 atoms), the reflections arrive through scalar loads.  Sums in fp64, one rounding to fp32 per value.
// HBM bound: 2 x 4 x 3n x d bytes per atom.
__global__ void rigid_rows_kernel(float* __restrict__ grad, const int* __restrict__ slots, const int* __restrict__ natoms,
                                  const int* __restrict__ modes, const double* __restrict__ V, const double* __restrict__ T, int n,
                                  int B, int d) {
    const int slot = slots[blockIdx.x];
    const int m = slot / n;
    if (slot < 0 || m >= B) return;
    const int rows = 3 * min(natoms[m], n);
    const int k = min(min(max(modes[m], 0), 6), rows);
    const double* __restrict__ Vm = V + (size_t)m * 3 * n * NV;
    const double* __restrict__ Tm = T + (size_t)m * 36;
    for (int c = threadIdx.x; c < d; c += blockDim.x) {
        float* g = grad + (size_t)blockIdx.x * 3 * n * d + c;
        double w[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int r = 0; r < rows; ++r) {
            const double v = (double)g[(size_t)r * d];
#pragma unroll
            for (int j = 0; j < 6; ++j) w[j] = fma(Vm[r * NV + j], v, w[j]);
        }
        double u[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            u[j] = 0.0;
#pragma unroll
            for (int i = 0; i < 6; ++i)
                if (i <= j) u[j] = fma(Tm[6 * i + j], w[i], u[j]);
        }
#pragma unroll 4
        for (int r = k; r < rows; ++r) {
            double v = (double)g[(size_t)r * d];
#pragma unroll
            for (int j = 0; j < 6; ++j) v = fma(-Vm[r * NV + j], u[j], v);
            g[(size_t)(r - k) * d] = (float)v;
        }
    }
}

__global__ void typed_segments_kernel(const int* __restrict__ slots, const int* __restrict__ type_offsets, int ne, int B, int n,
                                      int* __restrict__ seg) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ne * (B + 1)) return;
    const int e = t / (B + 1), m = t - e * (B + 1);
    const int o0 = type_offsets[e], o1 = type_offsets[e + 1];
    int lo = o0, hi = o1;                    // first atom whose slot is not before molecule m
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (slots[mid] < m * n) lo = mid + 1;
        else hi = mid;
    }
    seg[t] = lo - o0;
}

}  // namespace

extern "C" int qmll_typed_segments(const int* sorted_slots, const int* type_offsets, int ne, int B, int n, int* seg,
                                   qmll_stream_t stream) {
    QMLL_REQUIRE(ne > 0 && B >= 0 && n > 0, QMLL_ERR_INVALID, "qmll_typed_segments: bad size ne=%d B=%d n=%d", ne, B, n);
    QMLL_REQUIRE(sorted_slots && type_offsets && seg, QMLL_ERR_INVALID, "qmll_typed_segments: null pointer");
    hipLaunchKernelGGL(typed_segments_kernel, dim3((ne * (B + 1) + 255) / 256), dim3(256), 0, (hipStream_t)stream, sorted_slots,
                       type_offsets, ne, B, n, seg);
    QMLL_CHECK_LAUNCH("qmll_typed_segments");
    return QMLL_OK;
}

extern "C" size_t qmll_rigid_workspace_bytes(int B, int n) {
    if (B <= 0 || n <= 0) return 0;
    return ((size_t)B * 3 * n * NV + (size_t)B * 36) * sizeof(double);
}

extern "C" int qmll_rigid_modes(const float* X, const int* natoms, const int* modes, const int* row_offsets, int B, int n,
                                double* work, size_t work_bytes, const double* forces, double* targets,
                                qmll_stream_t stream) {
    QMLL_REQUIRE(B >= 0 && n >= 0, QMLL_ERR_INVALID, "qmll_rigid_modes: bad size B=%d n=%d", B, n);
    if (B == 0 || n == 0) return QMLL_OK;
    QMLL_REQUIRE(X && natoms && modes && row_offsets && work, QMLL_ERR_INVALID, "qmll_rigid_modes: null pointer");
    QMLL_REQUIRE(work_bytes >= qmll_rigid_workspace_bytes(B, n), QMLL_ERR_INVALID,
                 "qmll_rigid_modes: workspace of %zu bytes, %zu are needed", work_bytes, qmll_rigid_workspace_bytes(B, n));
    hipLaunchKernelGGL(rigid_modes_kernel, dim3(B), dim3(64), 0, (hipStream_t)stream, X, natoms, modes, row_offsets, n, work,
                       work + (size_t)B * 3 * n * NV, forces, targets);
    QMLL_CHECK_LAUNCH("qmll_rigid_modes");
    return QMLL_OK;
}

extern "C" int qmll_rigid_rows(float* grad, const int* slots, const int* natoms, const int* modes, const double* work, int A, int B,
                               int n, int d, qmll_stream_t stream) {
    QMLL_REQUIRE(A >= 0 && B >= 0 && n >= 0 && d > 0, QMLL_ERR_INVALID, "qmll_rigid_rows: bad size A=%d B=%d n=%d d=%d", A, B, n,
                 d);
    if (A == 0 || B == 0 || n == 0) return QMLL_OK;
    QMLL_REQUIRE(grad && slots && natoms && modes && work, QMLL_ERR_INVALID, "qmll_rigid_rows: null pointer");
    const int threads = d >= 256 ? 256 : (d + 63) / 64 * 64;
    hipLaunchKernelGGL(rigid_rows_kernel, dim3(A), dim3(threads), 0, (hipStream_t)stream, grad, slots, natoms, modes, work,
                       work + (size_t)B * 3 * n * NV, n, B, d);
    QMLL_CHECK_LAUNCH("qmll_rigid_rows");
    return QMLL_OK;
}
